"""The fp32 MFMA attention over window sizes, head dims and masks against 64 bits."""
import pytest
import torch

import nsw

pytestmark = pytest.mark.gpu


def _ref(qkv, heads, scale, mask=None):
    Bw, L, C3 = qkv.shape
    q, k, v = [t.reshape(Bw, L, heads, -1).transpose(1, 2).double() for t in qkv.split(C3 // 3, -1)]
    s = torch.matmul(q.contiguous(), k.transpose(-1, -2).contiguous()) * scale
    if mask is not None:
        s = s + mask.double().repeat(Bw // mask.shape[0], 1, 1)[:, None]
    return torch.matmul(torch.softmax(s, -1), v.contiguous()).transpose(1, 2).reshape(Bw, L, C3 // 3)


def _rel(o, want):
    return ((o.double() - want).norm() / want.norm()).item()


def _qkv(Bw, L, C, seed):
    g = torch.Generator(device="cuda:0").manual_seed(seed)
    return torch.randn(Bw, L, 3 * C, generator=g, device="cuda:0")


# L: one token, around a 16-key block, a chunk of 3 / 6 / 11 blocks, the 4- / 8-wave
# line (192) and the largest window of the kernel (384); past it the generic kernel
@pytest.mark.parametrize("hd,heads", [(4, 6), (8, 3), (16, 2), (32, 3), (64, 2), (128, 1)])
@pytest.mark.parametrize("L", [1, 17, 48, 96, 162, 177, 192, 193, 324, 384, 400])
@pytest.mark.parametrize("masked", [False, True])
def test_attention_f32_sizes(hd, heads, L, masked):
    qkv = _qkv(4, L, hd * heads, L)
    mask = None
    if masked:
        g = torch.Generator(device="cuda:0").manual_seed(L)
        mask = torch.randn(2, L, L, generator=g, device="cuda:0")
    o = nsw.ops.window_attention(qkv, heads, hd ** -0.5, mask=mask)
    # U sqrt(hd) |q||k| scale ~ 2^-24 hd in the exponent, 2^-24 sqrt(L) in the sums
    assert _rel(o, _ref(qkv, heads, hd ** -0.5, mask)) < 2.0 ** -24 * (hd + 2 * L ** 0.5 + 8)


# both sides of the line below which windows go to the generic kernel (4 to 13
# tokens); the bound as above
@pytest.mark.parametrize("hd,heads", [(4, 6), (8, 3), (16, 2), (32, 3), (64, 2), (128, 1)])
@pytest.mark.parametrize("L", [3, 4, 5, 8, 9, 12, 13])
def test_attention_f32_few_tokens(hd, heads, L):
    qkv = _qkv(6, L, hd * heads, L)
    g = torch.Generator(device="cuda:0").manual_seed(L)
    mask = torch.randn(2, L, L, generator=g, device="cuda:0")
    for m in (None, mask):
        o = nsw.ops.window_attention(qkv, heads, hd ** -0.5, mask=m)
        assert _rel(o, _ref(qkv, heads, hd ** -0.5, m)) < 2.0 ** -24 * (hd + 2 * L ** 0.5 + 8)


# more items than CUs (four waves an item up to 192 tokens; fewer items above take
# eight up from 65 tokens); the bound as above
@pytest.mark.parametrize("hd", [16, 32, 64, 128])
@pytest.mark.parametrize("L", [64, 65, 96, 162, 192])
@pytest.mark.parametrize("items", [256, 258])
def test_attention_f32_wave_counts(hd, L, items):
    qkv = _qkv(items // 2, L, 2 * hd, L)
    g = torch.Generator(device="cuda:0").manual_seed(L)
    for mask in (None, torch.randn(1, L, L, generator=g, device="cuda:0")):
        o = nsw.ops.window_attention(qkv, 2, hd ** -0.5, mask=mask)
        assert _rel(o, _ref(qkv, 2, hd ** -0.5, mask)) < 2.0 ** -24 * (hd + 2 * L ** 0.5 + 8)


@pytest.mark.parametrize("L", [100, 324])
def test_attention_f32_mask_extremes(L):
    """Keys masked with -inf (a whole leading chunk of them too), rows masked with
    the lowest float throughout (uniform weights) or with -inf (NaN), as softmax."""
    qkv = _qkv(2, L, 64, 3)
    mask = torch.zeros(1, L, L, device="cuda:0")
    mask[0, 1, : L - 3] = float("-inf")
    mask[0, 2, 5:] = float("-inf")
    mask[0, 3] = torch.finfo(torch.float32).min
    mask[0, 4, :50] = torch.finfo(torch.float32).min
    mask[0, 5] = float("-inf")
    o = nsw.ops.window_attention(qkv, 1, 0.125, mask=mask)
    assert torch.isnan(o[:, 5]).all()
    keep = [i for i in range(L) if i != 5]
    m64 = mask.clone()
    m64[0, 5] = 0
    m64[0, 3] = 0                                   # -3.4e38 swallows the logits in fp32: uniform
    want = _ref(qkv, 1, 0.125, m64)
    want[:, 3] = qkv[:, :, 128:].double().mean(1)
    assert _rel(o[:, keep], want[:, keep]) < 1e-5


@pytest.mark.parametrize("scale", [0.0, -0.3, 1e-37, 1e-30])
def test_attention_f32_scales(scale):
    """Scales that are not positive or whose -100 / scale is not finite (1e-37) go to
    the generic kernel, with the shift mask; 1e-30 is the smallest kind that does not."""
    H, W = 18, 36
    qkv = _qkv(4, 162, 64, 9)
    o = nsw.ops.window_attention(qkv, 2, scale, geometry=(H, W, (9, 18), (4, 9), 1))
    r = torch.arange(162, device="cuda:0") // 18 >= 5
    mask = torch.zeros(4, 162, 162, device="cuda:0")
    mask[2:] = torch.where(r[:, None] != r[None], -100.0, 0.0)
    assert _rel(o, _ref(qkv, 2, scale, mask)) < 1e-5


# head dims 4 and 8 pass keys in chunks of 7 blocks (112): around one, two and three
# chunks, with the shift mask from indices, a mask tensor (a whole leading chunk of
# -inf in one row) and none; the bound as above
@pytest.mark.parametrize("hd,heads", [(4, 3), (8, 2)])
@pytest.mark.parametrize("L", [15, 16, 111, 112, 113, 224, 225, 336, 337])
@pytest.mark.parametrize("kind", ["none", "mask"])
def test_attention_f32_narrow_chunks(hd, heads, L, kind):
    C = 16 * ((hd * heads + 15) // 16)
    heads = C // hd
    qkv = _qkv(3, L, C, L + hd)
    mask = None
    if kind == "mask":
        g = torch.Generator(device="cuda:0").manual_seed(L)
        mask = torch.randn(3, L, L, generator=g, device="cuda:0")
        mask[1, 0, : L - 1] = float("-inf")
    o = nsw.ops.window_attention(qkv, heads, hd ** -0.5, mask=mask)
    assert _rel(o, _ref(qkv, heads, hd ** -0.5, mask)) < 2.0 ** -24 * (hd + 2 * L ** 0.5 + 8)


@pytest.mark.parametrize("hd", [4, 8])
@pytest.mark.parametrize("T", [1, 2])
def test_attention_f32_narrow_shift(hd, T):
    H, W, L = 18, 36, 162 * T
    qkv = _qkv(4, L, 32, T)
    o = nsw.ops.window_attention(qkv, 32 // hd, hd ** -0.5, geometry=(H, W, (9, 18), (4, 9), T))
    r = torch.arange(L, device="cuda:0") % 162 // 18 >= 5
    mask = torch.zeros(4, L, L, device="cuda:0")
    mask[2:] = torch.where(r[:, None] != r[None], -100.0, 0.0)
    assert _rel(o, _ref(qkv, 32 // hd, hd ** -0.5, mask)) < 2.0 ** -24 * (hd + 2 * L ** 0.5 + 8)
