"""The fp32 GEMM on split 16-bit operands: accuracy against 64 bits at the edges
of its k stages and tiles, and values that the split parts do not hold."""
import pytest
import torch

import nsw
from nsw import _lib

pytestmark = pytest.mark.gpu

U = 2.0 ** -24          # fp32 unit roundoff


def _dev():
    return torch.device("cuda:0")


def _linear(x, w):
    return nsw.ops.linear(x, w, None, None, epilogue=_lib.NSW_EPI_NONE)


def _check(x, w):
    """Each element within U (K / 8 + 4) of sum |x||w|, a quarter of the bound
    that any order of K fp32 additions and multiplications keeps (K U) plus the
    parts' own rounding and the store (4 U)."""
    y = _linear(x, w).double()
    xd, wd = x.double(), w.double()
    want = xd @ wd.t()
    mag = xd.abs() @ wd.abs().t()
    assert ((y - want).abs() <= U * (x.shape[1] / 8 + 4) * mag).all()
    return ((y - want).norm() / want.norm()).item()


# K: one half stage, 1.5 stages, both sides of the two- / three-part line, an
# odd count of half stages past it, a long sum; M, N: below, at and past a tile
@pytest.mark.parametrize("K", [16, 48, 112, 128, 144, 1024])
@pytest.mark.parametrize("M,N", [(1, 8), (257, 264), (300, 520)])
def test_split_gemm_matches_64_bits(M, N, K):
    g = torch.Generator(device=_dev()).manual_seed(M + K)
    x = torch.randn(M, K, generator=g, device=_dev())
    w = 0.02 * torch.randn(N, K, generator=g, device=_dev())
    _check(x, w)


@pytest.mark.parametrize("K", [48, 256])
@pytest.mark.parametrize("case", ["tiny", "huge", "zero_start", "zero_rows", "small_start", "wide_rows"])
def test_split_gemm_scales(case, K):
    """Row magnitudes far from one and within a row: the scale of a row comes from
    its first 32 k (zero there: scanned; 2^20 times larger later: three parts)."""
    g = torch.Generator(device=_dev()).manual_seed(5)
    x = torch.randn(260, K, generator=g, device=_dev())
    w = torch.randn(272, K, generator=g, device=_dev())
    if case == "tiny":
        x *= 1e-18
        w *= 1e-12
    elif case == "huge":
        x *= 1e18
        w *= 1e15
    elif case == "zero_start":
        x[::3, :32] = 0
        w[1::3, :32] = 0
        x[::3] *= 1e-9
    elif case == "zero_rows":
        x[5:200] = 0
        w[::2] = 0
    elif case == "small_start":
        x[::5, :32] *= 2.0 ** -20
    else:
        x *= torch.exp2(torch.randint(-20, 20, (260, 1), generator=g, device=_dev()).float())
        w *= torch.exp2(torch.randint(-20, 20, (272, 1), generator=g, device=_dev()).float())
    _check(x, w)


# Values far above or below the rest of their row, where the other operand is
# zero or small, so that the rest of the row is the result: one column inside the
# first 32 k (every place in a lane's 4), after them and in a half stage, columns
# all along the row, single elements (a few listed units of a tile) and every
# element spread over 2^80.  Bound as _check; also the 2-norm within what a chain
# of K fp32 roundings of normal values gives (U sqrt(K), measured 5.7e-7 with the
# fp32 matrix instruction at K = 1024).
@pytest.mark.parametrize("K", [128, 144, 1040])
@pytest.mark.parametrize("ratio", [3e2, 1e4, 1e6, 1e10, 1e-4, 1e-9])
@pytest.mark.parametrize("where", ["0", "3", "29", "mid", "last", "eighths", "halves", "elements", "spread"])
def test_split_gemm_outliers(where, ratio, K):
    g = torch.Generator(device=_dev()).manual_seed(K)
    x = torch.randn(260, K, generator=g, device=_dev())
    w = 0.02 * torch.randn(272, K, generator=g, device=_dev())
    tol = U * K ** 0.5
    if where == "elements":
        x[torch.randint(260, (9,), generator=g, device=_dev()), torch.randint(K, (9,), generator=g, device=_dev())] *= ratio
        w[torch.randint(272, (9,), generator=g, device=_dev()), torch.randint(K, (9,), generator=g, device=_dev())] *= ratio
        _check(x, w)
        return
    if where == "spread":
        x *= torch.exp2(torch.randint(-40, 40, (K,), generator=g, device=_dev()).float())
        w *= torch.exp2(torch.randint(-40, 40, (K,), generator=g, device=_dev()).float()) * ratio
        _check(x, w)
        return
    cols = {"0": [0], "3": [3], "29": [29], "mid": [K // 2 + 1], "last": [K - 1], "eighths": list(range(5, K, 8)),
            "halves": list(range(0, K, 2))}[where]
    for zero in (True, False):
        a, b = x.clone(), w.clone()
        a[:, cols] = ratio * a[:, cols].abs().clamp_min(0.1)
        b[:, cols] = 0 if zero else b[:, cols] / ratio
        assert _check(a, b) <= tol
        a, b = x.clone(), w.clone()
        b[:, cols] = ratio * b[:, cols].abs().clamp_min(0.002)
        a[:, cols] = 0 if zero else a[:, cols] / ratio
        assert _check(a, b) <= tol


# One value of a tile far below the rest of its row, and a large one of the other
# operand at the same k (which has no parts, or is inside the window), where the
# results are as small as the one product (all other weights zero) or larger.
@pytest.mark.parametrize("small", [3e-6, 1e-7, 1e-9, 1e-20])
@pytest.mark.parametrize("other", [1.0, 1e3, 1e9])
@pytest.mark.parametrize("rest", [0.0, 1e-6, 1.0])
def test_split_gemm_single_small(small, other, rest):
    K = 256
    g = torch.Generator(device=_dev()).manual_seed(9)
    x = 0.5 + torch.rand(64, K, generator=g, device=_dev())
    w = (0.5 + torch.rand(128, K, generator=g, device=_dev())) * torch.where(
        torch.rand(128, K, generator=g, device=_dev()) < 0.5, -1.0, 1.0)
    w[:, 32:] *= rest
    w[:, :32] *= rest if rest < 1 else 1
    w[5:9, 77] = 0.7 * other
    x[3, 77] = 1.3 * small
    _check(x, w)
    _check(w, torch.cat([x, x]))


@pytest.mark.parametrize("where", ["x", "w", "both"])
def test_split_gemm_one_term(where):
    """Rows with one weight each (a selection): each result is one product, whose
    operands may be the smallest of their rows."""
    K = 1024
    g = torch.Generator(device=_dev()).manual_seed(7)
    sel = torch.zeros(264, K, device=_dev())
    sel[torch.arange(264), torch.randperm(K, generator=g, device=_dev())[:264]] = 0.7
    full = torch.randn(304, K, generator=g, device=_dev())
    full *= torch.exp2(-torch.randint(0, 50, (304, K), generator=g, device=_dev()).float())
    x, w = (full, sel) if where == "x" else (sel, full) if where == "w" else (full, full[:264] * sel.ne(0))
    _check(x, w)


@pytest.mark.parametrize("K", [48, 256])
def test_split_gemm_non_finite(K):
    """Infinities, NaN and the largest fp32 values give what fp32 arithmetic gives."""
    g = torch.Generator(device=_dev()).manual_seed(6)
    x = torch.rand(300, K, generator=g, device=_dev()) + 0.5
    w = torch.rand(264, K, generator=g, device=_dev()) + 0.5
    x[7, 3] = float("inf")
    x[9, K - 1] = -float("inf")
    x[11, 40] = float("nan")
    x[13] = 0
    x[13, 1] = torch.finfo(torch.float32).max    # bf16 rounds it to infinity
    w[:, 1] = 0.5
    y = _linear(x, w)
    assert (y[7] == float("inf")).all() and (y[9] == -float("inf")).all() and torch.isnan(y[11]).all()
    assert (y[13] == torch.finfo(torch.float32).max * 0.5).all()
    keep = torch.ones(300, dtype=torch.bool, device=_dev())
    keep[[7, 9, 11, 13]] = False
    want = x[keep].double() @ w.double().t()
    assert ((y[keep].double() - want).abs() <= U * (K / 8 + 4) * want).all()


def _tile_rows(M, N, K, dtype, row_epilogue=0):
    code = _lib.NSW_DTYPE_F32 if dtype == torch.float32 else _lib.NSW_DTYPE_BF16
    return _lib.lib().nsw_gemm_tile_rows(M, N, K, row_epilogue, code)


# The fp32 loops on each tile (64 x 128, 128 x 128, 256 x 256: other waves,
# copies, splits and barriers), rows and columns that end inside a tile, K with an
# odd half stage, on three parts (112), two (144, 272) and from one to the other.
@pytest.mark.parametrize("K", [112, 144, 272])
@pytest.mark.parametrize("M,N,rows", [(301, 264, 64), (5000, 1160, 128), (8100, 3080, 256)])
@pytest.mark.parametrize("case", ["normal", "outliers", "singles", "spread", "later", "zero_start", "non_finite"])
def test_split_gemm_on_each_tile(case, M, N, rows, K):
    assert _tile_rows(M, N, K, torch.float32) == rows
    g = torch.Generator(device=_dev()).manual_seed(M + K)
    rnd = lambda *s: torch.randn(*s, generator=g, device=_dev())
    x, w = rnd(M, K), 0.02 * rnd(N, K)
    if case == "outliers":                 # a column of x, one of w: every row block of a stage
        x[:, 3], w[:, 3] = 1e5, 0
        w[:, K - 5], x[:, K - 5] = 1e3, 0
    elif case == "singles":                # two single small values and a large one in most tiles
        x[::37, 20] = 1e-8
        w[::67, K - 9] = -1e-9
        x[11::131, 7] = 3e7
    elif case == "spread":
        x *= torch.exp2(torch.randint(-30, 30, (K,), generator=g, device=_dev()).float())
        w *= torch.exp2(torch.randint(-30, 30, (K,), generator=g, device=_dev()).float())
    elif case == "later":                  # two parts first, three from a later stage on
        x[:, K - 20:] *= torch.exp2(torch.randint(-40, 0, (M, 20), generator=g, device=_dev()).float())
    elif case == "zero_start":
        x[::3, :40] = 0
        w[1::3, :K - 3] = 0
    elif case == "non_finite":
        x[M - 2, K - 1], w[N - 3, 1] = float("inf"), float("nan")
        y = _linear(x, w)
        assert not torch.isfinite(y[M - 2]).any() and torch.isnan(y[:, N - 3]).all()
        x[M - 2, K - 1], w[N - 3, 1] = 0, 0
        clean = _linear(x, w)
        y[M - 2], y[:, N - 3] = clean[M - 2], clean[:, N - 3]
        # the values were outside the window or not: other rows differ in how one
        # unit of the tile was listed, by no more than the bound
        mag = x.double().abs() @ w.double().abs().t()
        assert ((y.double() - clean.double()).abs() <= 2 * U * (K / 8 + 4) * mag).all()
    _check(x, w)


@pytest.mark.parametrize("M,N", [(301, 264), (5000, 1160), (8100, 3080)])
def test_listed_units_repeat_bit_for_bit(M, N):
    """Several corrections meet in most results; their order is not the waves'."""
    K = 512
    g = torch.Generator(device=_dev()).manual_seed(10)
    x = torch.randn(M, K, generator=g, device=_dev())
    w = 0.02 * torch.randn(N, K, generator=g, device=_dev())
    for i, k in enumerate((70, 200, 330, 460)):
        x[i::64, k] = 1e6 * (i + 1)
        w[i::128, k + 33] = 1e4 * (i + 1)
        w[:, k], x[:, k + 33] = 1e-6 * w[:, k], 1e-4 * x[:, k + 33]
    first = _linear(x, w)
    _check(x, w)
    for _ in range(6):
        assert torch.equal(_linear(x, w), first)


# Shapes on both sides of the tile rule (64- / 32-row tiles; at 8100 x 1024 rows
# 128- / 64-row tiles; then 256), with rows and columns that end
# inside a tile, odd k stages, and every kind of write-out: plain, GELU,
# residual, the head norm, window maps with row sums, the head's image.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,W,C", [(9, 18, 96), (27, 54, 128), (45, 108, 192), (90, 90, 512), (90, 90, 1024),
                                   (90, 180, 1024)])
def test_tile_sizes(dtype, H, W, C):
    f32 = dtype == torch.float32
    mid, small = C == 1024 and H == W, C < 1024
    assert _tile_rows(H * W, C, C, dtype) == (64 if small else 128 if mid else 256)
    assert _tile_rows(H * W, C, C, dtype, 1) == ((64 if f32 else 32) if small else (128 if f32 else 64) if mid else 256)
    g = torch.Generator(device=_dev()).manual_seed(H + C)
    rnd = lambda *s: torch.randn(*s, generator=g, device=_dev()).to(dtype)
    M, hd = H * W, 32
    x, b, r = rnd(M, C), rnd(C), rnd(M, C)
    w = (0.05 * torch.randn(C, C, generator=g, device=_dev())).to(dtype)
    w3, b3 = (0.05 * torch.randn(3 * C, C, generator=g, device=_dev())).to(dtype), rnd(3 * C)
    qn, kn = rnd(hd), rnd(hd)
    d = lambda t: t.double()
    tol = 1e-6 if f32 else 5e-3     # U sqrt(K) / 2 <= 1e-6 (a chain of K roundings: U sqrt(K)); bf16 store 2^-8 / sqrt(3)

    def close(y, want):
        e = (d(y) - want).norm() / want.norm()
        assert e < tol, float(e)

    base = d(x) @ d(w).t()
    close(_linear(x, w), base)
    close(nsw.ops.linear(x, w, b, r), base + d(b) + d(r))
    close(nsw.ops.linear(x, w, b, None, epilogue=_lib.NSW_EPI_BIAS_GELU), torch.nn.functional.gelu(base + d(b)))
    eps = 1e-5
    qkv = (d(x) @ d(w3).t() + d(b3)).view(M, 3, C // hd, hd)
    n = qkv * torch.rsqrt(qkv.pow(2).mean(-1, keepdim=True) + eps)
    want = torch.stack([n[:, 0] * d(qn), n[:, 1] * d(kn), qkv[:, 2]], 1).view(M, 3 * C)
    close(nsw.ops.qkv_projection(x, w3, b3, qn, kn, C // hd, eps), want)
    # window rows to the next block's window order, with row sums
    y, ss = nsw.ops.linear_remap_residual(x, w, b, r, 2, image=(1, 1, H, W), window_size=(9, 18), shift_size=(0, 0),
                                          next_shift=(4, 9))
    rows = torch.arange(M, device=_dev()).view(H // 9, W // 18, 9, 18).permute(0, 2, 1, 3).reshape(H, W)
    nxt = torch.roll(rows, (-4, -9), (0, 1)).view(H // 9, 9, W // 18, 18).permute(0, 2, 1, 3).reshape(-1)
    want = (base + d(b) + d(r))[nxt]
    close(y, want)
    assert torch.allclose(ss.double().sum(1), d(y).pow(2).sum(1), rtol=1e-5)
    # tokens to image planes
    for p in (2, 16):
        ch = 5 * 4 // p if p < 16 else 1
        wh = (0.05 * torch.randn(ch * p * p, C, generator=g, device=_dev())).to(dtype)
        img = nsw.ops.head_unpatchify(x, wh, 1, ch, H * p, W * p, p)
        want = (d(x) @ d(wh).t()).view(H, W, ch, p, p).permute(2, 0, 3, 1, 4).reshape(1, 1, ch, H * p, W * p)
        close(img, want)


@pytest.mark.parametrize("K", [48, 112, 272])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_non_finite_rows_leave_the_others(value, K):
    """One row of x and one of w that are not finite: every other result keeps its
    bits, also those of the same 16 x 16 block."""
    g = torch.Generator(device=_dev()).manual_seed(8)
    x = torch.randn(300, K, generator=g, device=_dev())
    w = torch.randn(264, K, generator=g, device=_dev())
    clean = _linear(x, w)
    x[37, K // 2] = value
    w[130, 5] = value
    y = _linear(x, w)
    assert not torch.isfinite(y[37]).any() and not torch.isfinite(y[:, 130]).any()
    y[37], y[:, 130] = clean[37], clean[:, 130]
    assert torch.equal(y, clean)
