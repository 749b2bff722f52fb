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
    parts' own rounding and the store (4 U); rows scaled down to fp16 add at
    most 2^-29 of the row's maximum per value."""
    y = _linear(x, w).double()
    xd, wd = x.double(), w.double()
    want = xd @ wd.t()
    mag = xd.abs() @ wd.abs().t()
    K = x.shape[1]
    slack = 2.0 ** -29 * (xd.abs().amax(1, keepdim=True) * wd.abs().sum(1)[None] +
                          xd.abs().sum(1, keepdim=True) * wd.abs().amax(1)[None])
    assert ((y - want).abs() <= U * (K / 8 + 4) * mag + slack).all()


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
