"""The GEMM's tile rule as the host query states it (no GPU)."""
import pytest

from nsw import _lib


def _rows(M, N, K, row_epilogue=0, dtype=_lib.NSW_DTYPE_F32):
    return _lib.lib().nsw_gemm_tile_rows(M, N, K, row_epilogue, dtype)


@pytest.mark.parametrize("dtype,row,sizes", [(_lib.NSW_DTYPE_F32, 0, {64, 128, 256}), (_lib.NSW_DTYPE_F32, 1, {64, 128, 256}),
                                             (_lib.NSW_DTYPE_BF16, 0, {64, 128, 256}), (_lib.NSW_DTYPE_BF16, 1, {32, 64, 256})])
def test_every_tile_is_chosen(dtype, row, sizes):
    seen = {_rows(M, N, K, row, dtype) for M in (1, 648, 5000, 8100, 12000, 64800) for N in (8, 264, 1024, 3072)
            for K in (32, 128, 1024)}
    assert seen == sizes


def test_large_products_keep_the_large_tile():
    for dtype in (_lib.NSW_DTYPE_F32, _lib.NSW_DTYPE_BF16):
        for N, K in ((3072, 1024), (1024, 1024), (4096, 1024), (1024, 4096)):
            for row in (0, 1):
                assert _rows(64800, N, K, row, dtype) == 256


def test_refused():
    assert _rows(0, 8, 32) == 0 and _rows(8, -8, 32) == 0 and _rows(8, 8, 0) == 0 and _rows(8, 8, 32, 0, 99) == 0
