"""Row-major operands that torch's copy takes to columns faster than the library's
transpose stay with it, whatever their size: few rows, and short rows of small
elements."""
import pytest


@pytest.mark.parametrize("esz,n,k", [(4, 2, 3000000), (8, 32, 1000000), (1, 8, 1 << 26),
                                     (16, 128, 1000000), (1, 1 << 20, 24), (2, 1 << 20, 17),
                                     (4, 1 << 20, 5), (16, 1 << 18, 5)])
def test_torch(esz, n, k):
    from fastmat_amd import _device as D
    assert esz * n * k < D._transpose_bytes(esz, n, k)


@pytest.mark.parametrize("esz,n,k", [(4, 1 << 20, 32), (8, 48, 100000), (16, 1 << 18, 32),
                                     (1, 1 << 20, 16), (1, 1 << 20, 28), (1, 700000, 17), (1, 1 << 21, 20), (2, 1 << 20, 24),
                                     (4, 1 << 22, 2), (16, 1 << 20, 5)])
def test_library(esz, n, k):
    from fastmat_amd import _device as D
    assert esz * n * k >= D._transpose_bytes(esz, n, k)
