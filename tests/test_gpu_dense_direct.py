"""Dense products beyond the small-factor kernel (float32, float32 matrices on
complex64 data, complex64, float64, complex128), forward and adjoint, at the
sizes where their tiles, K steps and K splits have edges.

Bound: a sum of K products in precision u, in any order, is off by at most
about K u sum |a_l||x_l| (Higham, Accuracy and Stability, 3.1); a complex
product is four real ones, hence the factor 4 and a few roundings on top.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (m, n, k): single elements, one row or column, one past and one short of
# tiles (16, 32, 64, 128) and K steps (4, 8, 16), rows shorter than a vector,
# and one product of each tile shape
SIZES = [(1, 129, 1), (129, 1, 3), (130, 2, 17), (129, 3, 5), (257, 131, 1), (128, 129, 16),
         (65, 143, 33), (144, 145, 64), (300, 1000, 7), (1000, 333, 40), (515, 260, 129),
         (640, 160, 515), (2050, 130, 1030)]


def _rand(rng, shape, dtype):
    x = rng.standard_normal(shape)
    if np.dtype(dtype).kind == "c":
        x = x + 1j * rng.standard_normal(shape)
    return x.astype(dtype)


@pytest.mark.parametrize("adtype,xdtype", [("float32", "float32"), ("float32", "complex64"),
                                           ("complex64", "complex64"), ("float64", "float64"),
                                           ("complex128", "complex128")])
@pytest.mark.parametrize("m,n,k", SIZES)
def test_dense_direct(m, n, k, adtype, xdtype):
    import fastmat_amd as fm
    rng = np.random.default_rng(m * 7919 + n * 31 + k)
    A = _rand(rng, (m, n), adtype)
    M = fm.Matrix(A)
    wide = np.complex128 if np.dtype(xdtype).kind == "c" else np.float64
    u = np.finfo(np.dtype(xdtype)).eps
    for B, apply in ((A, M.forward), (A.conj().T, M.backward)):
        x = _rand(rng, (B.shape[1], k), xdtype)
        print("dense direct", B.shape, k, adtype, xdtype, flush=True)
        y = apply(x)
        assert y.dtype == np.dtype(xdtype)
        ref = B.astype(wide) @ x.astype(wide)
        bound = 4 * (B.shape[1] + 8) * u * (np.abs(B).astype(np.float64) @
                                            np.abs(x).astype(np.float64))
        assert np.all(np.abs(y - ref) <= bound)


@pytest.mark.parametrize("dtype", ["float32", "float64", "complex128"])
def test_dense_direct_keeps_rows_and_columns_apart(dtype):
    """An infinity or NaN in one row of A or one column of X reaches that row
    or column of the result only (edge tiles read clamped neighbours)."""
    import fastmat_amd as fm
    rng = np.random.default_rng(5)
    m, n, k = 147, 150, 21
    A, x = _rand(rng, (m, n), dtype), _rand(rng, (n, k), dtype)
    A[m - 1, 3] = np.inf
    x[n - 1, k - 1] = np.nan
    y = fm.Matrix(A).forward(x)
    assert np.all(np.isfinite(y[:m - 1, :k - 1]))
    assert np.all(np.isnan(y[:, k - 1])) and not np.any(np.isfinite(y[m - 1]))
