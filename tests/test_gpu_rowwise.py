"""The row-wise kernels (diagonal, gather, expand, axpby through Product and
Partial) at the edges of their column groups (8), row blocks (64, 256) and grid,
exact in integers; a selection's scatter with repeated and negative indices
against numpy's indexed assignment."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["int8", "int16", "int32", "int64", "complex64", "complex128"])
@pytest.mark.parametrize("n,k", [(1, 1), (63, 7), (64, 8), (65, 9), (257, 17), (1000, 1),
                                 (2, 524301)])
def test_rowwise_edges(n, k, dtype):
    import fastmat_amd as fm
    rng = np.random.default_rng(n + k)

    def ints(*s):
        a = rng.integers(-5, 6, size=s).astype(dtype)
        return a + 1j * rng.integers(-5, 6, size=s).astype(dtype) if a.dtype.kind == "c" else a
    x, d, sigma = ints(n, k), ints(n), rng.permutation(n)
    print("rowwise", n, k, dtype, flush=True)
    D = fm.Diag(d)
    np.testing.assert_array_equal(D.forward(x), (d[:, None] * x).astype(x.dtype))
    np.testing.assert_array_equal(D.backward(x), (np.conj(d)[:, None] * x).astype(x.dtype))
    np.testing.assert_array_equal(fm.Permutation(sigma).forward(x), x[sigma])
    S = (fm.Diag(d) + fm.Permutation(sigma)).forward(x)
    np.testing.assert_array_equal(S, (d[:, None] * x + x[sigma]).astype(S.dtype))
    sel = rng.integers(0, n, size=max(1, n // 2))
    P = fm.Partial(fm.Eye(n), cols=sel)
    full = np.zeros((n, k), dtype=dtype)
    full[sel] = x[:len(sel)]
    np.testing.assert_array_equal(P.forward(x[:len(sel)]), full)
    np.testing.assert_array_equal(P.backward(x), x[sel])


def test_partial_repeated_negative_indices():
    """[-1, 2, 2] passes the constructor's sum check: all three name row 2."""
    import fastmat_amd as fm
    x = np.arange(9, dtype=np.int32).reshape(3, 3)
    sel = np.array([-1, 2, 2])
    P = fm.Partial(fm.Eye(3), cols=sel)
    full = np.zeros((3, 3), dtype=np.int32)
    full[sel] = x
    np.testing.assert_array_equal(P.forward(x), full)
    np.testing.assert_array_equal(P.backward(x), x[sel])
