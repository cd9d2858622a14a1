"""Diag factors next to a Fourier factor of a Product run inside the transform's
passes: every arrangement (before, after, both sides, around F and F^H), forward
and adjoint, one- and multi-pass orders, both precisions, real and complex
diagonals, against the factors applied one by one and against FP64; and the
arrangements that keep the separate path.

Bound against the separate path: the same products in the same precision, at
most a few roundings per element apart: 16 u of the largest output."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _one_by_one(factors, x, adjoint):
    for f in (factors if adjoint else factors[::-1]):
        x = f.backward(x) if adjoint else f.forward(x)
    return x


@pytest.mark.parametrize("dtype", ["complex64", "complex128"])
@pytest.mark.parametrize("n,k", [(1, 2), (2, 1), (64, 3), (1024, 17), (8192, 2), (16384, 3),
                                 (1 << 18, 2), (48, 3)])
def test_product_with_diagonals(n, k, dtype):
    import fastmat_amd as fm
    from fastmat_amd import product
    rng = np.random.default_rng(n + k)

    def rand(*s):
        return (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(dtype)
    F = fm.Fourier(n, dtype=np.dtype(dtype))
    d1, d2 = fm.Diag(rand(n)), fm.Diag(rng.standard_normal(n).astype(np.float32))
    x = rand(n, k)
    calls = []
    run = F._run_diag
    F._run_diag = lambda *a: (calls.append(1), run(*a))[1]
    u = np.finfo(np.dtype(dtype)).eps
    for factors in ((F, d1), (d1, F), (d1, F, d2), (F.H, d1, F), (d2, F.H, d1, F, d2), (d1, F.H),
                    (F.H, d2), (d1, d2, F)):
        P = fm.Product(*factors)
        for adjoint in (False, True):
            calls.clear()
            print("product", n, k, dtype, [type(f).__name__ for f in factors], adjoint, flush=True)
            got = P.backward(x) if adjoint else P.forward(x)
            assert bool(calls) == (n & (n - 1) == 0)
            ref = _one_by_one(factors, x, adjoint)
            assert got.dtype == ref.dtype == np.dtype(dtype)
            assert np.max(np.abs(got - ref)) <= 16 * u * np.max(np.abs(ref))
    # 64 bits from plain numpy
    ref = np.fft.fft(d1.vecD.astype(np.complex128)[:, None] * x, axis=0)
    bar = 1e-5 if dtype == "complex64" else 1e-12
    assert np.max(np.abs(fm.Product(F, d1).forward(x) - ref)) <= bar * np.max(np.abs(ref))
    assert product._as_fourier(F.T)[0] is None


def test_diagonals_of_another_type_stay_separate():
    """A diagonal that widens the data, or data that is not of the compute type,
    keeps the factors' own type rules."""
    import fastmat_amd as fm
    rng = np.random.default_rng(3)
    F = fm.Fourier(32)
    d64 = fm.Diag(rng.standard_normal(32))
    P = fm.Product(F, d64)
    for x in (rng.standard_normal((32, 2)).astype(np.float32),
              (rng.standard_normal((32, 2)) + 0j).astype(np.complex64),
              rng.integers(-3, 4, size=(32, 2)).astype(np.int8)):
        ref = _one_by_one((F, d64), x.astype(np.result_type(x, P.dtype)), False)
        got = P.forward(x)
        assert got.dtype == ref.dtype
        np.testing.assert_allclose(got, ref, rtol=0, atol=1e-12 * np.max(np.abs(ref)))
