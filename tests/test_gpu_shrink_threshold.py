"""ISTA / FISTA refuse a shrinkage threshold that is not positive (its step would
divide 0 by 0), with the steps inside the convolution's passes as apart from them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lam", [0.0, -1e-3, float("nan")])
@pytest.mark.parametrize("solver", ["ISTA", "FISTA"])
@pytest.mark.parametrize("kind,n", [("c", 300), ("c", 16384), ("t", 9001), ("apart", 300)])
def test_refused(kind, n, solver, lam):
    import torch

    import fastmat_amd as fm
    from fastmat_amd import algorithms as fma
    rng = np.random.default_rng(n)
    g = (rng.standard_normal(2 * n - 1) + 1j * rng.standard_normal(2 * n - 1)).astype(np.complex64)
    A = fm.Toeplitz(g[:n], g[n:]) if kind == "t" else fm.Circulant(g[:n])
    if kind == "apart":
        A = fm.Product(A, fm.Eye(n))
    A._largestSV = 8.0 * n
    b = torch.from_numpy(g[:n].reshape(-1, 1).copy()).cuda()
    print("threshold", kind, n, solver, lam, flush=True)
    alg = getattr(fma, solver)(A, numLambda=lam, numMaxSteps=3)
    with pytest.raises(ValueError):
        alg.process(b)
