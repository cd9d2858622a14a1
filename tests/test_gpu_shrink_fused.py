"""ISTA / FISTA on Circulant and Toeplitz operators, whose whole step is one call
(residual and shrinkage inside the convolution's passes): one-pass and
multi-pass lengths, square and rectangular, single and double precision, one
and several columns, against the oracle's loop on the dense matrix (small) or
on 64-bit FFT products (long).

Tolerance: the project's solver bar (test_gpu_algorithms.py): 1e-4 relative in
single precision, 1e-9 in double.  The threshold (5e-5 of the data's scale) is
below it: a value that rounding puts on the other side changes by no more."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _reference(forward, adjoint, n, b, L, lam, steps, momentum):
    """ISTA.py:152-168 / FISTA.py:154-178 with 64-bit products."""
    alpha = L * lam * 0.5
    x = np.zeros((n, b.shape[1]), dtype=np.complex128)
    y, t = x, 1.0
    for _ in range(steps):
        step = y - L * adjoint(forward(y) - b)
        m = np.maximum(np.abs(step) - alpha, 0)
        old, x = x, m / (m + alpha) * step
        t0, t = t, (1 + np.sqrt(1 + 4 * t * t)) / 2
        y = x + (t0 - 1) / t * (x - old) if momentum else x
    return np.where(x != 0, step, x)


@pytest.mark.parametrize("solver", ["ISTA", "FISTA"])
@pytest.mark.parametrize("dtype", ["complex64", "complex128"])
@pytest.mark.parametrize("kind,m,n,k", [
    ("c", 32, 32, 1), ("c", 100, 100, 3), ("t", 130, 77, 2), ("c", 4096, 4096, 2),
    ("t", 700, 1500, 5), ("c", 8192, 8192, 3), ("c", 5000, 5000, 2), ("c", 16384, 16384, 1),
    ("t", 30011, 20003, 3), ("c", 1 << 18, 1 << 18, 2)])
def test_fused_step(solver, dtype, kind, m, n, k):
    import torch

    import fastmat_amd as fm
    from fastmat_amd import algorithms as fma
    from oracle import fast64
    rng = np.random.default_rng(m + 3 * n + k)

    def rand(*s):
        return (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(dtype)
    if kind == "c":
        g = rand(n) / n
        A = fm.Circulant(g)
        fwd, adj = (lambda v, a=a: fast64.circulant(g, v, adjoint=a) for a in (False, True))
    else:
        g = rand(m + n - 1) / n
        A = fm.Toeplitz(g[:m], g[m:])
        fwd, adj = (lambda v, a=a: fast64.toeplitz(g, m, v, adjoint=a) for a in (False, True))
    x0 = np.where(rng.random((n, k)) < 0.1, rand(n, k), 0)
    b = fwd(x0).astype(dtype)
    # an upper bound of the largest singular value serves the recursion as well
    A._largestSV = float(np.max(np.abs(np.fft.fft(g.astype(np.complex128)))))
    L, lam, steps = 1.0 / A._largestSV ** 2, 1e-4 * A._largestSV ** 2, 7
    alg = getattr(fma, solver)(A, numLambda=lam, numMaxSteps=steps)
    assert alg._fused(np.dtype(dtype), k) is not None
    print("fused", solver, dtype, kind, m, n, k, flush=True)
    got = alg.process(torch.from_numpy(b).cuda())
    ref = _reference(fwd, adj, n, b.astype(np.complex128), L, lam, steps, solver == "FISTA")
    err = np.max(np.abs(got.cpu().numpy() - ref)) / np.max(np.abs(ref))
    assert err < (1e-4 if dtype == "complex64" else 1e-9)
    # the callback loop writes every step's state and gives the same result
    seen = []
    alg = getattr(fma, solver)(A, numLambda=lam, numMaxSteps=steps)
    alg.cbStep = lambda a: seen.append(a.arrStep.clone())
    assert torch.equal(alg.process(torch.from_numpy(b).cuda()), got)
    assert len(seen) == steps and torch.equal(seen[-1], alg.arrStep)
