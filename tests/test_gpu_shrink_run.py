"""ISTA / FISTA runs of many steps in few calls: the steps of one call and across
calls are the steps taken one by one (a step leaves its next point's column
transform for the step after it), and a callback that writes to the iterate is seen
by the next step.

The steps one by one run the same kernels on the same numbers: equal bits.  After a
write the point's transform is formed by another kernel, as it is for a first step:
the solver bar (1e-4 relative in single precision)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _problem(kind, n, k):
    import torch

    import fastmat_amd as fm
    rng = np.random.default_rng(n + k)
    g = (rng.standard_normal(2 * n - 1) + 1j * rng.standard_normal(2 * n - 1)).astype(np.complex64)
    A = fm.Circulant(g[:n] / n) if kind == "c" else fm.Toeplitz(g[:n] / n, g[n:] / n)
    A._largestSV = 2.0
    b = rng.standard_normal((n, k)) + 1j * rng.standard_normal((n, k))
    return A, torch.from_numpy(b.astype(np.complex64)).cuda()


@pytest.mark.parametrize("solver", ["ISTA", "FISTA"])
@pytest.mark.parametrize("steps", [1, 2, 63, 64, 65, 130])
@pytest.mark.parametrize("kind,n,k", [("c", 300, 2), ("c", 16384, 1), ("t", 9001, 2)])
def test_many_steps_are_the_steps_one_by_one(kind, n, k, steps, solver):
    import torch

    from fastmat_amd import algorithms as fma
    A, b = _problem(kind, n, k)
    cls = getattr(fma, solver)
    print("run", solver, kind, n, k, steps, flush=True)
    alg = cls(A, numLambda=1e-3, numMaxSteps=steps)
    got = alg.process(b).clone()
    assert alg.numStep == steps - 1 and torch.isfinite(torch.view_as_real(got)).all()
    count = []
    one = cls(A, numLambda=1e-3, numMaxSteps=steps)
    one.cbStep = lambda a: count.append(a.numStep)
    assert torch.equal(one.process(b), got) and count == list(range(steps))


@pytest.mark.parametrize("kind,n,k", [("c", 300, 2), ("c", 16384, 1), ("t", 9001, 2)])
def test_a_callback_that_writes_the_iterate(kind, n, k):
    """ISTA's point is the iterate: scaling it in a callback is a restart from there."""
    from fastmat_amd import algorithms as fma
    A, b = _problem(kind, n, k)
    seen = {}

    def write(a):
        if a.numStep == 2:
            a.arrX.mul_(0.5)
            seen["x"] = a.arrX.clone()
        if a.numStep == 3:
            seen["next"] = a.arrX.clone()
    alg = fma.ISTA(A, numLambda=1e-3, numMaxSteps=5)
    alg.cbStep = write
    alg.process(b)
    x = seen["x"]
    L, alpha = alg.numL, alg.numL * alg.numLambda * 0.5
    step = x - L * A.backward(A.forward(x) - b)
    m = (step.abs() - alpha).clamp(min=0)
    ref = step * (m / (m + alpha))
    assert (seen["next"] - ref).abs().max() <= 1e-4 * ref.abs().max()
