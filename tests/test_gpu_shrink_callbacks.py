"""ISTA / FISTA callbacks against the run's own state: a write to the iterate counts
however it is made, a matrix set by a callback is the next step's.

Bound: the solver bar (1e-4 relative in single precision)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _problem(kind, n, k):
    import torch

    import fastmat_amd as fm
    rng = np.random.default_rng(n + k)
    g = (rng.standard_normal(2 * n - 1) + 1j * rng.standard_normal(2 * n - 1)).astype(np.complex64)
    g /= np.sqrt(n)  # (a product of the size of its operand: what the point was shows)
    A = fm.Circulant(g[:n]) if kind == "c" else fm.Toeplitz(g[:n], g[n:])
    A._largestSV = 8.0
    b = rng.standard_normal((n, k)) + 1j * rng.standard_normal((n, k))
    return A, torch.from_numpy(b.astype(np.complex64)).cuda()


def _ista_step(alg, A, b, x):
    L, alpha = alg.numL, alg.numL * alg.numLambda * 0.5
    step = x - L * A.backward(A.forward(x) - b)
    m = (step.abs() - alpha).clamp(min=0)
    return step * (m / (m + alpha))


def _write_data(x):
    x.data.mul_(0.5)


def _write_dlpack(x):
    import torch
    torch.utils.dlpack.from_dlpack(torch.view_as_real(x)).mul_(0.5)


def _write_library(x):
    """One of the library's own kernels, on the raw address."""
    from fastmat_amd import _device as D
    from fastmat_amd import _lib
    n, k = x.shape
    _lib.call("fm_axpby", _lib.FM_COMPLEX64, n, k, _lib.dvec(0.5), x.data_ptr(), n, 0,
              _lib.dvec(0.0), x.data_ptr(), n, D.stream())


@pytest.mark.parametrize("write", [_write_data, _write_dlpack, _write_library])
@pytest.mark.parametrize("kind,n,k", [("c", 300, 2), ("c", 16384, 1), ("t", 9001, 2)])
def test_a_write_that_torch_does_not_count(kind, n, k, write):
    from fastmat_amd import algorithms as fma
    A, b = _problem(kind, n, k)
    seen = {}

    def callback(a):
        if a.numStep == 2:
            write(a.arrX)
            seen["x"] = a.arrX.clone()
        if a.numStep == 3:
            seen["next"] = a.arrX.clone()
    print("write", kind, n, k, write.__name__, flush=True)
    alg = fma.ISTA(A, numLambda=1e-3, numMaxSteps=5)
    alg.cbStep = callback
    alg.process(b)
    ref = _ista_step(alg, A, b, seen["x"])
    assert (seen["next"] - ref).abs().max() <= 1e-4 * ref.abs().max()


@pytest.mark.parametrize("other", ["circulant", "product"])
@pytest.mark.parametrize("solver", ["ISTA", "FISTA"])
@pytest.mark.parametrize("kind,n,k", [("c", 300, 2), ("c", 16384, 1)])
def test_a_callback_that_sets_the_matrix(kind, n, k, solver, other):
    """The step after takes the products of the matrix that is set, the one before
    its own: a run that changes over to 3 A equals the steps by separate applies."""
    import fastmat_amd as fm
    from fastmat_amd import algorithms as fma
    A, b = _problem(kind, n, k)
    three = np.full(n, 3, np.complex64)
    B = (fm.Circulant((3 * A._gen128).astype(np.complex64)) if other == "circulant"
         else fm.Product(fm.Diag(three), A))
    runs = []
    for first in (A, fm.Product(A, fm.Eye(n))):
        first._largestSV = 24.0

        def callback(a):
            if a.numStep == 2:
                a.fmatA = B
        print("set", solver, kind, n, k, other, type(first).__name__, flush=True)
        alg = getattr(fma, solver)(first, numLambda=1e-3, numMaxSteps=6)
        alg.cbStep = callback
        runs.append(alg.process(b).clone())
        assert alg.numStep == 5
    assert (runs[0] - runs[1]).abs().max() <= 1e-4 * runs[1].abs().max()


@pytest.mark.parametrize("solver", ["ISTA", "FISTA"])
def test_less_than_one_step(solver):
    """0.5 steps, which the check lets through, are one."""
    import torch

    from fastmat_amd import algorithms as fma
    A, b = _problem("c", 300, 2)
    runs = [getattr(fma, solver)(A, numLambda=1e-3, numMaxSteps=s) for s in (0.5, 1)]
    x, ref = (alg.process(b) for alg in runs)
    assert torch.equal(x, ref) and runs[0].numStep == 0
