"""A selection's device tables are complete when they are kept: a call on another
stream right after the first one reads them, and a stream capture of one direction
after a warm-up of the other alone neither keeps tables that its kernels have not
filled nor needs what only a running stream gives.

Bounds: a captured call may keep the separate passes, where the eager one selects
inside the transform's: 16 u of the largest output apart, as those two are.  Whole
numbers are equal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _nested(name, n):
    import fastmat_amd as fm
    rng = np.random.default_rng(n)
    if name == "fourier":
        return fm.Fourier(n), np.complex64
    if name == "product":
        d = fm.Diag((rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(np.complex64))
        F = fm.Fourier(n)
        return fm.Product(F.H, d, F), np.complex64
    return fm.Hadamard(n.bit_length() - 1), np.int32


def _data(rows, k, dtype, seed):
    import torch
    rng = np.random.default_rng(seed)
    a = rng.integers(-9, 10, size=(k, rows)).astype(dtype)
    return torch.from_numpy(a).cuda().t()


def _close(got, ref, dtype):
    import torch
    if dtype == np.int32:
        assert torch.equal(got, ref)
    else:
        assert (got - ref).abs().max() <= 16 * 1.2e-7 * ref.abs().max()


def _partial(name, n, both):
    import fastmat_amd as fm
    M, dtype = _nested(name, n)
    rng = np.random.default_rng(n + 1)
    rows = rng.permutation(n)[:n // 3]
    cols = np.sort(rng.permutation(n)[:n // 2]) if both else None
    return lambda: fm.Partial(M, rows=rows, cols=cols), dtype


@pytest.mark.parametrize("adjoint", [False, True])
@pytest.mark.parametrize("both", [False, True])
@pytest.mark.parametrize("name", ["fourier", "product", "hadamard"])
def test_second_stream_right_after_the_first_call(name, both, adjoint):
    import torch
    n, k = 1 << 14, 3
    make, dtype = _partial(name, n, both)
    P = make()
    x = _data(P.numRows if adjoint else P.numCols, k, dtype, 5)
    run = (lambda p: p.backward(x)) if adjoint else (lambda p: p.forward(x))
    ref = run(P)
    torch.cuda.synchronize()
    print("streams", name, both, adjoint, flush=True)
    P = make()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(a):
        torch.cuda._sleep(10_000_000)
        first = run(P)
    with torch.cuda.stream(b):
        second = run(P)
    torch.cuda.synchronize()
    assert torch.equal(first, ref) and torch.equal(second, ref)


@pytest.mark.parametrize("adjoint", [False, True])
@pytest.mark.parametrize("both", [False, True])
@pytest.mark.parametrize("name", ["fourier", "hadamard"])
def test_capture_after_the_other_direction(name, both, adjoint):
    import torch
    n, k = 1 << 14, 3
    make, dtype = _partial(name, n, both)
    P = make()
    run, warm = (P.backward, P.forward) if adjoint else (P.forward, P.backward)
    size, warm_size = (P.numRows, P.numCols) if adjoint else (P.numCols, P.numRows)
    x = _data(size, k, dtype, 7)
    warm(_data(warm_size, k, dtype, 6))
    torch.cuda.synchronize()
    print("capture", name, both, adjoint, flush=True)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = run(x)
    _close(run(x), (make().backward if adjoint else make().forward)(x), dtype)
    for seed in (8, 9, 10):
        x.copy_(_data(x.shape[0], k, dtype, seed))
        ref = run(x)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        _close(y, ref, dtype)


@pytest.mark.parametrize("adjoint", [False, True])
@pytest.mark.parametrize("selected", [False, True])
def test_capture_of_a_product_after_the_other_direction(selected, adjoint):
    """F^H D F with a complex D: one direction multiplies by D, the other by its
    conjugate, a table of its own inside the passes."""
    import torch

    import fastmat_amd as fm
    n, k = 1 << 14, 3
    rng = np.random.default_rng(n)
    d = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(np.complex64)
    F = fm.Fourier(n)

    def make():
        M = fm.Product(F.H, fm.Diag(d), F)
        return fm.Partial(M, rows=np.arange(0, n, 3)) if selected else M
    P = make()
    run, warm = (P.backward, P.forward) if adjoint else (P.forward, P.backward)
    size, warm_size = (P.numRows, P.numCols) if adjoint else (P.numCols, P.numRows)
    x = _data(size, k, np.complex64, 7)
    warm(_data(warm_size, k, np.complex64, 6))
    torch.cuda.synchronize()
    print("capture product", selected, adjoint, flush=True)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = run(x)
    Q = make()
    _close(run(x), (Q.backward if adjoint else Q.forward)(x), np.complex64)
    for seed in (8, 9, 10):
        x.copy_(_data(size, k, np.complex64, seed))
        ref = run(x)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        _close(y, ref, np.complex64)
