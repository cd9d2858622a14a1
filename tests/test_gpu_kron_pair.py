"""The fused last pair of a Kron product (Circulant x dense float32 on complex64
data): every compiled shape, slab counts around the two workgroups a slab takes
and a partly filled last one, forward and adjoint, against FP64.

Bound: 1e-5 of the largest output, the single-precision bar of the other FFT
and dense tests (a 128-term product and two 128-point transforms are off by a
few times 1e-7)."""
import numpy as np
import pytest
import scipy.linalg as sla

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [64, 128])
@pytest.mark.parametrize("m", [64, 96, 128])
@pytest.mark.parametrize("f,k", [(1, 1), (2, 1), (4, 3), (8, 37)])
def test_kron_pair_shapes(n, m, f, k):
    import torch

    import fastmat_amd as fm
    from fastmat_amd import kron as fkron
    from oracle import accept, fast64
    rng = np.random.default_rng(n + 3 * m + 5 * f + 7 * k)

    def c64(*s):
        return (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64)
    c, A = c64(n), rng.standard_normal((m, m)).astype(np.float32)
    K = fm.Kron(fm.Fourier(f), fm.Circulant(c), fm.Matrix(A))
    assert fkron._fused_tail(K.content, torch.complex64)
    x = c64(f * n * m, k)
    C = sla.circulant(c.astype(np.complex128))
    A64 = A.astype(np.float64)
    print("kron pair", n, m, f, k, flush=True)
    ref = fast64.kron_apply([fast64.fourier, lambda v: C @ v, lambda v: A64 @ v], (f, n, m), x)
    assert accept.max_rel_error(K.forward(x), ref) < 1e-5
    ref = fast64.kron_apply([lambda v: fast64.fourier(v, adjoint=True),
                             lambda v: C.conj().T @ v, lambda v: A64.T @ v], (f, n, m), x)
    assert accept.max_rel_error(K.backward(x), ref) < 1e-5


@pytest.mark.parametrize("adjoint", [False, True])
def test_capture_after_the_other_direction(adjoint):
    """The pair takes the dense factor as it is or transposed, a table each: a capture
    of one direction after a warm-up of the other alone equals the eager call (the
    single precision bar, as the factors may run apart inside the capture)."""
    import torch

    import fastmat_amd as fm
    rng = np.random.default_rng(5)
    c = (rng.standard_normal(64) + 1j * rng.standard_normal(64)).astype(np.complex64)
    K = fm.Kron(fm.Circulant(c), fm.Matrix(rng.standard_normal((96, 96)).astype(np.float32)))
    x = torch.randn((3, 64 * 96), device="cuda", dtype=torch.complex64).t()
    run, warm = (K.backward, K.forward) if adjoint else (K.forward, K.backward)
    warm(x)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = run(x)
    for _ in range(3):
        x.copy_(torch.randn_like(x))
        ref = run(x)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert (y - ref).abs().max() <= 1e-5 * ref.abs().max()
