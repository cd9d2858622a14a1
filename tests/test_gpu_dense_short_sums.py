"""Real matrices on many complex64 columns: sums short enough that a wave takes them
alone, at the edges of its tile (64 rows of 32 columns), of its K steps (16) and of the
rule (sums of 512, a wave for every SIMD).

Bound: K products in precision u in any order are off by at most about K u sum
|a_l||x_l| (Higham, Accuracy and Stability, 3.1); each part of a complex result is one
such sum, and 2 covers the few roundings on top."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("adjoint", [False, True])
@pytest.mark.parametrize("m,n,k", [(129, 1, 11000), (130, 4, 10945), (191, 15, 10977),
                                   (192, 16, 10923), (193, 17, 8193), (1, 129, 32800),
                                   (63, 512, 32769), (64, 513, 32768), (65, 300, 16385), (16, 200, 32800),
                                   (17, 257, 65537), (17, 256, 32769),
                                   (2000, 33, 1024), (2049, 100, 993)])
def test_many_columns(m, n, k, adjoint):
    import torch

    from fastmat_amd import _device as D
    import fastmat_amd as fm
    rng = np.random.default_rng(m + n + k)
    A = rng.standard_normal((m, n)).astype(np.float32)
    M = fm.Matrix(A.T.copy() if adjoint else A)
    g = torch.Generator(device="cuda").manual_seed(k)
    x = torch.randn((k, n), generator=g, device="cuda", dtype=torch.complex64)
    print("columns", m, n, k, adjoint, flush=True)
    y = M._apply(x, adjoint)
    assert y.shape == (k, m) and D.np_dtype(y.dtype) == np.complex64
    a = torch.from_numpy(A).cuda().double().t().contiguous()
    for got, part in ((y.real, x.real), (y.imag, x.imag)):
        ref = part.double() @ a
        bound = 2 * (n + 8) * 1.2e-7 * (part.double().abs() @ a.abs())
        assert bool(((got.double() - ref).abs() <= bound).all())


def test_rows_and_columns_apart():
    """An infinity or NaN reaches its row or column of the result only."""
    import torch

    import fastmat_amd as fm
    m, n, k = 147, 20, 11011
    A = np.ones((m, n), np.float32)
    A[m - 1, 3] = np.inf
    x = torch.ones((k, n), device="cuda", dtype=torch.complex64)
    x[k - 1, n - 1] = float("nan")
    y = fm.Matrix(A)._apply(x, False)
    assert bool((y[:k - 1, :m - 1] == complex(n, 0)).all())
    assert bool(torch.isnan(y[k - 1].real).all())
    assert not bool(torch.isfinite(y[:, m - 1].real).any())
