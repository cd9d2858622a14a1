"""Selections around a Fourier matrix on real and integer data: converted once where
the transform's passes take the selections, by the general path alone where they do
not (orders of a one-pass chirp transform), with equal results either way."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("adjoint", [False, True])
@pytest.mark.parametrize("dtype", ["int8", "int64", "float32", "float64", "complex64",
                                   "complex128"])
@pytest.mark.parametrize("kind", ["F", "FD", "DF", "FHDF", "scaled"])
@pytest.mark.parametrize("n", [256, 300])
def test_types(n, kind, dtype, adjoint):
    import torch

    import fastmat_amd as fm
    rng = np.random.default_rng(n)
    F = fm.Fourier(n)
    D = fm.Diag((rng.integers(1, 4, n) + 1j * rng.integers(-2, 3, n)).astype(np.complex64))
    M = {"F": F, "FD": fm.Product(F, D), "DF": fm.Product(D, F),
         "FHDF": fm.Product(F.H, D, F), "scaled": fm.Product(2.0, F)}[kind]
    rows, cols = rng.permutation(n)[:n // 3], np.sort(rng.permutation(n)[:n // 2])
    P = fm.Partial(M, rows=rows, cols=cols)
    x = torch.from_numpy(rng.integers(-9, 10, (len(rows) if adjoint else len(cols), 3))
                         .astype(dtype)).cuda()
    print("types", n, kind, dtype, adjoint, flush=True)
    full = x.new_zeros((n, 3))
    full[torch.from_numpy(rows if adjoint else cols).cuda()] = x
    got = (P.backward if adjoint else P.forward)(x)
    ref = (M.backward if adjoint else M.forward)(full)
    ref = ref[torch.from_numpy(cols if adjoint else rows).cuda()]
    assert got.dtype == ref.dtype
    # the two paths' roundings: 16 u of the largest value each, as in the tables' tests
    u = 1.2e-7 if ref.dtype == torch.complex64 else 2.3e-16
    assert (got - ref).abs().max() <= 2 * 16 * u * ref.abs().max()


def test_data_is_not_converted_for_a_path_that_is_not_taken(monkeypatch):
    import torch

    import fastmat_amd as fm
    n = 300
    P = fm.Partial(fm.Fourier(n), rows=np.arange(0, n, 3))
    x = torch.ones((n, 2), dtype=torch.float64, device="cuda")
    P.forward(x)
    made = []
    to = torch.Tensor.to
    monkeypatch.setattr(torch.Tensor, "to", lambda t, *a, **k: made.append(a) or to(t, *a, **k))
    P.forward(x)
    assert made.count((torch.complex128,)) == 1
