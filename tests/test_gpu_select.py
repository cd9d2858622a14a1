"""Row and column selections of a Fourier matrix (alone, or with Diag factors and a
scalar in a Product) run inside the transform's passes: every side and direction,
one- and four-step orders, chirp orders, both precisions, selections in any order
and masks, against the selection as a separate pass over the
nested matrix's own product; and the forms that keep the separate passes.

Bound against the separate passes: the same transform of the same numbers in the same
precision, a few roundings per element apart at most: 16 u of the largest output.
What is not selected is an exact zero on the way in."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _separate(fm, M, rows, cols, x, adjoint):
    """Zero padding, the nested matrix and the gather, in numpy around M."""
    ins, outs = (rows, cols) if adjoint else (cols, rows)
    if ins is not None:
        full = np.zeros((M.numRows if adjoint else M.numCols, x.shape[1]), x.dtype)
        full[ins] = x
        x = full
    y = M.backward(x) if adjoint else M.forward(x)
    return y if outs is None else y[outs]


@pytest.mark.parametrize("dtype", ["complex64", "complex128"])
@pytest.mark.parametrize("n,k", [(1, 2), (2, 1), (64, 3), (1024, 17), (4096, 2), (8192, 3),
                                 (1 << 14, 1), (1 << 14, 40), (1 << 18, 2), (48, 3), (4097, 2),
                                 (6000, 5)])
def test_selected_elements_of_a_transform(n, k, dtype):
    import fastmat_amd as fm
    rng = np.random.default_rng(n + k)

    def rand(*s):
        return (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(dtype)
    F = fm.Fourier(n, dtype=np.dtype(dtype))
    calls = []
    run = F._run_select
    F._run_select = lambda *a: (calls.append(1), run(*a))[1]
    d1, d2 = fm.Diag(rand(n)), fm.Diag(rand(n))
    pick = rng.permutation(n)[:max(1, n // 3)]
    few = np.sort(rng.permutation(n)[:max(1, n // 50)])
    mask = np.zeros(n, bool)
    mask[pick] = True
    u = np.finfo(np.dtype(dtype)).eps
    one_pass = 8192 if dtype == "complex64" else 4096
    pow2 = n & (n - 1) == 0
    for name, M in (("F", F), ("F.H", F.H), ("F D", fm.Product(F, d1)), ("D F", fm.Product(d1, F)),
                    ("2i D F D", fm.Product(2j, d1, F, d2))):
        for rows, cols in ((pick, None), (None, pick), (few, pick), (mask, few),
                           (np.arange(n)[::-1], None)):
            P = fm.Partial(M, rows=rows, cols=cols)
            for adjoint in (False, True):
                x = rand(P.numRows if adjoint else P.numCols, k)
                print("select", n, k, dtype, name, adjoint, None if rows is None else len(rows),
                      None if cols is None else len(cols), flush=True)
                calls.clear()
                got = P.backward(x) if adjoint else P.forward(x)
                if pow2:
                    assert calls
                elif 2 * n - 1 <= one_pass:
                    assert not calls
                ref = _separate(fm, M, rows, cols, x, adjoint)
                assert got.dtype == ref.dtype and got.shape == ref.shape
                assert np.max(np.abs(got - ref)) <= 16 * u * max(np.max(np.abs(ref)), 1e-30)
    # 64 bits from plain numpy
    x = rand(n, k)
    ref = np.fft.fft(x.astype(np.complex128), axis=0)[pick]
    got = fm.Partial(F, rows=pick).forward(x)
    bar = 1e-5 if dtype == "complex64" else 1e-12
    assert np.max(np.abs(got - ref)) <= bar * np.max(np.abs(ref))


def test_selections_that_keep_the_separate_passes():
    """A row asked for twice, real data and a diagonal that widens it, and an
    index that numpy's rules refuse when it is used."""
    import fastmat_amd as fm
    rng = np.random.default_rng(4)
    n = 64
    F = fm.Fourier(n)
    x = (rng.standard_normal((n, 3)) + 1j * rng.standard_normal((n, 3))).astype(np.complex64)
    twice = np.array([5, 1, 5, 63, 0])
    P = fm.Partial(F, rows=twice)
    ref = _separate(fm, F, twice, None, x, False)
    np.testing.assert_array_equal(P.forward(x), ref)
    y = x[:5]
    ref = _separate(fm, F, twice, None, y, True)  # the last of equal rows stands
    assert np.max(np.abs(P.backward(y) - ref)) <= 16 * 1.2e-7 * np.max(np.abs(ref))
    P = fm.Partial(F, rows=np.array([3, 1]))
    for r in (x.real, x.real.astype(np.float64), np.arange(n * 2, dtype=np.int8).reshape(n, 2)):
        ref = F.forward(r)[[3, 1]]
        got = P.forward(r)
        assert got.dtype == ref.dtype
        assert np.max(np.abs(got - ref)) <= 16 * np.finfo(ref.dtype).eps * np.max(np.abs(ref))
    M = fm.Product(F, fm.Diag(rng.standard_normal(n)))  # float64 diagonal, complex64 data
    P = fm.Partial(M, rows=np.array([3, 1]), cols=np.arange(0, n, 2))
    got, ref = P.forward(x[::2]), _separate(fm, M, [3, 1], np.arange(0, n, 2), x[::2], False)
    assert got.dtype == ref.dtype
    assert np.max(np.abs(got - ref)) <= 1e-12 * np.max(np.abs(ref))
    empty = fm.Partial(F, rows=np.zeros(0, int))
    assert empty.forward(x).shape == (0, 3)
    assert not np.any(empty.backward(x[:0]))


def test_selected_transform_replays_in_a_graph():
    import fastmat_amd as fm
    import torch
    torch.manual_seed(3)
    n, k = 1 << 14, 5
    P = fm.Partial(fm.Fourier(n), rows=torch.randperm(n)[:5000].numpy())
    x = torch.randn((k, n), device="cuda", dtype=torch.complex64)
    P.forward(x.t())
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = P.forward(x.t())
    for _ in range(3):
        x.copy_(torch.randn_like(x))
        ref = P.forward(x.t())
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ref)
