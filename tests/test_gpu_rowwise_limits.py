"""The row-wise kernels beyond one launch's threads (2^32 in a grid dimension) and
beyond their largest grids, where they stride: a few rows of many columns, and many
rows.  Exact in bytes, on the device."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bytes(k, n, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(-100, 100, (k, n), generator=g, device="cuda", dtype=torch.int8)


@pytest.mark.parametrize("n,k", [(2, (1 << 24) + 3), (1025, (1 << 21) + 5)])
def test_many_columns(n, k):
    import torch

    import fastmat_amd as fm
    X = _bytes(k, n, 1)
    sigma = np.random.default_rng(n).permutation(n)
    s = torch.from_numpy(sigma).cuda()
    print("columns", n, k, flush=True)
    assert torch.equal(fm.Permutation(sigma)._apply(X, False), X[:, s])
    P = fm.Partial(fm.Eye(n), rows=sigma[:n - 1])
    assert torch.equal(P._apply(X, False), X[:, s[:n - 1]])
    full = torch.zeros_like(X)
    full[:, s[:n - 1]] = X[:, :n - 1]
    assert torch.equal(P._apply(X[:, :n - 1].contiguous(), True), full)
    d = np.arange(n).astype(np.int8)
    assert torch.equal(fm.Diag(d)._apply(X, False), X * torch.from_numpy(d).cuda())


def test_many_rows():
    import torch

    from fastmat_amd import _device as D
    from fastmat_amd import _lib
    n = (1 << 30) + 71
    X = _bytes(1, n, 2)
    Y = X.clone()
    print("rows", n, flush=True)
    _lib.call("fm_axpby", D.fm_type(np.int8), n, 1, _lib.dvec(3.0), X.data_ptr(), n, 0,
              _lib.dvec(1.0), Y.data_ptr(), n, D.stream())
    assert torch.equal(Y, X * 4)
    d = _bytes(1, n, 3)
    _lib.call("fm_diag_apply", D.fm_type(np.int8), 0, n, d.data_ptr(), X.data_ptr(), n,
              Y.data_ptr(), n, 1, D.stream())
    assert torch.equal(Y, X * d)
