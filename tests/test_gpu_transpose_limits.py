"""Row-major operands of more columns than one launch's grid has column tiles (65535
of 32): taken as any other, by the operators and by the library's transpose.  Exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rows(n, k, dtype):
    import torch
    g = torch.Generator(device="cuda").manual_seed(n)
    return torch.randint(-100, 100, (n, k), generator=g, device="cuda", dtype=torch.int8).to(dtype)


@pytest.mark.parametrize("n,k", [(2, 2097121), (2, 3000000), (129, 2097153)])
def test_operators(n, k):
    import torch

    import fastmat_amd as fm
    x = _rows(n, k, torch.float32)
    print("rows", n, k, flush=True)
    assert torch.equal(fm.Eye(n).forward(x), x)
    d = np.arange(1, n + 1, dtype=np.float32)
    y = fm.Diag(d).backward(x)
    assert torch.equal(y, x * torch.from_numpy(d).cuda()[:, None])


@pytest.mark.parametrize("dtype", ["int8", "int16", "int32", "int64", "complex128"])
@pytest.mark.parametrize("n,k", [(2, 2097121), (129, 2097153)])
def test_transpose(n, k, dtype):
    import torch

    from fastmat_amd import _device as D
    from fastmat_amd import _lib
    x = _rows(n, k, getattr(torch, dtype))
    y = x.new_full((k, n), 7)
    print("transpose", n, k, dtype, flush=True)
    _lib.call("fm_transpose", x.element_size(), n, k, x.data_ptr(), k, y.data_ptr(), n,
              D.stream())
    assert torch.equal(y, x.t())
