"""Dense products of more tiles than one launch takes (2^32 threads): a matrix of one
long column or row.  Exact."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,m,adjoint", [("float32", (1 << 29) + 70, 0),
                                             ("float32", (1 << 27) + 5, 1),
                                             ("float64", (1 << 27) + 5, 1)])
def test_more_tiles_than_a_launch_takes(dtype, m, adjoint):
    """One column (row) times a number: every product is exact."""
    import torch

    from fastmat_amd import _device as D
    from fastmat_amd import _lib
    t = getattr(torch, dtype)
    a = torch.arange(m, device="cuda", dtype=torch.int32).remainder_(8191).to(t)
    x = torch.full((1, 1), 3.0, device="cuda", dtype=t)
    y = torch.empty((1, m), device="cuda", dtype=t)
    rows, cols = (1, m) if adjoint else (m, 1)
    print("tiles", dtype, m, adjoint, flush=True)
    _lib.call("fm_dense_apply", D.fm_type(t), D.fm_type(t), adjoint, rows, cols, a.data_ptr(), cols,
              x.data_ptr(), 1, y.data_ptr(), m, 1, D.stream())
    assert torch.equal(y[0], a * 3)
