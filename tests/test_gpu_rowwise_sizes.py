"""The row-wise kernels (Diag, gather, expand, zero and scatter, axpby) where their
elements per thread change (2^20 elements) and at the edges of a workgroup's share,
with a few rows of many columns and many rows of a few, exact for every type; the
column of an element by its row count's reciprocal at counts that are hard on it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(1, (1 << 20) - 1), (1, 1 << 20), (3, 349526), (7, 149797), (1023, 1025), (1025, 1023),
         ((1 << 20) + 1, 1), ((1 << 19) + 1, 2), (1 << 18, 5), (65537, 17), (999983, 3), (2, 300)]


@pytest.mark.parametrize("dtype", ["int8", "int16", "int32", "int64", "float32", "float64",
                                   "complex64", "complex128"])
@pytest.mark.parametrize("n,k", SIZES)
def test_rowwise(n, k, dtype):
    import torch

    from fastmat_amd import _device as D
    from fastmat_amd import _lib
    t = getattr(torch, dtype)
    g = torch.Generator(device="cuda").manual_seed(n)

    def ints(*shape):
        a = torch.randint(-5, 6, shape, generator=g, device="cuda", dtype=torch.int8)
        return torch.complex(a.to(torch.float64), a.flip(0).to(torch.float64)).to(t) \
            if t.is_complex else a.to(t)
    print("rowwise", n, k, dtype, flush=True)
    ft, s, p = D.fm_type(t), D.stream(), _lib.ptr
    x, y, d = ints(k, n), ints(k, n), ints(n)
    out = torch.empty_like(x)
    for conj in (0, 1):
        _lib.call("fm_diag_apply", ft, conj, n, p(d), p(x), n, p(out), n, k, s)
        assert torch.equal(out, x * (d.conj() if conj else d))
    perm = torch.randperm(n, device="cuda", generator=g)
    m = (n + 1) // 2
    sel = perm[:m].contiguous()
    got = x.new_empty((k, m))
    _lib.call("fm_gather_rows", ft, m, p(sel), p(x), n, p(got), m, k, s)
    assert torch.equal(got, x[:, sel])
    full = torch.zeros_like(x)
    full[:, sel] = got
    _lib.call("fm_scatter_rows", ft, m, p(sel), p(got), m, p(out), n, n, k, s)
    assert torch.equal(out, full)
    inverse = torch.full((n,), -1, dtype=torch.int64, device="cuda")
    inverse[sel] = torch.arange(m, device="cuda")
    out.fill_(7)
    _lib.call("fm_expand_rows", ft, n, p(inverse), p(got), m, p(out), n, k, s)
    assert torch.equal(out, full)
    out.copy_(y)
    _lib.call("fm_axpby", ft, n, k, _lib.dvec(3.0), p(x), n, 0, _lib.dvec(-2.0), p(out), n, s)
    assert torch.equal(out, x * 3 - y * 2)
    _lib.call("fm_axpby", ft, n, k, _lib.dvec(3.0), p(x), n, 1, _lib.dvec(0.0), p(out), n, s)
    assert torch.equal(out, x.conj().resolve_conj() * 3)


@pytest.mark.parametrize("n,k,ld", [(3, 400000, 5), (300, 4000, 301), (5, 9, 8)])
def test_leading_dimensions(n, k, ld):
    """Columns of wider blocks; what lies between them stays."""
    import torch

    from fastmat_amd import _device as D
    from fastmat_amd import _lib
    x = torch.arange(k * ld, device="cuda", dtype=torch.int32).reshape(k, ld) % 1000
    y = torch.full((k, ld + 1), -7, dtype=torch.int32, device="cuda")
    d = torch.arange(1, n + 1, device="cuda", dtype=torch.int32)
    print("ld", n, k, ld, flush=True)
    _lib.call("fm_diag_apply", D.fm_type(np.int32), 0, n, _lib.ptr(d), _lib.ptr(x), ld,
              _lib.ptr(y), ld + 1, k, D.stream())
    assert torch.equal(y[:, :n], x[:, :n] * d) and bool((y[:, n:] == -7).all())
    idx = torch.arange(n - 1, -1, -1, device="cuda")
    _lib.call("fm_gather_rows", D.fm_type(np.int32), n, _lib.ptr(idx), _lib.ptr(x), ld,
              _lib.ptr(y), ld + 1, k, D.stream())
    assert torch.equal(y[:, :n], x[:, :n].flip(1)) and bool((y[:, n:] == -7).all())
