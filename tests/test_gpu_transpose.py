"""Row-major device operands: the library's transpose to column blocks (exact, for
every element size), at the edges of its tiles, for row-strided views, and the
layouts that it leaves to torch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["int8", "int16", "int32", "float32", "int64", "complex64",
                                   "complex128"])
@pytest.mark.parametrize("n,k", [(4096, 1), (2049, 2), (2500, 3), (1025, 4), (700, 8), (333, 16),
                                 (129, 32), (128, 33), (257, 64), (63, 1001)])
def test_contiguous_block(n, k, dtype, monkeypatch):
    import torch

    from fastmat_amd import _device as D
    monkeypatch.setattr(D, "_TRANSPOSE_BYTES", 0)  # the transpose at every size
    rng = np.random.default_rng(n + k)
    a = rng.integers(-100, 100, size=(n + 1, k + 5)).astype(dtype)
    if a.dtype.kind == "c":
        a = a + 1j * rng.integers(-100, 100, size=a.shape).astype(dtype)
    t = torch.from_numpy(np.ascontiguousarray(a)).cuda()
    for v, r in ((t, a), (t[1:, :k], a[1:, :k]), (t[:n, 5:], a[:n, 5:]), (t[::2], a[::2]),
                 (t.t().contiguous().t(), a), (t[:, ::2], a[:, ::2])):
        print("block", n, k, dtype, tuple(v.shape), v.stride(), flush=True)
        out = D.contiguous_block(v.t())
        assert out.is_contiguous()
        np.testing.assert_array_equal(out.cpu().numpy(), r.T)
    if t.is_complex():
        out = D.contiguous_block(t.conj().t())
        np.testing.assert_array_equal(out.resolve_conj().cpu().numpy(), a.conj().T)
