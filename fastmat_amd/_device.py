"""Device-side array plumbing shared by all operators.

Internal block format: a contiguous torch tensor of shape (k, n) on the HIP
device, i.e. k right-hand-side vectors of length n stored one after another.
This is exactly the F-contiguous (n, k) array fastmat's C-style classes work
on (Matrix.pyx:1892-1901, core/cmath.pyx:343-386), so every block can be
handed to the C ABI as a column-major (n, k) array with leading dimension n.

User-facing inputs may be numpy arrays or torch tensors, 1-D (n,) or 2-D
(n, k) (Matrix.pyx:1770-1790).  Results are returned in the caller's kind:
numpy in -> numpy out (F-ordered, like fastmat), torch in -> torch out as an
(m, k) view whose columns are contiguous.
"""
import numpy as np
import torch

from . import _lib

_NP2T = {
    np.dtype(np.int8): torch.int8, np.dtype(np.int16): torch.int16,
    np.dtype(np.int32): torch.int32, np.dtype(np.int64): torch.int64,
    np.dtype(np.float32): torch.float32, np.dtype(np.float64): torch.float64,
    np.dtype(np.complex64): torch.complex64, np.dtype(np.complex128): torch.complex128,
}
_T2NP = {v: k for k, v in _NP2T.items()}

SUPPORTED = tuple(_NP2T)


def np_dtype(dt):
    """numpy dtype of a numpy dtype-like or torch dtype."""
    if isinstance(dt, np.dtype):
        return dt
    r = _T2NP.get(dt)
    if r is not None:
        return r
    if isinstance(dt, torch.dtype):
        raise TypeError("Unsupported data type %s" % dt)
    return np.dtype(dt)


def torch_dtype(dt):
    t = _NP2T.get(np_dtype(dt))
    if t is None:
        raise TypeError("Unsupported data type %s" % np_dtype(dt))
    return t


def fm_type(dt):
    return _lib.NP_TO_FM[np_dtype(dt)]


# Type rules are looked up on every apply of a small operand: their results, per
# pair of types, are kept (the types are few).
_promoted = {}
_input_types = {}


def promote(a, b):
    """numpy promotion (the reference's promotion table equals
    np.promote_types, core/types.pyx:418-453)."""
    r = _promoted.get((a, b))
    if r is None:
        r = _promoted[a, b] = np.promote_types(np_dtype(a), np_dtype(b))
    return r


def input_type(in_dtype, min_type, dtype, widen):
    """torch type in which an operator of type `dtype` takes data of the torch
    type `in_dtype` (Matrix._prepareInputArray, Matrix.pyx:1737-1817):
    promote(input, minType), widened to the output's type where asked."""
    key = (in_dtype, min_type, dtype, widen)
    r = _input_types.get(key)
    if r is None:
        fin = promote(in_dtype, min_type)
        r = _input_types[key] = torch_dtype(promote(fin, dtype) if widen else fin)
    return r


def safe_type_expansion(dtype):
    """int8/int16 -> float32, int32/int64 -> float64 (core/types.pyx:378-394)."""
    dt = np_dtype(dtype)
    if dt in (np.dtype(np.int8), np.dtype(np.int16)):
        return np.dtype(np.float32)
    if dt in (np.dtype(np.int32), np.dtype(np.int64)):
        return np.dtype(np.float64)
    return dt


_device = None


def device():
    global _device
    if _device is None:
        if not torch.cuda.is_available():
            raise _lib.FastmatAmdError(
                "fastmat_amd needs a HIP device; none is visible")
        _device = torch.device("cuda", torch.cuda.current_device())
    return _device


class Boundary:
    """Records how the caller passed an array, to return results alike."""

    __slots__ = ("kind", "was1d", "dev")

    def __init__(self, kind, was1d, dev):
        self.kind = kind
        self.was1d = was1d
        self.dev = dev

    def finish(self, Y):
        """Y: internal (k, m) block -> caller's format."""
        out = Y.t()  # (m, k), columns contiguous
        if self.was1d:
            out = out[:, 0]
        if self.kind == "numpy":
            return out.cpu().numpy()
        if self.kind == "torch-cpu":
            return out.cpu()
        return out


def to_block(arr, required):
    """Validate and convert a caller array into an internal (k, n) block.

    Errors follow Matrix._prepareInputArray (Matrix.pyx:1770-1782).
    """
    if isinstance(arr, torch.Tensor):
        kind = "torch" if arr.is_cuda else "torch-cpu"
        t = arr
    else:
        a = np.asarray(arr)
        if a.dtype not in _NP2T:
            if a.dtype == np.bool_ or a.dtype.kind in "ui":
                a = a.astype(np.promote_types(a.dtype, np.int8)) if a.dtype.kind != "u" \
                    else a.astype(np.int64)
            else:
                raise TypeError("Unsupported data type %s" % a.dtype)
        kind = "numpy"
        t = torch.from_numpy(np.ascontiguousarray(a.T) if a.ndim == 2 else np.ascontiguousarray(a))
        t = t.t() if a.ndim == 2 else t
    if t.dim() < 1 or t.dim() > 2:
        raise ValueError("Input data array must be 1D or 2D")
    if t.shape[0] != required:
        raise ValueError("Mismatch of vector size %d to relevant matrix axis %d" % (
            t.shape[0], required))
    if t.dtype not in _T2NP:
        raise TypeError("Unsupported data type %s" % t.dtype)
    was1d = t.dim() == 1
    if was1d:
        t = t.reshape(required, 1)
    dev = device()
    block = t.t()
    if block.device != dev:
        block = block.to(dev, non_blocking=False)
    return contiguous_block(block), Boundary(kind, was1d, dev)


# Row-major operands from this size on go through the library's transpose; torch's
# strided copy costs the host 1.5 us less and is as fast below (2 MB complex128: 4.4 us).
_TRANSPOSE_BYTES = 4 << 20


def _transpose_bytes(esz, n, k):
    """Size from which the library's transpose of n rows of k elements is the faster
    one.  Measured, own / torch's copy in us:
    - rows that fill its tiles: 2^18 x 8 float32 5.4 / 7.7, 2^20 x 32 33 / 625,
      2^18 x 32 float64 20 / 49, complex128 46 / 77, 2^20 x 8 complex128 47 / 154;
    - shorter ones only when large: 2^20 x 5 float32 9.4 / 7.9, 2^18 x 5 complex128
      13 / 8, but 2^22 x 2 float32 10 / 14, 2^20 x 5 complex128 42 / 67;
    - small elements by whole tiles of 16 or 32: 2^20 x 12 int8 15 / 11, x 24 33 / 23,
      but x 16 14 / 20 and x 28 34 / 33; 2^19 x 17 int16 17 / 13, but x 24 19 / 22; or
      where the columns of torch's copy do not all read a row on the same XCD (row
      counts that are no multiple of 8192: 700000 x 24 int8 24 / 52) or its L2 does not
      hold the rows (2^21 x 20 int8 57 / 71);
    - few rows leave its tiles empty, and torch's copy is in runs of rows:
      2 x 2500000 float32 97 / 8, 32 x 100000 float64 13 / 11, but 48 x 100000 14 / 18;
      128 x 100000 complex128 118 / 99, but 256 x 5000 13 / 16."""
    if esz >= 4:
        pays = n >= (256 if esz == 16 else 48)
        return _TRANSPOSE_BYTES * ((1 if k >= 8 else 8) if pays else 1 << 30)
    pays = n >= 48 and k >= 16 and (k == 16 or k >= (28 if esz == 1 else 20) or
                                    n % 8192 != 0 or (k >= 20 and n > 1 << 20))
    return _TRANSPOSE_BYTES * (1 if pays else 1 << 30)


def contiguous_block(block):
    """The (k, n) view `block` as a contiguous tensor.  Columns of a large
    row-major (n, k) array on the device go through the library's transpose
    (see _transpose_bytes); small ones, other layouts, lazily conjugated or
    negated tensors and tensor subclasses through torch."""
    if block.is_contiguous():
        return block
    k, n = block.shape
    esz = block.element_size()
    if k * n * esz >= _transpose_bytes(esz, n, k) and type(block) is torch.Tensor:
        s0, s1 = block.stride()
        if (s0 == 1 and s1 >= k and block.dtype in _T2NP and block.device == device() and
                not block.is_conj() and not block.is_neg() and
                (esz < 16 or block.data_ptr() % 16 == 0)):
            out = block.new_empty((k, n))
            _lib.call("fm_transpose", esz, n, k, block.data_ptr(), s1, out.data_ptr(), n,
                      stream())
            return out
    return block.contiguous()


def empty(k, n, dtype):
    return torch.empty((k, n), dtype=torch_dtype(dtype), device=device())


# Raw handle of the current stream without building a Stream object (2 us of a
# small apply); older torch versions lack it.
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def stream():
    """hipStream_t of torch's current stream on the device, as an address."""
    if _raw_stream is None:
        return _lib.stream_handle(device())
    return _raw_stream(device().index)


def ld(t):
    """Leading dimension (elements between rows) of a (k, w) view with unit
    element stride; a single row may report any row stride, so its width is
    used."""
    return int(t.shape[1]) if t.shape[0] == 1 else int(t.stride(0))


def workspace(nbytes):
    """Device scratch of at least nbytes (uint8 tensor; caller keeps it alive
    until the stream has consumed it, which torch's caching allocator
    guarantees for tensors freed after enqueueing on the current stream)."""
    if nbytes <= 0:
        return None
    return torch.empty(int(nbytes), dtype=torch.uint8, device=device())


def squeeze1d(a):
    """Squeezed, at least 1-D copy (core/cmath.pyx:389-441, _arrSqueezedCopy)."""
    return np.atleast_1d(np.squeeze(np.array(a))).copy()


def as_tensor(values, dtype):
    """Host array -> device tensor of `dtype` (1-D or 2-D)."""
    a = np.ascontiguousarray(np.asarray(values).astype(np_dtype(dtype)))
    return torch.from_numpy(a).to(device())
