"""Partial: row/column sub-selection of a matrix (fastmat/Partial.pyx).

Forward scatters x into a zero-padded vector of the nested matrix's width at
``colSelection``, applies the matrix and gathers ``rowSelection``
(Partial.pyx:268-280); backward mirrors it (:282-294).  Around a Fourier matrix
(alone or with Diag factors) both selections run inside the transform's passes;
otherwise scatter (through the selection's inverse) and gather are library
kernels."""
import numpy as np
import torch

from . import _device as D
from . import _lib
from .fourier import Fourier
from .matrix import Hermitian, Matrix
from .product import Product, select_chain


# Matrices whose passes may take the selections (select_chain).
_FOURIER = (Product, Fourier, Hermitian)

# Selections of vectors up to this length are inverted on the host and go to the device
# with their indices in one copy; of longer ones the device makes the inverse and the
# host waits for it.  First forward of a third of the rows of a Fourier matrix, us,
# host / device / separate passes without an inverse: 1024 points 66 / 84 / 61,
# 4096 63 / 82 / 66, 16384 82 / 87 / 77, 100003 170 / 112 / 127, 2^18 350 / 132 / 215;
# rows and columns of 1024 points 78 / 136 / 93.
_HOST_TABLE = 1 << 14


def _padded(size):
    """Entries of an inverse in a buffer with others: whole cache lines (256 bytes), as
    the passes read a table across lines slower (2^18 x 32: 162 us with the table 4
    bytes off, 160 without)."""
    return -(-size // 64) * 64


def _check_selection(sel, size, name):
    if sel is None:
        return None
    sel = np.array(sel)
    if sel.dtype == bool:
        sel = np.arange(size)[sel]
    elif np.issubdtype(sel.dtype, np.integer):
        pass
    else:
        raise TypeError("Partial: Type of %s indices must be int or bool." % (name,))
    bounded = ((len(sel) != size or np.sum(sel - np.arange(size)) != 0) and
               np.any((sel >= size) | (sel < 0)))
    if bounded:
        raise ValueError("Partial: A %s index exceeds matrix dimensions." % (name,))
    return sel.astype(np.int64)


def _device_index(sel, size):
    """Row indices for the scatter / gather kernels with numpy's indexing
    rules: an index in [-size, -1] counts from the end, anything outside
    [-size, size) raises IndexError when the selection is used (the
    reference's check above lets e.g. [-1, 1, 3] of size 3 through, and
    numpy then raises at apply time, Partial.pyx:272-279)."""
    if sel.size == 0 or (sel.min() >= 0 and sel.max() < size):
        return sel
    bad = (sel < -size) | (sel >= size)
    if np.any(bad):
        raise IndexError("index %d is out of bounds for axis 0 with size %d"
                         % (int(sel[np.argmax(bad)]), size))
    return np.where(sel < 0, sel + size, sel).astype(np.int64)


class Partial(Matrix):
    def __init__(self, mat, **options):
        if not isinstance(mat, Matrix):
            raise TypeError("Partial: fastmat Matrix required.")
        if "N" in options:
            options["rows"] = options.pop("N")
        if "M" in options:
            options["cols"] = options.pop("M")
        self._content = (mat,)
        self._rowSelection = _check_selection(options.pop("rows", None), mat.numRows, "row")
        self._colSelection = _check_selection(options.pop("cols", None), mat.numCols, "col")
        self._dev = {}
        self._initProperties(
            len(self._rowSelection) if self._rowSelection is not None else mat.numRows,
            len(self._colSelection) if self._colSelection is not None else mat.numCols,
            mat.dtype, **options)

    @property
    def rowSelection(self):
        return self._rowSelection

    @property
    def colSelection(self):
        return self._colSelection

    def _getColNorms(self):
        # Partial.pyx:234-241: without a row selection the norms are the
        # parent's, restricted to the selected columns
        if self._rowSelection is not None:
            return super()._getColNorms()
        norms = self._content[0].colNorms
        return norms if self._colSelection is None else norms[self._colSelection]

    def _getRowNorms(self):
        # Partial.pyx:243-250
        if self._colSelection is not None:
            return super()._getRowNorms()
        norms = self._content[0].rowNorms
        return norms if self._rowSelection is None else norms[self._rowSelection]

    def _selections(self):
        """(name, selection, size of what it selects from) of those given."""
        M = self._content[0]
        both = (("r", self._rowSelection, M.numRows), ("c", self._colSelection, M.numCols))
        return [s for s in both if s[1] is not None]

    def _idx(self, name):
        """The selection's indices on the device."""
        t = self._dev.get(name)
        if t is None:
            sel, size = next(s[1:] for s in self._selections() if s[0] == name)
            t = self._keep(name, D.as_tensor(_device_index(sel, size), np.int64))
        return t

    def _keep(self, key, table):
        """Keep a device table unless there is one: a captured graph holds the address
        of the one that was there at its capture, which therefore stays."""
        return self._dev.setdefault(key, table)

    def _upload(self, sels, dtype):
        """Indices and inverses (_inverse) of the selections to the device, in one
        copy."""
        indices, inverses = [], []
        for name, sel, size in sels:
            idx = _device_index(sel, size)
            inverse = np.full(_padded(size), -1, dtype=D.np_dtype(dtype))
            inverse[idx] = np.arange(len(idx))
            self._keep("distinct" + name, np.count_nonzero(inverse >= 0) == len(idx))
            indices.append(idx)
            inverses.append(inverse.view(np.int64))
        parts = inverses + indices
        t = torch.from_numpy(np.concatenate(parts)).to(D.device())
        t = t.split([len(p) for p in parts])
        for (name, _, _), inverse, idx in zip(sels, t, t[len(sels):]):
            self._keep((name, dtype), inverse.view(dtype))
            self._keep(name, idx)

    def _inverse(self, name, dtype=torch.int64):
        """Row of the selection that lands on each row of the nested matrix's
        operand, -1 for none (the last one of equal indices, as numpy's
        indexed assignment leaves it).  The table is complete before it is kept:
        a later call may run on another stream.  None where it would have to be
        made inside a stream capture, which does not run its kernels."""
        if (name, dtype) not in self._dev and not torch.cuda.is_current_stream_capturing():
            # (the transform's passes take both, an expansion its own)
            sels = [s for s in self._selections() if dtype == torch.int32 or s[0] == name]
            if max(s[2] for s in sels) <= _HOST_TABLE:
                self._upload(sels, dtype)
            else:
                self._invert(sels, dtype)
        return self._dev.get((name, dtype))

    def _invert(self, sels, dtype):
        """Inverses of the selections by the device, with one wait for all of them."""
        flags = torch.empty(len(sels), dtype=dtype, device=D.device())
        tables = [flags.new_empty(size) for _, _, size in sels]
        for q, (table, (name, sel, size)) in enumerate(zip(tables, sels)):
            _lib.call("fm_invert_index", table.element_size(), len(sel),
                      _lib.ptr(self._idx(name)), size, _lib.ptr(table), _lib.ptr(flags[q:]),
                      D.stream())
        for twice, table, (name, _, _) in zip(flags.tolist(), tables, sels):
            self._keep((name, dtype), table)
            self._keep("distinct" + name, not twice)

    def _distinct(self, name):
        """True when no element is selected twice; False inside a stream capture
        where it is not known yet."""
        if "distinct" + name not in self._dev:
            self._inverse(name, torch.int32)
        return self._dev.get("distinct" + name, False)

    def _selected(self, X, adjoint):
        """The product with both selections inside the passes of the nested
        Fourier matrix (select_chain), or None: other matrices, selections that
        name an element twice for the result, empty ones, and a capture before
        the tables are there."""
        M = self._content[0]
        if type(M) not in _FOURIER or X.shape[0] == 0:
            return None
        ins, outs = ("c", self._colSelection), ("r", self._rowSelection)
        if adjoint:
            ins, outs = outs, ins
        given = [s for _, s in (ins, outs) if s is not None]
        if not given or any(len(s) == 0 for s in given):
            return None

        def tables():
            made = [None if sel is None else self._inverse(name, torch.int32)
                    for name, sel in (ins, outs)]
            if any(s is not None and t is None for t, (_, s) in zip(made, (ins, outs))):
                return None
            return made if outs[1] is None or self._distinct(outs[0]) else None
        return select_chain(M, X, adjoint, ins[1] is not None, outs[1] is not None, tables,
                            self.numCols if adjoint else self.numRows)

    def _scatter(self, X, sel, name, n_full):
        k, n = X.shape
        Y = D.empty(k, n_full, X.dtype)
        if n == 0:
            return Y.zero_()
        inverse = self._inverse(name)
        if inverse is None:  # (a capture that no call of this direction came before)
            _lib.call("fm_scatter_rows", D.fm_type(X.dtype), n, _lib.ptr(self._idx(name)),
                      _lib.ptr(X), n, _lib.ptr(Y), n_full, n_full, k, D.stream())
        else:
            _lib.call("fm_expand_rows", D.fm_type(X.dtype), n_full, _lib.ptr(inverse),
                      _lib.ptr(X), n, _lib.ptr(Y), n_full, k, D.stream())
        return Y

    def _gather(self, X, sel, name):
        k, n = X.shape
        m = len(sel)
        Y = D.empty(k, m, X.dtype)
        _lib.call("fm_gather_rows", D.fm_type(X.dtype), m, _lib.ptr(self._idx(name)),
                  _lib.ptr(X), n, _lib.ptr(Y), m, k, D.stream())
        return Y

    def _fwd(self, X):
        M = self._content[0]
        Y = self._selected(X, False)
        if Y is not None:
            return Y
        if self._colSelection is not None:
            X = self._scatter(X, self._colSelection, "c", M.numCols)
        Y = M._apply(X, False)
        if self._rowSelection is not None:
            Y = self._gather(Y, self._rowSelection, "r")
        return Y

    def _bwd(self, X):
        M = self._content[0]
        Y = self._selected(X, True)
        if Y is not None:
            return Y
        if self._rowSelection is not None:
            X = self._scatter(X, self._rowSelection, "r", M.numRows)
        Y = M._apply(X, True)
        if self._colSelection is not None:
            Y = self._gather(Y, self._colSelection, "c")
        return Y

    def _reference(self):
        full = self._content[0].reference()
        if self._rowSelection is not None:
            full = full[self._rowSelection, :]
        if self._colSelection is not None:
            full = full[:, self._colSelection]
        return full
