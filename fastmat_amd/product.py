"""Product: s * A1 A2 ... An (fastmat/Product.pyx).

Forward applies the last factor first, backward the first factor's adjoint
first with conj(s) (Product.pyx:205-240); nested Products flatten and their
scalars multiply (:101-105); dtype = promote(factors, scalars) expanded by
``typeExpansion`` (default safeTypeExpansion, :120-122)."""
import numpy as np

from . import _device as D
from .diag import Diag
from .fourier import Fourier
from .matrix import Hermitian, Matrix, scale_block


class Product(Matrix):
    def __init__(self, *matrices, **options):
        factors = []
        scalar = [np.int8(1)]
        dtype = [np.dtype(np.int8)]

        def add(items):
            for f in items:
                if np.isscalar(f):
                    dtype[0] = np.promote_types(dtype[0], np.array(f).dtype)
                    scalar[0] = np.inner(scalar[0], f)
                    continue
                if not isinstance(f, Matrix):
                    raise TypeError("Product: Term not scalar nor Matrix.")
                if isinstance(f, Product):
                    if f._scalar != 1:
                        scalar[0] = scalar[0] * f._scalar
                    add(f.content)
                else:
                    factors.append(f)
                dtype[0] = np.promote_types(dtype[0], f.dtype)

        add(matrices)
        dt = dtype[0]
        typeExpansion = options.pop("typeExpansion", D.safe_type_expansion(dt))
        dt = dt if typeExpansion is None else np.promote_types(dt, typeExpansion)
        options.pop("debug", None)
        if len(factors) < 1:
            raise ValueError("Product has no terms.")
        numRows, numCols = factors[0].numRows, factors[0].numCols
        for ii in range(1, len(factors)):
            if factors[ii].numRows != numCols:
                raise ValueError("Product: Dimension mismatch for term %d [%dx%d]" % (
                    ii, numRows, numCols))
            numCols = factors[ii].numCols
        self._scalar = np.asarray(scalar[0]).astype(dt)
        self._content = tuple(factors)
        self._initProperties(numRows, numCols, dt, **options)

    @property
    def scalar(self):
        return self._scalar

    def _prep(self, X, conj):
        dt = D.promote(X.dtype, self.dtype)
        if D.np_dtype(X.dtype) != dt:
            X = X.to(D.torch_dtype(dt))
        if self._scalar != 1:
            s = complex(self._scalar)
            if conj:
                s = s.conjugate()
            X = scale_block(X, s)
        return X

    def _fwd(self, X):
        return _apply_chain(self._content[::-1], self._prep(X, False), False)

    def _bwd(self, X):
        return _apply_chain(self._content, self._prep(X, np.iscomplexobj(self._scalar)), True)

    def _reference(self):
        dt = np.promote_types(np.float64, self.dtype)
        res = np.inner(self._content[-1].reference(), self._scalar.astype(dt))
        for f in self._content[-2::-1]:
            res = f.reference().dot(res)
        return res


def _apply_chain(factors, X, adjoint):
    """The factors (their adjoints) applied to X one after another, the first in
    the sequence first.  A Fourier factor takes neighbouring Diag factors into
    its passes (fm_fourier_apply_diag): they multiply as the transform reads and
    writes, instead of a pass over the data each."""
    i = 0
    while i < len(factors):
        fused = _fourier_with_diags(factors, i, X, adjoint)
        if fused is None:
            X = factors[i]._apply(X, adjoint)
            i += 1
        else:
            X, i = fused
    return X


def _fourier_with_diags(factors, i, X, adjoint):
    """(result, next index) of a Diag / Fourier / Diag run starting at i that
    has a Fourier and at least one Diag, or None."""
    pre = factors[i] if type(factors[i]) is Diag else None
    f = i + (pre is not None)
    if f >= len(factors):
        return None
    F, flip = _as_fourier(factors[f])
    post = factors[f + 1] if f + 1 < len(factors) and type(factors[f + 1]) is Diag else None
    if F is None or (pre is None and post is None) or not _diags_ok(F, X.dtype, pre, post):
        return None
    # the transform conjugates its tables when it is an adjoint one; a Diag's
    # adjoint is its conjugate
    inverse = adjoint != flip
    tables = _diag_tables(D.np_dtype(X.dtype), inverse != adjoint, pre, post)
    if tables is None:
        return None
    return F._run_diag(X, inverse, *tables), f + 1 + (post is not None)


def _diag_tables(dt, conj, *diags):
    """Tables of the Diag factors (None for None), or None where one is missing
    (Diag._table): the factors then run apart."""
    tables = [None if d is None else d._table(dt, conj) for d in diags]
    if any(t is None and d is not None for t, d in zip(tables, diags)):
        return None
    return tables


def _diags_ok(F, dtype, *diags):
    """True when the Diag factors (or None) can run inside F's transform of data of
    the torch type."""
    dt = D.np_dtype(dtype)
    return F._diag_ok(dtype) and all(
        d is None or (D.promote(dt, d.dtype) == dt and D.promote(dt, d._minType) == dt)
        for d in diags)


def select_chain(M, X, adjoint, select_in, select_out, tables, m):
    """M X or M^H X with the elements of X's columns and / or those of the result
    (m of them) selected by the index tables that tables() returns
    (Fourier._run_select; tables() is None where there are none), for a Fourier
    matrix or a Product of one with a Diag on either or both sides of it; None
    where the passes cannot do that.

    The Diag factors run inside the passes where that holds without selection;
    otherwise a Diag on a side that is not selected runs apart."""
    if type(M) is Product:
        factors = M._content if adjoint else M._content[::-1]
        scalar = M._scalar != 1
    else:
        factors, scalar = (M,), False
    if len(factors) > 3:
        return None
    pre = factors[0] if type(factors[0]) is Diag else None
    f = int(pre is not None)
    F, flip = _as_fourier(factors[f]) if f < len(factors) else (None, False)
    post = factors[f + 1] if f + 1 < len(factors) and type(factors[f + 1]) is Diag else None
    if F is None or f + 1 + (post is not None) != len(factors):
        return None
    # the type that the transform takes, by M's rules and (real data becomes complex) its
    # own; the data follows once it is to run here
    t = D.input_type(X.dtype, M._minType, M.dtype, M._widenInputDatatype)
    if type(M) is Product:
        t = D.torch_dtype(D.promote(t, M.dtype))
    if pre is None:
        t = D.torch_dtype(F.compute_dtype(
            D.input_type(t, F._minType, F.dtype, F._widenInputDatatype)))
    if not F._select_ok(t):
        return None
    inside = _diags_ok(F, t, pre, post)
    if not inside and ((pre is not None and select_in) or (post is not None and select_out)):
        return None
    inverse = adjoint != flip
    diags = _diag_tables(D.np_dtype(t), inverse != adjoint,
                         *((pre, post) if inside else (None, None)))
    index = None if diags is None else tables()
    if index is None:
        return None
    if X.dtype is not t:
        X = X.to(t)
    if scalar:
        X = M._prep(X, adjoint and np.iscomplexobj(M._scalar))
    if pre is not None and not inside:
        X = pre._apply(X, adjoint)
        if not F._select_ok(X.dtype):
            return None
    Y = F._run_select(X, inverse, *diags, *index, m)
    if Y is not None and post is not None and not inside:
        Y = post._apply(Y, adjoint)
    return Y


def _as_fourier(f):
    """(Fourier, False) for a Fourier matrix, (Fourier, True) for its Hermitian,
    (None, False) otherwise."""
    if type(f) is Fourier:
        return f, False
    if type(f) is Hermitian and type(f._nested) is Fourier:
        return f._nested, True
    return None, False
