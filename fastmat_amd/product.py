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
    if F is None or (pre is None and post is None) or not F._diag_ok(X):
        return None
    dt = D.np_dtype(X.dtype)
    if not all(d is None or (D.promote(dt, d.dtype) == dt and D.promote(dt, d._minType) == dt)
               for d in (pre, post)):
        return None
    # the transform conjugates its tables when it is an adjoint one; a Diag's
    # adjoint is its conjugate
    inverse = adjoint != flip
    Y = F._run_diag(X, inverse, None if pre is None else pre._table(dt, inverse != adjoint),
                    None if post is None else post._table(dt, inverse != adjoint))
    return Y, f + 1 + (post is not None)


def _as_fourier(f):
    """(Fourier, False) for a Fourier matrix, (Fourier, True) for its Hermitian,
    (None, False) otherwise."""
    if type(f) is Fourier:
        return f, False
    if type(f) is Hermitian and type(f._nested) is Fourier:
        return f._nested, True
    return None, False
