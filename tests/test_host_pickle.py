"""Operators without native plans go through pickle (a spawned worker's arguments),
also inside containers, and make and free their plans as before."""
import pickle
import weakref

import numpy as np
import pytest

import fastmat_amd as fm


@pytest.mark.parametrize("make", [
    lambda: fm.Fourier(8), lambda: fm.Circulant(np.arange(5.)),
    lambda: fm.Toeplitz(np.arange(4.), np.arange(3.)),
    lambda: fm.Kron(fm.Fourier(4), fm.Eye(3)), lambda: fm.Partial(fm.Fourier(6), rows=[1, 2]),
    lambda: fm.Product(fm.Fourier(4).H, fm.Diag(np.arange(4.)), fm.Fourier(4))])
def test_round_trip(make):
    op = make()
    back = pickle.loads(pickle.dumps(op))
    assert type(back) is type(op) and back.shape == op.shape and back.dtype == op.dtype
    np.testing.assert_array_equal(back.reference(), op.reference())
    again = pickle.loads(pickle.dumps([back, {"op": back}]))
    assert again[0] is again[1]["op"]


def test_the_cache_asks_the_owner_that_was_loaded(monkeypatch):
    made = []

    def _make_plan(self, prec):
        made.append((self, prec))
        return 1
    monkeypatch.setattr(fm.Fourier, "_make_plan", _make_plan)
    back = pickle.loads(pickle.dumps(fm.Fourier(8)))
    assert back._plans.get(6) == 1 and made[0][0] is back
    gone = weakref.ref(back)
    back._plans._plans.clear()
    made.clear()
    del back
    assert gone() is None
