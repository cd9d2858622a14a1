"""An operator is freed with its last reference: no cycle through its plan cache
leaves the freeing of its device memory to the cycle collector, which may run
inside a stream capture."""
import gc
import weakref

import numpy as np
import pytest

import fastmat_amd as fm


@pytest.mark.parametrize("make", [lambda: fm.Fourier(8), lambda: fm.Circulant(np.arange(5.)),
                                  lambda: fm.Toeplitz(np.arange(4.), np.arange(3.))])
def test_operator_goes_with_its_last_reference(make):
    gc.collect()
    gc.disable()
    try:
        op = make()
        if hasattr(op, "_clone_plan"):
            from fastmat_amd.fourier import _PlanCache
            op._gplans = _PlanCache(op._clone_plan, "fm_conv_plan_destroy")
        gone = weakref.ref(op)
        del op
        assert gone() is None
    finally:
        gc.enable()


def test_plan_cache_asks_its_owner_once():
    from fastmat_amd.fourier import _PlanCache

    class Owner:
        def __init__(self):
            self.made = []
            self.cache = _PlanCache(self.make, "none")

        def make(self, prec):
            self.made.append(prec)
            return object()
    o = Owner()
    assert o.cache.get(6) is o.cache.get(6) and o.cache.get(7) is not o.cache.get(6)
    assert o.made == [6, 7]
