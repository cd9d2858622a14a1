"""A selection's tables are kept for good once they are there: a captured graph holds
their addresses."""
import numpy as np
import pytest


@pytest.mark.parametrize("nested", ["fourier", "eye"])
@pytest.mark.parametrize("first", ["index", "int32", "int64"])
def test_a_kept_table_stays(nested, first, monkeypatch):
    import torch

    import fastmat_amd as fm
    from fastmat_amd import _device as D
    monkeypatch.setattr(D, "_device", torch.device("cpu"))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    n = 64
    P = fm.Partial(fm.Fourier(n) if nested == "fourier" else fm.Eye(n),
                   rows=np.arange(0, n, 3), cols=np.arange(5, n))
    make = {"index": lambda s: P._idx(s), "int32": lambda s: P._inverse(s, torch.int32),
            "int64": lambda s: P._inverse(s, torch.int64)}
    kept = {s: make[first](s) for s in "rc"}
    for how in make.values():
        for s in "cr":
            how(s)
    for s in "rc":
        assert make[first](s) is kept[s]
        sel = P.rowSelection if s == "r" else P.colSelection
        ref = np.full(n, -1)
        ref[sel] = np.arange(len(sel))
        for dtype in (torch.int32, torch.int64):
            np.testing.assert_array_equal(P._inverse(s, dtype).numpy()[:n], ref)
        np.testing.assert_array_equal(P._idx(s).numpy(), sel)
