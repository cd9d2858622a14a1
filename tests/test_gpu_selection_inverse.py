"""A selection's inverse from the host and from the device: the same tables, for
repeated and negative indices too (the last of equal ones), and the same products."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _selection(rng, n, kind):
    if kind == "all":
        return rng.permutation(n)
    if kind == "repeated":
        return rng.integers(0, n, n)
    if kind == "one":
        return np.array([n - 1])
    if kind == "negative":  # (let through at full length and of arange's sum)
        return np.concatenate([[-1, 2], np.arange(2, n)])
    return np.sort(rng.permutation(n)[:max(1, n // 3)])


@pytest.mark.parametrize("dtype", ["int32", "int64"])
@pytest.mark.parametrize("kind", ["some", "all", "repeated", "one"])
@pytest.mark.parametrize("n,m", [(2, 3), (255, 1), (256, 257), (1000, 4099)])
def test_tables(n, m, kind, dtype, monkeypatch):
    import torch

    import fastmat_amd as fm
    from fastmat_amd import partial
    rng = np.random.default_rng(n + m)
    rows, cols = _selection(rng, n, kind), _selection(rng, m, kind)
    M = fm.Matrix(np.ones((n, m), np.float32))
    dt = getattr(torch, dtype)
    made = []
    print("tables", n, m, kind, dtype, flush=True)
    for host in (1 << 20, 0):
        monkeypatch.setattr(partial, "_HOST_TABLE", host)
        P = fm.Partial(M, rows=rows, cols=cols)
        made.append([(P._inverse(s, dt).cpu().numpy()[:size], P._distinct(s),
                      P._idx(s).cpu().numpy()) for s, size in (("r", n), ("c", m))])
    for sel, size, a, b in zip((rows, cols), (n, m), *made):
        ref = np.full(size, -1)
        ref[sel] = np.arange(len(sel))
        for table, distinct, idx in (a, b):
            np.testing.assert_array_equal(table, ref)
            np.testing.assert_array_equal(idx, sel)
            assert distinct == (len(np.unique(sel)) == len(sel))


@pytest.mark.parametrize("adjoint", [False, True])
@pytest.mark.parametrize("kind", ["some", "repeated", "negative"])
@pytest.mark.parametrize("name", ["fourier", "hadamard"])
def test_products(name, kind, adjoint, monkeypatch):
    import torch

    import fastmat_amd as fm
    from fastmat_amd import partial
    n, k = 256, 3
    rng = np.random.default_rng(n)
    rows = _selection(rng, n, kind)
    cols = _selection(rng, n, "some")
    M = fm.Fourier(n) if name == "fourier" else fm.Hadamard(8)
    x = rng.integers(-9, 10, (len(rows) if adjoint else len(cols), k)).astype(np.complex64)
    outs = []
    print("products", name, kind, adjoint, flush=True)
    for host in (1 << 20, 0):
        monkeypatch.setattr(partial, "_HOST_TABLE", host)
        P = fm.Partial(M, rows=rows, cols=cols)
        outs.append((P.backward if adjoint else P.forward)(torch.from_numpy(x).cuda()))
    assert torch.equal(*outs)
    full = np.zeros((n, k), np.complex128)
    dense = np.fft.fft(np.eye(n)) if name == "fourier" else M.reference().astype(np.complex128)
    if adjoint:
        full[rows] = x
        ref = (dense.conj().T @ full)[cols]
    else:
        full[cols] = x
        ref = (dense @ full)[rows]
    # 16 u of the largest value, as for the transform alone
    assert np.abs(outs[0].cpu().numpy() - ref).max() <= 16 * 1.2e-7 * np.abs(ref).max()
