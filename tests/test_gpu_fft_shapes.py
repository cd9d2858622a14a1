"""One-pass transforms and convolutions in both launch shapes of contiguous columns: up
to 2^20 elements and above, at every length, with a last tile that is not full.

Bounds: an FFT of length N in precision u is off by at most about 6 u log2(N) of its
result's norm (Higham, Accuracy and Stability, 24.1: eta = mu + sqrt(2) gamma_4 a level,
mu the twiddles' error); a convolution is two of them and a product by the spectrum, of
the operand's norm times the spectrum's largest value."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [(np.complex64, 13), (np.complex128, 12)]


def _data(k, n, dtype, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn((k, n), generator=g, device="cuda", dtype=torch.complex128).to(dtype)


@pytest.mark.parametrize("over", [False, True])
@pytest.mark.parametrize("dtype,logn", [(d, e) for d, top in CASES for e in range(1, top + 1)])
def test_one_pass(dtype, logn, over):
    import torch

    import fastmat_amd as fm
    n = 1 << logn
    k = (1 << 20) // n + (3 if over else 0)
    u = float(np.finfo(dtype).eps) / 2
    t = torch.complex64 if dtype is np.complex64 else torch.complex128
    X = _data(k, n, t, logn)
    Xd = X.to(torch.complex128)
    norm = Xd.norm(dim=1)
    print("one pass", np.dtype(dtype).name, n, k, flush=True)
    F = fm.Fourier(n)
    for adjoint in (False, True):
        ref = torch.fft.ifft(Xd, norm="forward") if adjoint else torch.fft.fft(Xd)
        err = (F._apply(X, adjoint).to(torch.complex128) - ref).norm(dim=1)
        assert bool((err <= 6 * u * logn * math.sqrt(n) * norm).all())
    c = _data(1, n, torch.complex128, 99)[0]
    C = fm.Circulant(c.to(t).cpu().numpy())
    S = torch.fft.fft(c.to(t).to(torch.complex128))
    for adjoint in (False, True):
        ref = torch.fft.ifft(torch.fft.fft(Xd) * (S.conj() if adjoint else S))
        err = (C._apply(X, adjoint).to(torch.complex128) - ref).norm(dim=1)
        assert bool((err <= (12 * logn + 8) * u * S.abs().max() * norm).all())
