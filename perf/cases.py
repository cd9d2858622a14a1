"""The work that a user of fastmat_amd has it do, as cases that can be timed.

Every case is one pass over the public entry points with its data resident on
the GPU: an operator's forward and backward (its adjoint), a training step
with gradients, or a solver run.  ``listed()`` are the cases, ``draw(rng)``
gives further ones of the same ranges, ``prepare`` makes inputs and operators
from a seed, ``run`` is one pass, ``work`` its unavoidable bytes and flops and
``exact`` its result in 64 bits from plain torch.

``layout`` says how the caller holds an (n, k) block of k vectors: "rows" is
torch's default, the vectors' elements k apart; "cols" keeps every vector
contiguous, the (n, k) view that the operators themselves return.
"""
import math

import numpy as np
import torch

import fastmat_amd as fm
from fastmat_amd import algorithms as fma
from fastmat_amd import autograd as fa
from fastmat_amd.batch import ConvBatch

DTYPES = {"int8": torch.int8, "int32": torch.int32, "float32": torch.float32,
          "float64": torch.float64, "complex64": torch.complex64,
          "complex128": torch.complex128}


def listed():
    return [
        # one short vector: the latency of a call in a user's own loop
        dict(name="fourier_vector", kind="fourier", n=1024, k=1, dtype="complex64",
             layout="cols"),
        # a small block in double precision, forward and adjoint
        dict(name="circulant_double", kind="circulant", n=4096, k=32, dtype="complex128",
             layout="rows"),
        # long transforms over many columns, a power of two and a prime length
        dict(name="fourier_2p20", kind="fourier", n=1 << 20, k=64, dtype="complex64",
             layout="cols"),
        dict(name="fourier_prime", kind="fourier", n=1000003, k=64, dtype="complex64",
             layout="cols"),
        dict(name="hadamard_2p20", kind="hadamard", order=20, k=64, dtype="float32",
             layout="cols"),
        # mode-wise product of three factors on 2^20-element vectors
        dict(name="kron_three", kind="kron", f=64, c=128, d=128, k=16, layout="cols"),
        # a filter of ragged size that is trained: output, input gradient and
        # generator gradient of one rectangular Toeplitz operator
        dict(name="toeplitz_train", kind="toeplitz", m=60011, n=45007, k=24, layout="rows"),
        # dense factors: a real matrix in single precision, and a ragged
        # complex one in double precision
        dict(name="dense_single", kind="dense", m=2048, n=3072, k=1024, dtype="float32",
             layout="rows"),
        dict(name="dense_double", kind="dense", m=1000, n=777, k=130, dtype="complex128",
             layout="rows"),
        # compressed sensing: random rows of a Fourier matrix behind a diagonal
        dict(name="sensing", kind="sensing", n=1 << 18, rows=70001, k=32, layout="rows"),
        # sparse recovery: 50 FISTA iterations on a circulant operator
        dict(name="fista", kind="fista", n=1 << 18, k=8, steps=50, layout="cols"),
        # training step of 256 uneven operators: loss, all input gradients and
        # all generator gradients, replayed from a captured graph
        dict(name="batch_train", kind="batch", ops=256, lo=256, hi=65536, kmax=32, spec=20261206),
    ]


def _log(rng, lo, hi):
    """A size whose logarithm is uniform over [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["fourier", "fourier", "circulant", "hadamard", "kron", "toeplitz",
                       "dense", "sensing", "fista", "batch"])
    layout = rng.choice(["rows", "cols"])
    if kind == "fourier":
        n = 1 << rng.randint(6, 20) if rng.random() < 0.5 else _log(rng, 60, 1000003)
        k = _log(rng, 1, min(4096, 64000000 // n))
        dtype = rng.choice(["complex64", "complex64", "complex128"])
        return dict(kind=kind, n=n, k=max(1, k // 2) if dtype == "complex128" else k,
                    dtype=dtype, layout=layout)
    if kind == "circulant":
        n = 1 << rng.randint(8, 19) if rng.random() < 0.4 else _log(rng, 250, 500000)
        return dict(kind=kind, n=n, k=_log(rng, 1, min(512, 16000000 // n)),
                    dtype=rng.choice(["complex64", "complex128"]), layout=layout)
    if kind == "hadamard":
        order = rng.randint(8, 20)
        return dict(kind=kind, order=order, k=_log(rng, 1, min(4096, (1 << 26) >> order)),
                    dtype=rng.choice(["int8", "int32", "float32", "float32", "float64"]),
                    layout=layout)
    if kind == "kron":
        f, c, d = 1 << rng.randint(4, 7), rng.choice([64, 100, 128, 128]), rng.choice(
            [64, 96, 128, 128])
        return dict(kind=kind, f=f, c=c, d=d, k=_log(rng, 1, (1 << 24) // (f * c * d)),
                    layout=layout)
    if kind == "toeplitz":
        m = _log(rng, 256, 100000)
        n = max(2, int(m * rng.uniform(0.5, 1.5)))
        return dict(kind=kind, m=m, n=n, k=_log(rng, 1, min(64, 4000000 // m)), layout=layout)
    if kind == "dense":
        m, n, k = _log(rng, 50, 2500), _log(rng, 50, 2500), _log(rng, 1, 1000)
        return dict(kind=kind, m=m, n=n, k=k, layout=layout,
                    dtype=rng.choice(["float32", "float32", "complex64", "float64",
                                      "complex128"]))
    if kind == "sensing":
        n = 1 << rng.randint(10, 18) if rng.random() < 0.6 else _log(rng, 1000, 200000)
        return dict(kind=kind, n=n, rows=max(1, int(n * rng.uniform(0.1, 0.6))),
                    k=_log(rng, 1, min(256, 8000000 // n)), layout=layout)
    if kind == "fista":
        n = 1 << rng.randint(11, 18) if rng.random() < 0.6 else _log(rng, 2000, 120000)
        return dict(kind=kind, n=n, k=_log(rng, 1, min(64, 2000000 // n)),
                    steps=rng.randint(10, 50), layout="cols")
    return dict(kind=kind, ops=rng.randint(16, 160), lo=256, hi=_log(rng, 2000, 65536),
                kmax=rng.randint(4, 32), spec=rng.randint(1, 1 << 30))


# ---------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _values(g, shape, dtype):
    if dtype in (torch.int8, torch.int32):
        return torch.randint(-8, 9, shape, generator=g, device="cuda", dtype=dtype)
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype)


def _block(g, n, k, dtype, layout):
    if layout == "rows":
        return _values(g, (n, k), dtype)
    return _values(g, (k, n), dtype).t()


def _host(t):
    return t.cpu().numpy()


def _batch_spec(case):
    """[(kind, rows, cols, columns of data)] of the uneven batch: half
    Circulant, half Toeplitz, sizes log-uniform."""
    rng = np.random.default_rng(case["spec"])
    lo, hi = math.log(case["lo"]), math.log(case["hi"])
    out = []
    for i in range(case["ops"]):
        k = int(rng.integers(1, case["kmax"] + 1))
        m = int(round(math.exp(rng.uniform(lo, hi))))
        if i % 2 == 0:
            out.append(("circulant", m, m, k))
        else:
            n = min(max(int(round(m / rng.uniform(0.5, 2.0))), case["lo"]), case["hi"])
            out.append(("toeplitz", m, n, k))
    return out


def _batch_data(case, seed):
    spec = _batch_spec(case)
    g = _gen(seed)
    lens = [n if kind == "circulant" else m + n - 1 for kind, m, n, _ in spec]
    c64 = torch.complex64
    theta = _values(g, (sum(lens),), c64)
    xp = _values(g, (sum(n * k for _, _, n, k in spec),), c64)
    yp = _values(g, (sum(m * k for _, m, _, k in spec),), c64)
    return spec, lens, theta, xp, yp


def _fista_data(case, seed):
    """A decaying band-limited kernel with largest singular value near one,
    and the measurements of spiky vectors behind it with a little noise."""
    n, k = case["n"], case["k"]
    g = _gen(seed)
    f = torch.arange(n, device="cuda", dtype=torch.float64)
    f = torch.minimum(f, n - f) / n
    jitter = torch.rand((), generator=g, device="cuda", dtype=torch.float64)
    c = torch.fft.ifft(0.2 + 0.8 * torch.exp(-(f * (6 + jitter)) ** 2)).real.float()
    x = torch.randn((k, n), generator=g, device="cuda")
    x = x * (torch.rand((k, n), generator=g, device="cuda") < 0.0625)
    b = torch.fft.ifft(torch.fft.fft(c.double()) * torch.fft.fft(x.double()))
    b = b + 1e-3 * torch.randn((k, n), generator=g, device="cuda", dtype=torch.complex128)
    return c, b.to(torch.complex64).t()


FISTA_LAMBDA = 2e-4


def _operands(case, seed):
    """Inputs of the operator cases, from the seed alone: the operator's
    defining arrays and the forward's and the adjoint's data."""
    g = _gen(seed)
    kind, k, lay = case["kind"], case["k"], case["layout"]
    dt = DTYPES[case.get("dtype", "complex64")]
    if kind == "fourier":
        return (), _block(g, case["n"], k, dt, lay), _block(g, case["n"], k, dt, lay)
    if kind == "circulant":
        c = _values(g, (case["n"],), dt)
        return (c,), _block(g, case["n"], k, dt, lay), _block(g, case["n"], k, dt, lay)
    if kind == "hadamard":
        n = 1 << case["order"]
        return (), _block(g, n, k, dt, lay), _block(g, n, k, dt, lay)
    if kind == "kron":
        c = _values(g, (case["c"],), dt)
        a = _values(g, (case["d"], case["d"]), torch.float32) / math.sqrt(case["d"])
        n = case["f"] * case["c"] * case["d"]
        return (c, a), _block(g, n, k, dt, lay), _block(g, n, k, dt, lay)
    if kind == "toeplitz":
        t = _values(g, (case["m"] + case["n"] - 1,), dt)
        return (t,), _block(g, case["n"], k, dt, lay), _block(g, case["m"], k, dt, lay)
    if kind == "dense":
        a = _values(g, (case["m"], case["n"]), dt)
        return (a,), _block(g, case["n"], k, dt, lay), _block(g, case["m"], k, dt, lay)
    d = _values(g, (case["n"],), dt)  # sensing
    sel = torch.randperm(case["n"], generator=g, device="cuda")[:case["rows"]]
    return (d, sel), _block(g, case["n"], k, dt, lay), _block(g, case["rows"], k, dt, lay)


def _operator(case, arrays):
    kind = case["kind"]
    if kind == "fourier":
        return fm.Fourier(case["n"], dtype=np.dtype(case["dtype"]))
    if kind == "circulant":
        return fm.Circulant(_host(arrays[0]))
    if kind == "hadamard":
        return fm.Hadamard(case["order"])
    if kind == "kron":
        return fm.Kron(fm.Fourier(case["f"]), fm.Circulant(_host(arrays[0])),
                       fm.Matrix(_host(arrays[1])))
    if kind == "toeplitz":
        t = _host(arrays[0])
        return fm.Toeplitz(t[:case["m"]], t[case["m"]:])
    if kind == "dense":
        return fm.Matrix(_host(arrays[0]))
    d, sel = arrays
    return fm.Partial(fm.Product(fm.Fourier(case["n"]), fm.Diag(_host(d))), rows=_host(sel))


def prepare(case, seed):
    if case["kind"] == "batch":
        return _prepare_batch(case, seed)
    if case["kind"] == "fista":
        c, b = _fista_data(case, seed)
        return dict(kind="fista", b=b, solver=fma.FISTA(
            fm.Circulant(_host(c)), numLambda=FISTA_LAMBDA, numMaxSteps=case["steps"]))
    arrays, x, y = _operands(case, seed)
    state = dict(kind=case["kind"], op=_operator(case, arrays), x=x, y=y)
    if case["kind"] == "toeplitz":
        state["gen"] = arrays[0].requires_grad_(True)
        state["x"] = x.requires_grad_(True)
    return state


def _prepare_batch(case, seed):
    """The operators, packed data and flat parameter vector of a training
    loop, with its step captured after eager warm-up steps."""
    spec, lens, theta, xp, yp = _batch_data(case, seed)
    ops, ks = [], []
    for (kind, m, _, k), gen in zip(spec, np.split(_host(theta), np.cumsum(lens)[:-1])):
        ops.append(fm.Circulant(gen) if kind == "circulant" else fm.Toeplitz(gen[:m], gen[m:]))
        ks.append(k)
    batch = ConvBatch(ops, ks)
    batch.set_schedule(8, 512, 3)
    theta.requires_grad_(True)
    xp.requires_grad_(True)

    def step():
        theta.grad = xp.grad = None
        loss = fa.batch_least_squares_packed(batch, theta.split(lens), xp, yp)
        loss.backward()
        return loss

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    theta.grad = xp.grad = None
    with torch.cuda.graph(graph):
        loss = step()
    return dict(kind="batch", batch=batch, graph=graph, theta=theta, xp=xp, yp=yp,
                out=[loss.detach(), xp.grad, theta.grad])


# ------------------------------------------------------------------ run
def run(state):
    kind = state["kind"]
    if kind == "batch":
        state["graph"].replay()
        return state["out"]
    if kind == "fista":
        return state["solver"].process(state["b"])
    if kind == "toeplitz":
        out = fa.conv_matvec(state["op"], state["gen"], state["x"])
        gx, gt = torch.autograd.grad(out, (state["x"], state["gen"]), state["y"])
        return [out.detach(), gx, gt]
    op = state["op"]
    return [op.forward(state["x"]), op.backward(state["y"])]


# ----------------------------------------------------------------- work
def _fft_flops(n, k):
    return 5.0 * n * max(1.0, math.log2(n)) * k


def work(case):
    kind = case["kind"]
    if kind == "batch":
        by = fl = 0.0
        for name, m, n, k in _batch_spec(case):
            gen = n if name == "circulant" else m + n - 1
            # x, target, x gradient; generator and its gradient
            by += 8.0 * ((2 * n + m) * k + 2 * gen)
            # transforms of x, residual, output and x gradient, and of the
            # generator and its gradient
            fl += 4 * _fft_flops(m + n, k) + 2 * _fft_flops(m + n, 1)
        return {"bytes": by, "flops": fl}
    k = case["k"]
    esz = DTYPES[case.get("dtype", "complex64")].itemsize
    if kind == "fourier":
        n = case["n"]
        return {"bytes": 4.0 * n * k * esz, "flops": 2 * _fft_flops(n, k)}
    if kind == "circulant":
        n = case["n"]
        return {"bytes": (4.0 * n * k + n) * esz, "flops": 4 * _fft_flops(n, k)}
    if kind == "hadamard":
        n = 1 << case["order"]
        return {"bytes": 4.0 * n * k * esz, "flops": 2.0 * n * case["order"] * k}
    if kind == "kron":
        f, c, d = case["f"], case["c"], case["d"]
        n = f * c * d
        return {"bytes": 4.0 * n * k * 8 + 4.0 * d * d + 8.0 * c,
                "flops": 2 * (_fft_flops(f, n // f * k) + 2 * _fft_flops(c, n // c * k) +
                              4.0 * d * n * k)}
    if kind == "toeplitz":
        m, n = case["m"], case["n"]
        return {"bytes": 8.0 * (2 * (m + n) * k + 2 * (m + n - 1)),
                "flops": 4 * _fft_flops(m + n, k) + 2 * _fft_flops(m + n, 1)}
    if kind == "dense":
        m, n = case["m"], case["n"]
        mul = 8.0 if case["dtype"].startswith("complex") else 2.0
        return {"bytes": (m * n + 2.0 * (m + n) * k) * esz, "flops": 2 * mul * m * n * k}
    if kind == "sensing":
        n, rows = case["n"], case["rows"]
        return {"bytes": 8.0 * (2 * (n + rows) * k + n) + 8.0 * rows,
                "flops": 2 * _fft_flops(n, k) + 12.0 * n * k}
    n, steps = case["n"], case["steps"]  # fista
    return {"bytes": 8.0 * (2 * n * k + n),
            "flops": steps * (4 * _fft_flops(n, k) + 30.0 * n * k)}


# ---------------------------------------------------------------- exact
def _circular64(a, b, L):
    """Circular convolution of length L of (k, <= L) blocks or vectors, as a
    linear one of power-of-two length folded onto L (torch builds a plan for
    every length it meets, and a batch has many)."""
    P = 1 << (2 * L - 1).bit_length()
    y = torch.fft.ifft(torch.fft.fft(a, n=P) * torch.fft.fft(b, n=P))
    return y[..., :L] + y[..., L:2 * L]


def _mirror64(a, L):
    """conj(a[-j mod L]) of (k, <= L) blocks or vectors zero-padded to L."""
    a = torch.nn.functional.pad(a, (0, L - a.shape[-1])).conj()
    return torch.cat((a[..., :1], a[..., 1:].flip(-1)), dim=-1)


def _conv64(t, x, rows, adjoint=False):
    """Product of the length-L circulant of t (complex128) with the (k, n)
    block x zero-padded to L, its first `rows` entries: a Circulant's c, or a
    Toeplitz matrix's [vecC, vecR], whose L is m + n - 1."""
    L = t.numel()
    return _circular64(_mirror64(t, L) if adjoint else t, x, L)[:, :rows]


def _grad64(x, g, t):
    """sum over columns of the circular correlation of g with x."""
    return _circular64(g, _mirror64(x, t.numel()), t.numel()).sum(0)


def exact(case, seed):
    kind = case["kind"]
    c128 = torch.complex128
    if kind == "batch":
        spec, lens, theta, xp, yp = _batch_data(case, seed)
        loss, gx, gt = 0.0, [], []
        xo = yo = go = 0
        for (name, m, n, k), length in zip(spec, lens):
            t = theta[go:go + length].to(c128)
            x = xp[xo:xo + n * k].view(k, n).to(c128)
            y = yp[yo:yo + m * k].view(k, m).to(c128)
            r = _conv64(t, x, m) - y
            loss += float((r.real ** 2 + r.imag ** 2).sum())
            gx.append(_conv64(t, 2 * r, n, adjoint=True).reshape(-1))
            gt.append(_grad64(x, 2 * r, t))
            xo, yo, go = xo + n * k, yo + m * k, go + length
        return [torch.tensor(loss, dtype=torch.float64), torch.cat(gx), torch.cat(gt)]
    if kind == "fista":
        return _fista64(case, seed)
    arrays, x, y = _operands(case, seed)
    if kind == "hadamard":
        return [_hadamard64(x), _hadamard64(y)]
    if kind == "dense":
        wide = c128 if x.is_complex() else torch.float64
        a = arrays[0].to(wide)
        return [a @ x.to(wide).contiguous(), a.mH.contiguous() @ y.to(wide).contiguous()]
    X, Y = x.to(c128).t().contiguous(), y.to(c128).t().contiguous()
    if kind == "fourier":
        return [torch.fft.fft(X, dim=1).t(), torch.fft.ifft(Y, dim=1, norm="forward").t()]
    if kind == "circulant":
        t = arrays[0].to(c128)
        return [_conv64(t, X, t.numel()).t(), _conv64(t, Y, t.numel(), adjoint=True).t()]
    if kind == "toeplitz":
        t = arrays[0].to(c128)
        return [_conv64(t, X, case["m"]).t(), _conv64(t, Y, case["n"], adjoint=True).t(),
                _grad64(X, Y, t)]
    if kind == "kron":
        return [_kron64(case, arrays, X, False).t(), _kron64(case, arrays, Y, True).t()]
    d, sel = arrays[0].to(c128), arrays[1]  # sensing
    back = torch.zeros_like(X)
    back[:, sel] = Y
    return [torch.fft.fft(X * d, dim=1)[:, sel].t(),
            (torch.fft.ifft(back, dim=1, norm="forward") * d.conj()).t()]


def _hadamard64(x):
    n, k = x.shape
    v = x.t().contiguous().to(torch.int64 if x.dtype in (torch.int8, torch.int32)
                              else torch.float64)
    h = 1
    while h < n:
        w = v.view(k, n // (2 * h), 2, h)
        v = torch.stack((w[:, :, 0] + w[:, :, 1], w[:, :, 0] - w[:, :, 1]), dim=2).view(k, n)
        h *= 2
    return v.t().to(x.dtype) if v.dtype == torch.int64 else v.t()


def _kron64(case, arrays, X, adjoint):
    f, c, d = case["f"], case["c"], case["d"]
    k = X.shape[0]
    v = X.view(k, f, c, d)
    if adjoint:
        v = torch.fft.ifft(v, dim=1, norm="forward")
    else:
        v = torch.fft.fft(v, dim=1)
    s = torch.fft.fft(arrays[0].to(torch.complex128)).view(1, 1, c, 1)
    v = torch.fft.ifft(torch.fft.fft(v, dim=2) * (s.conj() if adjoint else s), dim=2)
    a = arrays[1].to(torch.complex128)
    a = (a if adjoint else a.t()).contiguous()
    return (v.reshape(-1, d).contiguous() @ a).view(k, f * c * d)


def _fista64(case, seed):
    c, b = _fista_data(case, seed)
    s = torch.fft.fft(c.to(torch.complex128))
    B = b.to(torch.complex128).t().contiguous()
    L = float(1.0 / s.abs().max() ** 2)
    alpha = L * FISTA_LAMBDA * 0.5
    x = torch.zeros_like(B)
    y, t = x, 1.0
    for _ in range(case["steps"]):
        old, t_old = x, t
        r = torch.fft.ifft(torch.fft.fft(y, dim=1) * s, dim=1) - B
        step = y - L * torch.fft.ifft(torch.fft.fft(r, dim=1) * s.conj(), dim=1)
        m = torch.clamp(step.abs() - alpha, min=0)
        x = m / (m + alpha) * step
        t = (1 + math.sqrt(1 + 4 * t * t)) / 2
        y = x + (t_old - 1) / t * (x - old)
    return torch.where(x != 0, step, x).t()
