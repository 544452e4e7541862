"""Workloads of the adjoint NFFT library, for measuring it.

Each case is one call (or one short sequence of calls) that a program using the
package makes, through its public entry points, on inputs of the kind it meets:
unevenly sampled light curves, clustered or uniform sample positions, FP64 times
with a frequency step, both precisions, the reference-compatible interface
(device and host) and the extensions (several value vectors, type-2 transform,
gradients, bootstrap, Lomb-Scargle).

`exact` restates each path in 64 bits with plain torch: a Gaussian-gridding
transform at oversampling 4 and half-width 16 (its own error is below 1e-14 of
the result's norm), or the reference formula with its per-point decisions taken
in the precision of the library under measurement.
"""
import math
import random

import numpy as np
import torch

import cunfft_adjoint_amd as cu
from cunfft_adjoint_amd.autograd import adjoint_nfft

DEV = "cuda"
REAL = {"f32": torch.float32, "f64": torch.float64}
CPLX = {"f32": torch.complex64, "f64": torch.complex128}
SIZE = {"f32": 4, "f64": 8}
HALF_WIDTH = {"f32": 8, "f64": 13}  # default m of the two libraries
BASELINE_DAYS = 3650.0
SEED = 2024


def listed():
    return [
        # One short light curve, plan kept: the smallest call, launches and host work only.
        {"name": "adjoint_small_f32", "kind": "adjoint", "n": 1000, "M": 1 << 11, "dtype": "f32", "points": "uniform"},
        # The package's headline: a million clustered points, a million modes, plan kept, new values.
        {"name": "adjoint_large_f32", "kind": "adjoint", "n": 1000000, "M": 1 << 20, "dtype": "f32", "points": "clustered"},
        # The same range in double precision, with a ragged point count.
        {"name": "adjoint_large_f64", "kind": "adjoint", "n": 999983, "M": 1 << 20, "dtype": "f64", "points": "clustered"},
        # Several value vectors of one sampling (bands, or data and noise realisations): the largest transform call.
        {"name": "many_f32", "kind": "many", "n": 1000000, "M": 1 << 20, "nrhs": 8, "dtype": "f32", "points": "clustered"},
        # Type-2 transform: a spectrum evaluated at uneven sample positions.
        {"name": "forward_f32", "kind": "forward", "n": 300007, "M": 1 << 18, "dtype": "f32", "points": "clustered"},
        # A training step through the transform: new positions, output and both gradients.
        {"name": "train_f32", "kind": "train", "curves": 64, "n": 20000, "M": 1 << 16, "dtype": "f32"},
        # A survey's light curves, FP64 times seen for the first time: plan and spectra of a ragged batch.
        {"name": "survey_f32", "kind": "survey", "curves": 256, "nmin": 100, "nmax": 20000, "M": 1 << 14, "dtype": "f32"},
        # Bootstrap of a ragged batch, spectra of the resampled data and of their window.
        {"name": "bootstrap_f32", "kind": "bootstrap", "curves": 128, "nmin": 100, "nmax": 50000, "M": 1 << 14, "nbs": 25, "dtype": "f32"},
        # Periodogram percentiles of the same kind of batch: Lomb-Scargle power of every replicate.
        {"name": "bootstrap_ls_f32", "kind": "ls", "curves": 64, "nmin": 100, "nmax": 20000, "M": 1 << 13, "nbs": 25, "dtype": "f32"},
        # The reference's formula on a grid of R*N cells, as its test program asks for it.
        {"name": "compat_any_ng_f32", "kind": "compat", "n": 100000, "ng": 300000, "dtype": "f32"},
        # The reference's bootstrap entry, double precision library.
        {"name": "compat_boot_f64", "kind": "compat_boot", "n": 5000, "ng": 1 << 14, "nbs": 64, "dtype": "f64"},
        # The reference's one-call host interface: host arrays in, host spectrum out.
        {"name": "host_call_f64", "kind": "host", "n": 20011, "ng": 1 << 16, "dtype": "f64"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["adjoint", "adjoint", "many", "forward", "train", "survey", "bootstrap", "ls", "compat",
                       "compat", "compat_boot", "host"])
    dtype = rng.choice(["f32", "f64"])
    points = rng.choice(["uniform", "clustered"])
    if kind in ("adjoint", "forward"):
        lg = rng.randint(11, 20 if kind == "adjoint" else 18)
        n = min(1000000, _log_int(rng, (1 << lg) / 4, (1 << lg) * 2))
        return {"kind": kind, "n": n, "M": 1 << lg, "dtype": dtype, "points": points}
    if kind == "many":
        lg = rng.randint(12, 19)
        n = _log_int(rng, (1 << lg) / 4, 1 << lg)
        return {"kind": kind, "n": n, "M": 1 << lg, "nrhs": rng.randint(2, 8), "dtype": dtype, "points": points}
    if kind == "train":
        lg = rng.randint(12, 16)
        curves = _log_int(rng, 1, 64 if lg < 16 else 32)
        return {"kind": kind, "curves": curves, "n": _log_int(rng, (1 << lg) / 8, 20000), "M": 1 << lg, "dtype": dtype}
    if kind == "survey":
        return {"kind": kind, "curves": _log_int(rng, 16, 256), "nmin": 100, "nmax": _log_int(rng, 2000, 20000),
                "M": 1 << rng.randint(12, 14), "dtype": dtype}
    if kind in ("bootstrap", "ls"):
        # grids of at most 2^15 cells (f32) / 2^14 (f64) have the fused kernel
        lg = rng.randint(11, 14 if dtype == "f32" else 13)
        return {"kind": kind, "curves": _log_int(rng, 8, 64), "nmin": 100, "nmax": _log_int(rng, 2000, 20000),
                "M": 1 << lg, "nbs": rng.randint(5, 25), "dtype": dtype}
    if kind == "compat":
        n = _log_int(rng, 1000, 100000)
        ng = rng.choice([2 * n, 3 * n, 3 * n + rng.randint(1, 100), 1 << max(4, (2 * n).bit_length())])
        return {"kind": kind, "n": n, "ng": ng, "dtype": dtype}
    if kind == "compat_boot":
        n = _log_int(rng, 300, 5000)
        ng = rng.choice([2 * n + 1, 3 * n, 1 << (2 * n).bit_length()])
        return {"kind": kind, "n": n, "ng": ng, "nbs": rng.randint(8, 48), "dtype": dtype}
    n = _log_int(rng, 300, 20000)
    return {"kind": kind, "n": n, "ng": 1 << (2 * n).bit_length(), "dtype": dtype}


# ------------------------------------------------------------------ inputs --
def _lengths(case):
    """Light-curve lengths, log-uniform over [nmin, nmax], in a fixed mixed order."""
    c, lo, hi = case["curves"], case["nmin"], case["nmax"]
    n = [int(round(lo * (hi / lo) ** ((i + 0.5) / c))) for i in range(c)]
    random.Random(c).shuffle(n)
    return n


def _offsets(case):
    return np.concatenate([[0], np.cumsum(_lengths(case))]).astype(np.int32)


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _points(n, kind, g):
    """Sample positions in [-1/2, 1/2): uniform, or 80 % in 50 Gaussian clumps of width 0.005."""
    x = torch.rand(n, generator=g, device=DEV, dtype=torch.float64) - 0.5
    if kind == "clustered":
        nc = int(round(0.8 * n))
        centres = torch.rand(50, generator=g, device=DEV, dtype=torch.float64) - 0.5
        which = torch.randint(0, 50, (nc,), generator=g, device=DEV)
        x[:nc] = centres[which] + 0.005 * torch.randn(nc, generator=g, device=DEV, dtype=torch.float64)
        x = x[torch.randperm(n, generator=g, device=DEV)]
        x = torch.remainder(x + 0.5, 1.0) - 0.5
    return x


def _real(x, dtype):
    """Positions rounded to the library's precision, still inside [-1/2, 1/2)."""
    x = x.to(REAL[dtype])
    return torch.where(x >= 0.5, torch.full_like(x, -0.5), x).contiguous()


def _signal(x, g, dtype):
    """Three sinusoids plus noise at positions x (cycles over the unit interval)."""
    y = 0.3 * torch.randn(x.shape, generator=g, device=DEV, dtype=torch.float64)
    f = 10.0 + 1e4 * torch.rand(3, generator=g, device=DEV, dtype=torch.float64)
    a = 0.1 + 0.9 * torch.rand(3, generator=g, device=DEV, dtype=torch.float64)
    for i in range(3):
        y = y + a[i] * torch.sin(2 * math.pi * f[i] * x)
    return y.to(REAL[dtype]).contiguous()


def _spectrum(shape, g, dtype):
    r = torch.randn(shape + (2,), generator=g, device=DEV, dtype=REAL[dtype])
    return torch.view_as_complex(r)


def _inputs(case, seed):
    """The arrays of a case, made from the seed alone."""
    g = _gen(seed)
    kind, dt = case["kind"], case["dtype"]
    if kind in ("adjoint", "many"):
        x = _real(_points(case["n"], case["points"], g), dt)
        if kind == "many":
            y = torch.stack([_signal(x.double(), g, dt) for _ in range(case["nrhs"])]).contiguous()
        else:
            y = _signal(x.double(), g, dt)
        return {"x": x, "y": y}
    if kind == "forward":
        x = _real(_points(case["n"], case["points"], g), dt)
        return {"x": x, "fhat": _spectrum((1, case["M"]), g, dt)}
    if kind == "train":
        x = _real(torch.rand(case["curves"], case["n"], generator=g, device=DEV, dtype=torch.float64) - 0.5, dt)
        return {"x": x, "y": _signal(x.double(), g, dt), "g": _spectrum((case["curves"], case["M"]), g, dt)}
    if kind in ("survey", "bootstrap", "ls"):
        offs = _offsets(case)
        t = BASELINE_DAYS * torch.rand(int(offs[-1]), generator=g, device=DEV, dtype=torch.float64)
        cid = torch.repeat_interleave(torch.arange(case["curves"], device=DEV),
                                      torch.tensor(np.diff(offs), device=DEV).long())
        t = torch.sort(t + cid * BASELINE_DAYS)[0] - cid * BASELINE_DAYS  # each curve in time order
        period = torch.exp(math.log(0.1) + math.log(1000.0)
                           * torch.rand(case["curves"], generator=g, device=DEV, dtype=torch.float64))
        y = torch.sin(2 * math.pi * t / period[cid]) + torch.randn(t.shape, generator=g, device=DEV, dtype=torch.float64)
        return {"t": t, "y": y.to(REAL[dt]).contiguous(), "offs": offs, "df": 1.0 / BASELINE_DAYS}
    # the reference interface: positions in [-1/2, 1/2)
    x = _real(_points(case["n"], "uniform", g), dt)
    y = _signal(x.double(), g, dt)
    if kind == "host":
        return {"x": x.cpu().numpy(), "y": y.cpu().numpy()}
    return {"x": x, "y": y}


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    kind, dt = case["kind"], case["dtype"]
    if kind in ("adjoint", "many", "forward"):
        s["plan"] = cu.NFFTPlan(s["x"], case["M"])
    elif kind in ("bootstrap", "ls"):
        s["plan"] = cu.NFFTPlan(t=s["t"], df=s["df"], offsets=s["offs"], M=case["M"], window2=True, dtype=REAL[dt])
    elif kind in ("compat", "compat_boot"):
        s["fp"] = cu.generate_filter_properties(s["x"], case["n"], case["ng"])
    elif kind == "train":
        s["x"].requires_grad_(True)
        s["y"].requires_grad_(True)
    torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    kind, dt = case["kind"], case["dtype"]
    if kind == "adjoint":
        return s["plan"].adjoint(s["y"])
    if kind == "many":
        return s["plan"].adjoint_many(s["y"])
    if kind == "forward":
        return s["plan"].forward(s["fhat"])
    if kind == "train":
        f = adjoint_nfft(s["x"], s["y"], case["M"])
        dx, dy = torch.autograd.grad(f, (s["x"], s["y"]), grad_outputs=s["g"])
        return {"f": f.detach(), "dx": dx, "dy": dy}
    if kind == "survey":
        plan = cu.NFFTPlan(t=s["t"], df=s["df"], offsets=s["offs"], M=case["M"], dtype=REAL[dt])
        return plan.adjoint(s["y"])
    if kind == "bootstrap":
        return s["plan"].bootstrap(s["y"], case["nbs"], seed=SEED, window=True)
    if kind == "ls":
        return s["plan"].bootstrap_ls(s["y"], case["nbs"], seed=SEED, power=True, peak=False)["power"]
    if kind == "compat":
        out = torch.empty(case["ng"], dtype=CPLX[dt], device=DEV)
        cu.cunfft_adjoint_raw_async(s["x"], s["y"], out, case["n"], case["ng"], s["fp"])
        return out
    if kind == "compat_boot":
        out = torch.empty((case["nbs"], case["ng"]), dtype=CPLX[dt], device=DEV)
        cu.cunfft_adjoint_raw_async_bootstrap(s["x"], s["y"], out, case["n"], case["ng"], case["nbs"], s["fp"],
                                              seed=SEED)
        return out
    return cu.cunfft_adjoint(s["x"], s["y"], case["ng"])


# -------------------------------------------------------------------- work --
def work(case):
    """Points read, values read, spectra written; taps and FFT operations of the transforms."""
    kind, b = case["kind"], SIZE[case["dtype"]]
    m2 = 2 * HALF_WIDTH[case["dtype"]]
    if kind in ("survey", "bootstrap", "ls"):
        npts = sum(_lengths(case))
    elif kind == "train":
        npts = case["curves"] * case["n"]
    else:
        npts = case["n"]

    def fft(G):
        return 2.5 * G * math.log2(G)

    if kind in ("adjoint", "many"):
        k = case.get("nrhs", 1)
        M = case["M"]
        return {"bytes": npts * b * (1 + k) + 2 * b * M * k, "flops": k * (2.0 * m2 * npts + fft(2 * M))}
    if kind == "forward":
        M = case["M"]
        return {"bytes": npts * 3 * b + 2 * b * M, "flops": 4.0 * m2 * npts + 2 * fft(2 * M)}
    if kind == "train":
        c, M = case["curves"], case["M"]
        return {"bytes": npts * 4 * b + 2 * (2 * b * M * c), "flops": 6.0 * m2 * npts + 2 * c * fft(2 * M)}
    if kind == "survey":
        c, M = case["curves"], case["M"]
        return {"bytes": npts * (8 + b) + 2 * b * M * c, "flops": 2.0 * m2 * npts + c * fft(2 * M)}
    if kind in ("bootstrap", "ls"):
        c, M, r = case["curves"], case["M"], case["nbs"]
        out = 2 * (2 * b * M) if kind == "bootstrap" else b * (M // 2)
        return {"bytes": npts * (8 + b) + out * c * r, "flops": 2 * r * (2.0 * m2 * npts + c * fft(2 * M))}
    taps = 2 * (6 if case["dtype"] == "f32" else 12) - 1
    k = case.get("nbs", 1)
    ng = case["ng"]
    return {"bytes": 2 * b * npts + 2 * b * ng * k, "flops": k * (2.0 * taps * npts + fft(ng))}


# ----------------------------------------------------- 64-bit restatement --
_SIGMA, _HW = 4, 16
_BETA = 2.0 * _SIGMA * _HW / ((2.0 * _SIGMA - 1.0) * math.pi)


def _taps(x, G):
    """Anchor cell, and the offset of x from it, on a periodic grid of G cells."""
    p = x * G
    a = torch.floor(p)
    return a.long(), p - a


def _deconv(M, G):
    k = torch.arange(-(M // 2), M // 2, device=DEV, dtype=torch.float64)
    return torch.exp(math.pi ** 2 * _BETA * (k / G) ** 2) / math.sqrt(math.pi * _BETA)


def _type1(x, y, M):
    """sum_j y[r, j] e^{2 pi i k x_j}, k = -M/2 .. M/2-1, for each row r of real values."""
    G = _SIGMA * M
    a, e = _taps(x, G)
    grid = torch.zeros((y.shape[0], G), device=DEV, dtype=torch.float64)
    for o in range(-_HW + 1, _HW + 1):
        grid.index_add_(1, (a + o) & (G - 1), y * torch.exp(-(o - e) ** 2 / _BETA))
    f = torch.fft.ifft(grid, norm="forward")
    f = torch.cat([f[:, G - M // 2:], f[:, : M // 2]], dim=1)
    return f * _deconv(M, G)


def _type2(x, f):
    """sum_k f[k] e^{-2 pi i k x_j} for complex f of M values."""
    M = f.numel()
    G = _SIGMA * M
    c = f * _deconv(M, G)
    u = torch.zeros(G, device=DEV, dtype=torch.complex128)
    u[G - M // 2:] = c[: M // 2]
    u[: M // 2] = c[M // 2:]
    u = torch.fft.fft(u)
    a, e = _taps(x, G)
    out = torch.zeros(x.shape, device=DEV, dtype=torch.complex128)
    for o in range(-_HW + 1, _HW + 1):
        out += u[(a + o) & (G - 1)] * torch.exp(-(o - e) ** 2 / _BETA)
    return out


_U32 = 0xFFFFFFFF


def _draws(n, nbs):
    """Bootstrap draws d[r, p] = xorshift(wang(SEED + r n + p)) mod n in 32-bit arithmetic."""
    s = (torch.arange(nbs * n, device=DEV, dtype=torch.int64) + SEED) & _U32
    s = (s ^ 61) ^ (s >> 16)
    s = (s * 9) & _U32
    s = s ^ (s >> 4)
    s = (s * 0x27D4EB2D) & _U32
    s = s ^ (s >> 15)
    s = (s ^ (s << 13)) & _U32
    s = s ^ (s >> 17)
    s = (s ^ (s << 5)) & _U32
    return (s % n).reshape(nbs, n)


def _compat_point(x, ng, dtype):
    """The reference formula's decisions per point, in the library's precision: anchor j and eps."""
    rf = 6 if dtype == "f32" else 12
    prod = x * ng  # one rounding, in x's type
    eps = prod - torch.trunc(prod - rf)
    j = torch.trunc((x.double() + 0.5) * (ng - 1)).long().clamp(0, ng - 1)
    return j, eps.double(), rf


def _compat_b(n, ng, dtype):
    if dtype == "f64":
        r = ng / n
        return 2.0 * r / (2.0 * r - 1.0) * (12.0 / math.pi)
    r = np.float32(ng) / np.float32(n)
    q = np.float32(2) * r / (np.float32(2) * r - np.float32(1))
    return float(np.float32(float(q) * (6.0 / math.pi)))


def _compat(j, eps, y, n, ng, rf, dtype):
    """Rows of the reference formula: eps and y are (rows, n), j is (n,)."""
    b = _compat_b(n, ng, dtype)
    grid = torch.zeros((y.shape[0], ng), device=DEV, dtype=torch.float64)
    for o in range(-rf + 1, rf):
        cell = j + o
        ok = (cell >= 0) & (cell < ng)
        w = y * torch.exp(-(eps - o) ** 2 / b) / math.sqrt(math.pi * b)
        grid.index_add_(1, cell[ok], w[:, ok])
    r = torch.arange(ng, device=DEV, dtype=torch.float64) / ng
    f = torch.fft.ifft(grid, norm="forward")
    return f * (math.sqrt(2.0 * math.pi) * torch.exp(r * r * b / 4.0))


def _ls_power(f, w, n, yy):
    h = w.abs()
    one = torch.ones_like(h)
    c2 = torch.where(h > 0, w.real / h, one)
    cw = torch.sqrt(((1 + c2) / 2).clamp(min=0))
    sw = torch.copysign(torch.sqrt(((1 - c2) / 2).clamp(min=0)), w.imag)
    yc = f.real * cw + f.imag * sw
    ys = f.imag * cw - f.real * sw
    cc, ss = (n + h) / 2, (n - h) / 2
    tiny = 1e-14 * n
    zero = torch.zeros_like(h)
    return (torch.where(cc > tiny, yc * yc / cc, zero) + torch.where(ss > tiny, ys * ys / ss, zero)) / yy


def exact(case, seed):
    s = _inputs(case, seed)
    kind, dt = case["kind"], case["dtype"]
    if kind in ("adjoint", "many"):
        y = s["y"].double().reshape(-1, case["n"])
        return torch.cat([_type1(s["x"].double(), row[None], case["M"]) for row in y])
    if kind == "forward":
        return _type2(s["x"].double(), s["fhat"][0].to(torch.complex128))
    if kind == "train":
        M = case["M"]
        k = torch.arange(-(M // 2), M // 2, device=DEV, dtype=torch.float64)
        f, dx, dy = [], [], []
        for x, y, g in zip(s["x"].double(), s["y"].double(), s["g"].to(torch.complex128)):
            f.append(_type1(x, y[None], M)[0])
            dy.append(_type2(x, g).real)
            dx.append(y * _type2(x, g * (-2j * math.pi) * k).real)
        return {"f": torch.stack(f), "dx": torch.stack(dx), "dy": torch.stack(dy)}
    if kind in ("survey", "bootstrap", "ls"):
        M, offs = case["M"], s["offs"]
        first, second = [], []
        for c in range(case["curves"]):
            x = s["t"][offs[c]:offs[c + 1]] * s["df"]
            y = s["y"][offs[c]:offs[c + 1]].double()
            if kind == "survey":
                first.append(_type1(x, y[None], M))
                continue
            n, nbs = x.numel(), case["nbs"]
            count = torch.zeros((nbs, n), device=DEV, dtype=torch.float64)
            count.scatter_add_(1, _draws(n, nbs), torch.ones((nbs, n), device=DEV, dtype=torch.float64))
            if kind == "bootstrap":
                first.append(_type1(x, count * y, M))
                second.append(_type1(2.0 * x, count, M))
                continue
            d = y - (count * y).sum(1, keepdim=True) / n
            yy = (count * d * d).sum(1, keepdim=True)
            f = _type1(x, count * d, M)[:, M // 2:]
            w = _type1(2.0 * x, count, M)[:, M // 2:]
            first.append(_ls_power(f, w, n, yy))
        return (torch.cat(first), torch.cat(second)) if second else torch.cat(first)
    n, ng = case["n"], case["ng"]
    x = torch.as_tensor(s["x"], device=DEV)
    y = torch.as_tensor(s["y"], device=DEV).double()
    j, eps, rf = _compat_point(x, ng, dt)
    if kind == "compat_boot":
        d = _draws(n, case["nbs"])
        return _compat(j, eps[d], y[d], n, ng, rf, dt)
    out = _compat(j, eps[None], y[None], n, ng, rf, dt)[0]
    return out.cpu().numpy() if kind == "host" else out
