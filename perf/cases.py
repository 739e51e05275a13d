"""The workloads that the framework's speed is measured on.

Each case is one call (or one served burst) through the public entry points
of the package, at the sizes its programs are used at: the datasets of the
benchmarks that the entry points come from, the benchmark's own workloads,
and generic sizes around them.

  * prices of many strikes on one grid (LocVolCalib's `main`): from a quote
    of a few strikes on a small grid to the precision workload, in the f32
    and the FP64 form;
  * many unrelated problems at once (`main_batch`) and a burst of requests
    through the continuous-batching server;
  * the ocean model's vertical solves (`tridagNestedSeq`, `tridagNested`);
  * Monte-Carlo prices of the three contracts (OptionPricing's `main`);
  * the swaption calibration (InterestCalib's `main`).
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "futhark-benchmarks_amd"))

import locvolcalib as lvc  # noqa: E402
from locvolcalib import interestcalib, optionpricing  # noqa: E402

DEVICE = "cuda:0"
PROBLEM = ("numX", "numY", "numT", "s0", "strike", "t", "alpha", "nu", "beta")
LARGEST = 256 * 256 * 256 * 127  # grid point steps of the largest strike set


# ---- the cases ---------------------------------------------------------------

def listed():
    return [
        # a trader's quote: a handful of strikes on a coarse grid; the call's
        # latency is what counts
        {"name": "strikes_quote", "kind": "strikes", "form": "refine",
         "outer": 4, "nx": 32, "ny": 32, "nt": 16},
        # the benchmark's CPU-sized workload: a narrow grid, many time steps
        {"name": "strikes_narrow", "kind": "strikes", "form": "refine",
         "outer": 16, "nx": 32, "ny": 256, "nt": 256},
        # the headline workload: a strip of 128 strikes
        {"name": "strikes_128", "kind": "strikes", "form": "refine",
         "outer": 128, "nx": 256, "ny": 256, "nt": 64},
        # the same strip in double precision (a risk run's reference prices)
        {"name": "strikes_128_fp64", "kind": "strikes", "form": "fp64",
         "outer": 128, "nx": 256, "ny": 256, "nt": 64},
        # the precision workload, the largest: 256 strikes, twice the steps
        {"name": "strikes_256", "kind": "strikes", "form": "refine",
         "outer": 256, "nx": 256, "ny": 256, "nt": 128},
        # a calibration's objective: unrelated problems, uneven sizes
        {"name": "batch_512", "kind": "batch", "form": "refine",
         "n": 512, "lo": 32, "hi": 256, "nt_lo": 32, "nt_hi": 256},
        # a burst of requests at a pricing service, ragged sizes
        {"name": "served_burst", "kind": "served", "form": "refine",
         "n": 96, "lo": 32, "hi": 128, "nt_lo": 16, "nt_hi": 64},
        # the ocean model's columns: one implicit vertical step, both forms
        {"name": "columns_seq", "kind": "columns", "form": "seq", "n": 57600, "m": 115},
        {"name": "columns_scan", "kind": "columns", "form": "scan", "n": 57600, "m": 115},
        # Monte-Carlo prices: five dates of a basket, 367 dates of a barrier
        {"name": "paths_basket", "kind": "paths", "contract": 2, "paths": 1048576, "models": 1},
        {"name": "paths_barrier", "kind": "paths", "contract": 3, "paths": 131072, "models": 1},
        # the swaption calibration at the small dataset's size
        {"name": "rates", "kind": "rates", "pop": 256, "iters": 128, "swaptions": 196},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["strikes", "strikes", "strikes", "batch", "served", "columns",
                       "paths", "paths", "rates"])
    if kind == "strikes":
        nx, ny, nt = _log(rng, 24, 512), _log(rng, 24, 512), _log(rng, 12, 256)
        most = max(1, min(256, LARGEST // (nx * ny * (nt - 1))))
        return {"kind": kind, "form": rng.choice(["refine", "refine", "fp64", "fp32"]),
                "outer": _log(rng, 1, most), "nx": nx, "ny": ny, "nt": nt}
    if kind in ("batch", "served"):
        n = _log(rng, 8, 512 if kind == "batch" else 128)
        hi = _log(rng, 40, 256 if kind == "batch" else 160)
        nt_hi = _log(rng, 24, 256 if kind == "batch" else 80)
        return {"kind": kind, "form": rng.choice(["refine", "fp64"]), "n": n,
                "lo": rng.randint(16, 36), "hi": hi, "nt_lo": rng.randint(12, 22),
                "nt_hi": nt_hi}
    if kind == "columns":
        return {"kind": kind, "form": rng.choice(["seq", "scan"]), "n": _log(rng, 500, 57600),
                "m": rng.randint(20, 128)}
    if kind == "paths":
        contract = rng.choice([1, 2, 3])
        lo, hi = {1: (1 << 16, 1 << 23), 2: (1 << 14, 1 << 20), 3: (1 << 12, 1 << 17)}[contract]
        return {"kind": kind, "contract": contract, "paths": _log(rng, lo, hi), "models": 1}
    return {"kind": "rates", "pop": _log(rng, 24, 256), "iters": _log(rng, 12, 128),
            "swaptions": _log(rng, 14, 196)}


def work(case):
    kind = case["kind"]
    if kind == "strikes":
        points = case["nx"] * case["ny"] * (case["nt"] - 1) * case["outer"]
        real = 8 if case["form"] == "fp64" else 4
        # a point step: two tridiagonal solves and the explicit operator
        return {"bytes": case["outer"] * real, "flops": 26.0 * points}
    if kind in ("batch", "served"):
        p = _problems(case, 1)
        points = float((p["numX"].astype(float) * p["numY"] * (p["numT"] - 1)).sum())
        return {"bytes": case["n"] * 68, "flops": 26.0 * points}
    if kind == "columns":
        size = case["n"] * case["m"]
        return {"bytes": 20 * size, "flops": (8.0 if case["form"] == "seq" else 30.0) * size}
    if kind == "paths":
        dates, und = _SHAPES[case["contract"]]
        dims = dates * und
        # a path's dimension: the inverse Gaussian, the bridge step and the
        # asset's step
        return {"bytes": dims * 120 + case["models"] * 4,
                "flops": 60.0 * case["paths"] * dims * case["models"]}
    periods = 2.0 * float(_swaptions(case, 1)[:, 2].sum())
    # per period of a schedule: three root searches and the quadrature
    return {"bytes": case["swaptions"] * 28,
            "flops": 250.0 * case["pop"] * (case["iters"] + 1) * periods}


# ---- inputs ------------------------------------------------------------------

_contexts = {}


def _context(make, *key, **options):
    """A program's one context of a library (with the options it uses)."""
    at = (make.__name__,) + key
    if at not in _contexts:
        _contexts[at] = make(device=0, **options)
    return _contexts[at]


_PRECISION = {"fp32": lvc.PRECISION_FP32, "refine": lvc.PRECISION_FP32_REFINE,
              "fp64": lvc.PRECISION_FP64}


def _market(rng, n=None):
    """Model parameters: spot, maturity, volatility, vol of vol, elasticity."""
    return dict(s0=rng.uniform(0.02, 0.05, n), t=rng.uniform(1.0, 10.0, n),
                alpha=rng.uniform(0.1, 0.3, n), nu=rng.uniform(0.4, 0.8, n),
                beta=rng.uniform(0.3, 0.7, n))


def _sizes(rng, case):
    """Sizes between lo and hi: powers of two where both are, else any."""
    lo, hi, n = case["lo"], case["hi"], case["n"]
    if (lo & (lo - 1)) == 0 and (hi & (hi - 1)) == 0:
        return 1 << rng.integers(lo.bit_length() - 1, hi.bit_length(), n)
    return rng.integers(lo, hi + 1, n)


def _problems(case, seed):
    rng = np.random.default_rng([seed, 11])
    # the sizes are the case's, the market the seed's
    sizes = np.random.default_rng(5)
    p = dict(numX=_sizes(sizes, case).astype(np.int32), numY=_sizes(sizes, case).astype(np.int32),
             numT=sizes.integers(case["nt_lo"], case["nt_hi"] + 1, case["n"]).astype(np.int32),
             strike=rng.uniform(0.0, 0.05, case["n"]))
    p.update(_market(rng, case["n"]))
    return p


def _strikes_args(case, seed):
    m = _market(np.random.default_rng([seed, 7]))
    return tuple(float(m[k]) for k in ("s0", "t", "alpha", "nu", "beta"))


def _columns(case, seed):
    """Implicit vertical mixing: 1 + dt * diffusivity / dz^2 couplings, the
    top and bottom cells closed."""
    g = torch.Generator(device=DEVICE).manual_seed(int(seed) % (1 << 31))
    n, m = case["n"], case["m"]
    k = 4.0 * torch.rand((n, m + 1), generator=g, device=DEVICE)
    k[:, 0] = 0
    k[:, m] = 0
    a, c = -k[:, :m], -k[:, 1:]
    b = 1.0 - a - c
    y = 20.0 * torch.rand((n, m), generator=g, device=DEVICE) - 2.0
    return [v.contiguous() for v in (a, b, c, y)]


_SHAPES = {1: (1, 1), 2: (5, 3), 3: (367, 3)}
_BITS = 30


def _direction_vectors(dims, rng):
    """Direction vectors of digital sequences: the first dimension the radical
    inverse, the others with random odd direction numbers."""
    v = np.empty((dims, _BITS), np.int64)
    for b in range(_BITS):
        v[:, b] = (2 * rng.integers(0, 1 << b, dims) + 1) << (_BITS - 1 - b)
    v[0] = 1 << np.arange(_BITS - 1, -1, -1)
    return v.astype(np.int32)


def _bridge(times):
    """Brownian bridge over `times` (increasing, after 0): the last date, then
    each middle date between its built neighbours, left part first."""
    d = len(times)
    inds, data = np.zeros((3, d), np.int32), np.zeros((3, d), np.float32)
    t = np.concatenate([[0.0], times])
    inds[0, 0], data[0, 0] = d, math.sqrt(t[d])
    step, todo = 1, [(0, d)]
    while todo:
        lo, hi = todo.pop()
        if hi - lo < 2:
            continue
        mid = (lo + hi) // 2
        whole = t[hi] - t[lo]
        inds[:, step] = mid, lo, hi
        data[:, step] = (math.sqrt((t[mid] - t[lo]) * (t[hi] - t[mid]) / whole),
                         (t[hi] - t[mid]) / whole if lo else 0.0, (t[mid] - t[lo]) / whole)
        step += 1
        todo += [(mid, hi), (lo, mid)]
    return inds, data


def _paths(case, seed):
    """The nine arrays of OptionPricing's main: an index basket's market."""
    rng = np.random.default_rng([seed, 3])
    dates, und = _SHAPES[case["contract"]]
    models = case["models"]
    dt = 1.0 / 366 if case["contract"] == 3 else 1.0
    times = dt * np.arange(1, dates + 1)
    inds, data = _bridge(times)
    corr = np.array([[1.0, 0.6, 0.8], [0.6, 1.0, 0.6], [0.8, 0.6, 1.0]])[:und, :und]
    chol = np.linalg.cholesky(corr)
    vols = rng.uniform(0.14, 0.22, (models, 1, und)).repeat(dates, 1)
    drifts = (rng.uniform(0.0, 0.03, (models, dates, und)) - 0.5 * vols ** 2) * dt
    starts = np.array([3758.05, 11840.0, 1200.0])[:und] * rng.uniform(0.95, 1.05, (models, und))
    pays = {1: 1, 2: 5, 3: 2}[case["contract"]]
    discounts = np.exp(-rng.uniform(0.015, 0.03, (models, 1)) *
                       (np.arange(1, pays + 1) if pays == 5 else np.ones(pays)))
    f = lambda v: np.ascontiguousarray(v, np.float32)  # noqa: E731
    return [_direction_vectors(dates * und, rng), f(np.repeat(chol[None], models, 0)), f(vols),
            f(drifts), f(starts), f(np.full((models, 1), 1.0)), f(discounts), inds, data]


_YEARS = (1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 15, 20, 25, 30)


def _swaptions(case, seed):
    """A swaption matrix: maturity and term in years, semi-annual payments,
    volatilities that fall with both."""
    rng = np.random.default_rng([seed, 19])
    rows = [(float(m), 6.0, float(n)) for n in _YEARS for m in _YEARS]
    keep = np.linspace(0, len(rows) - 1, case["swaptions"]).astype(int)
    s = np.array([rows[i] for i in keep])
    vol = 0.19 + 0.8 * np.exp(-0.35 * (s[:, 0] - 1)) * np.exp(-0.18 * (s[:, 2] - 1))
    vol *= rng.uniform(0.96, 1.04, len(s))
    return np.concatenate([s, vol[:, None]], 1).astype(np.float32)


def _rates(case, seed):
    x, w = np.polynomial.hermite.hermgauss(11)
    order = np.argsort(np.abs(x), kind="stable")
    return (_swaptions(case, seed), x[order].astype(np.float32),
            (w * np.exp(x * x))[order].astype(np.float32),
            (1 << np.arange(_BITS - 1, -1, -1)).astype(np.int32))


# ---- states ------------------------------------------------------------------

class _State:
    """What a user's program holds between calls."""

    def __init__(self, case, **held):
        self.case = case
        self.__dict__.update(held)
        self.release = []

    def __del__(self):
        for f in reversed(self.release):
            try:
                f()
            except Exception:  # the context may be gone at the process's end
                pass


class _OnDevice:
    """A library array's device memory as torch sees it."""

    def __init__(self, pointer, shape):
        self.__cuda_array_interface__ = {"data": (int(pointer), False), "shape": tuple(shape),
                                         "typestr": "<f4", "version": 2}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "strikes":
        ctx = _context(lvc.LocVolCalib, case["form"] == "fp32",
                       precision=lvc.PRECISION_FP32 if case["form"] == "fp32" else None)
        return _State(case, ctx=ctx, args=_strikes_args(case, seed))
    if kind == "batch":
        return _State(case, ctx=_context(lvc.LocVolCalib, False), problems=_problems(case, seed))
    if kind == "served":
        ctx = _context(lvc.LocVolCalib, False)
        p = _problems(case, seed)
        requests = [tuple(p[k][i].item() for k in PROBLEM) for i in range(case["n"])]
        server = lvc.Server(ctx, max_slots=64, mem_budget=1 << 28,
                            precision=_PRECISION[case["form"]])
        s = _State(case, server=server, requests=requests)
        s.release.append(server.free)
        return s
    if kind == "columns":
        ctx = _context(lvc.LocVolCalib, False)
        s = _State(case, ctx=ctx, handles=[], result=None)
        for v in _columns(case, seed):
            h = ctx.upload_f32_2d(v.cpu().numpy())
            s.handles.append(h)
            s.release.append(lambda h=h: ctx.free_f32_2d(h))
        return s
    if kind == "paths":
        ctx = _context(optionpricing.OptionPricing)
        handles = ctx.upload_arguments(_paths(case, seed))
        s = _State(case, ctx=ctx, handles=handles)
        s.release.append(lambda: ctx.free_arguments(handles))
        return s
    ctx = _context(interestcalib.InterestCalib)
    handles = ctx.upload_inputs(*_rates(case, seed))
    s = _State(case, ctx=ctx, handles=handles)
    s.release.append(lambda: ctx.free_inputs(handles))
    return s


def run(state):
    case = state.case
    kind = case["kind"]
    if kind == "strikes":
        entry = state.ctx.main_f64 if case["form"] == "fp64" else state.ctx.main
        return entry(case["outer"], case["nx"], case["ny"], case["nt"], *state.args)
    if kind == "batch":
        return state.ctx.main_batch(**state.problems, precision=_PRECISION[case["form"]])
    if kind == "served":
        server = state.server
        ids = [server.submit(*r) for r in state.requests]
        server.drain()
        return np.array([server.poll(i) for i in ids])
    if kind == "columns":
        # the result stays on the device, as the next stage of a model step
        # takes it; the last pass's one is given back first
        ctx = state.ctx
        if state.result is not None:
            ctx.free_f32_2d(state.result)
        else:
            state.release.append(lambda: ctx.free_f32_2d(state.result))
        state.result = ctx.tridag_nested_raw(*state.handles, seq=case["form"] == "seq")
        pointer = lvc.lib().futhark_values_raw_f32_2d(ctx.handle, state.result)
        return torch.as_tensor(_OnDevice(pointer, (case["n"], case["m"])), device=DEVICE)
    if kind == "paths":
        h = state.ctx.main_raw(case["contract"], case["paths"], state.handles)
        try:
            return state.ctx.values_f32(h)
        finally:
            state.ctx.free_f32(h)
    scalars, summary = state.ctx.main_raw(case["pop"], case["iters"], state.handles)
    state.ctx.free_summary(summary)
    return scalars


# ---- the same in 64 bits -----------------------------------------------------

def _solve(a, b, c, d):
    """Tridiagonal systems along the first dimension (b, d change)."""
    n = d.shape[0]
    for i in range(1, n):
        w = a[i] / b[i - 1]
        b[i] -= w * c[i - 1]
        d[i] -= w * d[i - 1]
    d[n - 1] /= b[n - 1]
    for i in range(n - 2, -1, -1):
        d[i] = (d[i] - c[i] * d[i + 1]) / b[i]
    return d


def _prices(problems, strikes, grid32):
    """The finite-difference prices of strikes[p, k] on problem p's grid: per
    time step the explicit operator, an implicit step in x, one in y.  grid32:
    the grid's index, spacing and first point from f32 scalars, as the f32
    entry defines them."""
    P, K = strikes.shape
    f8 = dict(dtype=torch.float64, device=DEVICE)
    X, Y = int(problems["numX"].max()), int(problems["numY"].max())
    col = lambda v: torch.as_tensor(np.asarray(v, np.float64), **f8)  # noqa: E731
    real = np.float32 if grid32 else np.float64
    s0, t, al = (problems[k].astype(real) for k in ("s0", "t", "alpha"))
    dx = real(20) * al * s0 * np.sqrt(t) / problems["numX"].astype(real)
    xi = np.trunc(s0 / dx).astype(np.int64)
    yi = problems["numY"] // 2
    nu = problems["nu"].astype(np.float64)
    dy = 10.0 * nu * np.sqrt(problems["t"].astype(np.float64)) / problems["numY"]
    x = (col(dx) * (torch.arange(X, **f8)[:, None] - col(xi)) + col(problems["s0"]))
    y = (col(dy) * (torch.arange(Y, **f8)[:, None] - col(yi)) +
         col(np.log(problems["alpha"].astype(np.float64))))
    inx = (torch.arange(X, device=DEVICE)[:, None] > 0) & (
        torch.arange(X, device=DEVICE)[:, None] < torch.as_tensor(problems["numX"] - 1, device=DEVICE))
    iny = (torch.arange(Y, device=DEVICE)[:, None] > 0) & (
        torch.arange(Y, device=DEVICE)[:, None] < torch.as_tensor(problems["numY"] - 1, device=DEVICE))
    zero = torch.zeros((), **f8)
    # a quarter of the variance over the squared spacing, without the x
    # operator's factor exp(2 y - nu^2 t)
    vx = torch.where(inx, torch.exp(2 * col(problems["beta"]) * torch.log(x.clamp(min=1e-300))) /
                     (4 * col(dx) ** 2), zero)
    vy = torch.where(iny, (col(nu) ** 2 / (4 * col(dy) ** 2)).expand(Y, P), zero)
    r = torch.clamp(x[:, None, :, None] - torch.as_tensor(strikes, **f8), min=0.0)
    r = r.expand(X, Y, P, K).contiguous()

    def second(v, dim):
        """v's second difference along dim, 0 at both ends."""
        out = torch.zeros_like(v)
        n = v.shape[dim]
        mid, lo, hi = (v.narrow(dim, k, n - 2) for k in (1, 0, 2))
        out.narrow(dim, 1, n - 2).copy_(lo - 2 * mid + hi)
        return out

    steps = problems["numT"].astype(np.int64) - 1
    tt = problems["t"].astype(np.float64)
    s = col(steps / tt)
    ay = vy[:, :, None, None].permute(0, 2, 1, 3)  # [Y, 1, P, 1]
    for step in range(int(steps.max())):
        k = steps - 1 - step  # the time index, from the last one down
        tau = col(np.exp(-nu * nu * tt * np.maximum(k, 0) / steps))
        ax = vx[:, None, :, None] * (torch.exp(2 * y) * tau)[None, :, :, None]  # [X, Y, P, 1]
        v = vy[None, :, :, None] * second(r, 1)
        u = s[:, None] * r + ax * second(r, 0) + 2 * v
        u = _solve(-ax, s[:, None] + 2 * ax, -ax, u)
        u = (s[:, None] * u - v).permute(1, 0, 2, 3).contiguous()
        u = _solve(-ay, (s[:, None] + 2 * ay).clone(), -ay, u)
        live = torch.as_tensor(k >= 0, device=DEVICE)[:, None]
        r = torch.where(live, u.permute(1, 0, 2, 3), r)
    at = torch.arange(P, device=DEVICE)
    return r[torch.as_tensor(xi, device=DEVICE), torch.as_tensor(yi, device=DEVICE), at].cpu().numpy()


def _exact_paths(case, seed):
    dv, cs, vols, drifts, sts, detvals, discts, inds, data = _paths(case, seed)
    dates, und = _SHAPES[case["contract"]]
    n = case["paths"]
    f8 = dict(dtype=torch.float64, device=DEVICE)
    index = torch.arange(1, n + 1, dtype=torch.int64, device=DEVICE)
    gray = index ^ (index >> 1)
    of = lambda v: torch.as_tensor(np.asarray(v, np.float64), **f8)  # noqa: E731

    def normals(date):
        z = []
        for u in range(und):
            q = torch.zeros_like(gray)
            for b in range(_BITS):
                q ^= torch.where((gray >> b) & 1 == 1, int(dv[date * und + u, b]), 0)
            z.append(torch.special.ndtri(q.double() / float(1 << _BITS)))
        return torch.stack(z)

    rows = torch.zeros((dates, und, n), **f8)
    sd, lw, rw = (of(v) for v in data)
    rows[inds[0, 0] - 1] = sd[0] * normals(0)
    for i in range(1, dates):
        v = rw[i] * rows[inds[2, i] - 1] + sd[i] * normals(i)
        if inds[1, i]:
            v = v + lw[i] * rows[inds[1, i] - 1]
        rows[inds[0, i] - 1] = v
    out = []
    for m in range(case["models"]):
        level = torch.zeros((und, n), **f8)
        price = []
        barrier = torch.zeros(n, dtype=torch.bool, device=DEVICE)
        for d in range(dates):
            z = rows[d] - rows[d - 1] if d else rows[d]
            z = torch.tril(of(cs[m])) @ z
            level = level + of(drifts[m, d])[:, None] + z * of(vols[m, d])[:, None]
            last = of(sts[m])[:, None] * torch.exp(level)
            if case["contract"] == 2:
                price.append(last)
            if case["contract"] == 3:
                barrier |= (last <= of([2630.635, 8288.0, 840.0])[:, None]).any(0)
        disc = [float(v) for v in discts[m]]
        rel = lambda v: (v / of([3758.05, 11840.0, 1200.0])[:, None]).amin(0)  # noqa: E731
        if case["contract"] == 1:
            pay = torch.clamp((last[0] - 4000.0) * float(detvals[m, 0]), min=0.0) * disc[0]
        elif case["contract"] == 2:
            x = rel(price[4])
            pay = torch.where(x >= 1, 1750.0, torch.where(x > 0.75, 1000.0, 1000.0 * x)) * disc[4]
            for d, amount in ((3, 1600.0), (2, 1450.0), (1, 1300.0), (0, 1150.0)):
                pay = torch.where(rel(price[d]) >= 1, amount * disc[d], pay)
        else:
            x = rel(last)
            pay = 100.0 * disc[0] + torch.where(barrier & (x < 1), 1000.0 * x, 1000.0) * disc[1]
        out.append(float(pay.mean()))
    return np.array(out)


def exact(case, seed):
    kind = case["kind"]
    if kind == "strikes":
        f32 = case["form"] != "fp64"
        real = np.float32 if f32 else np.float64
        m = dict(zip(("s0", "t", "alpha", "nu", "beta"), _strikes_args(case, seed)))
        p = {k: np.array([v]).astype(real) for k, v in m.items()}
        p.update(numX=np.array([case["nx"]]), numY=np.array([case["ny"]]),
                 numT=np.array([case["nt"]]))
        strikes = (real(0.001) * np.arange(case["outer"]).astype(real))[None]
        return _prices(p, strikes.astype(np.float64), f32)[0]
    if kind in ("batch", "served"):
        p = _problems(case, seed)
        return _prices(p, p["strike"][:, None], False)[:, 0]
    if kind == "columns":
        a, b, c, d = (v.double().T.contiguous() for v in _columns(case, seed))
        return _solve(a, b, c, d).T.contiguous()
    if kind == "paths":
        return _exact_paths(case, seed)
    # the calibration accepts or rejects by its own f32 likelihoods: its
    # result has no 64-bit value
    return None
