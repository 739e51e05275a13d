"""Which problems of an FP64 batch go by the modes and which by the sweeps: by
the kernels that the profiling report counts, the prices on both sides of the
line against the FP64 oracle.  Tolerance: the FP64 form's bar of 1e-10.
"""
import json

import numpy as np
import pytest

from oracle import oracle
import locvolcalib as lvc

pytestmark = pytest.mark.gpu

KEYS = ("numX", "numY", "numT", "s0", "strike", "t", "alpha", "nu", "beta")
MARKET = (0.03, 5.0, 0.2, 0.6, 0.5)


def route(ctx, call):
    """The call's result and the kernels it launched."""
    before = json.loads(ctx.report())
    out = call()
    after = json.loads(ctx.report())
    count = {k: v["count"] - before.get(k, {"count": 0})["count"] for k, v in after.items()
             if isinstance(v, dict)}
    return out, {k for k, c in count.items() if c}


def problem(nx, ny, nt, strike):
    s0, t, alpha, nu, beta = MARKET
    return dict(numX=[nx], numY=[ny], numT=[nt], s0=[s0], strike=[strike], t=[t], alpha=[alpha],
                nu=[nu], beta=[beta])


# (numX, numY, numT), by the modes: narrow grids always; wide ones where
# numY (numT - 1) reaches 2.25 (numX - 48) and numX^2 / 300
@pytest.mark.parametrize("shape,modes", [
    ((64, 3, 7), True), ((65, 6, 7), False), ((65, 7, 7), True), ((256, 18, 27), True),
    ((256, 18, 26), False), ((512, 58, 19), True), ((512, 58, 18), False),
    ((1024, 16, 8), False), ((1024, 583, 7), True), ((1024, 582, 7), False)])
def test_batch_by_size(shape, modes):
    print(f"case: route of {shape}", flush=True)
    p = problem(*shape, 0.02)
    with lvc.LocVolCalib(profiling=True) as ctx:
        got, kernels = route(ctx, lambda: ctx.main_batch(**p, precision=lvc.PRECISION_FP64))
        assert ("lvc_modes" in kernels) == modes and ("lvc_xsweep" in kernels) != modes
        # main's strikes share one grid's modes at every size
        by_main, kernels = route(ctx, lambda: ctx.main_f64(21, *shape, *MARKET))
        assert "lvc_modes" in kernels and "lvc_xsweep" not in kernels
    ref = oracle.batch(*[p[k] for k in KEYS], dtype=np.float64, thomas=True, nthreads=8)
    assert abs(got[0] - ref[0]) < 1e-10 * ref[0]
    assert abs(by_main[20] - ref[0]) < 1e-10 * ref[0]


@pytest.mark.parametrize("precision", [lvc.PRECISION_FP32_REFINE, lvc.PRECISION_FP64])
def test_main_autotunes_its_class(tmp_path, precision):
    """With "lvc.autotune" a call of main leaves its class's segment lengths in
    the cache file, for the sweeps of the batch, the server and the
    allocation-free entry, whichever way main itself goes."""
    print(f"case: main autotunes, precision {precision}", flush=True)
    cache = tmp_path / "lvc.tuning"
    with lvc.LocVolCalib(cache_file=str(cache), precision=precision,
                         tuning={"lvc.autotune": 1}) as ctx:
        got = ctx.main(3, 40, 36, 20, *MARKET)
        if precision == lvc.PRECISION_FP64:
            ctx.main_f64(3, 48, 36, 20, *MARKET)
    lines = [tuple(int(v) for v in line.split()[:3]) for line in cache.read_text().splitlines()]
    want = [(precision, 40, 36)] + [(precision, 48, 36)] * (precision == lvc.PRECISION_FP64)
    assert lines == want
    with lvc.LocVolCalib(precision=precision) as ctx:
        assert np.array_equal(got, ctx.main(3, 40, 36, 20, *MARKET))


def test_noalloc_is_not_profiled():
    """Profiling does not cover the allocation-free entry (an event made for it
    would be an allocation, and its caller may be capturing)."""
    print("case: main_noalloc with profiling", flush=True)
    with lvc.LocVolCalib(profiling=True) as ctx:
        got, kernels = route(ctx, lambda: ctx.main_noalloc(5, 40, 36, 20, *MARKET))
        assert not kernels
        want, kernels = route(ctx, lambda: ctx.main(5, 40, 36, 20, *MARKET))
        assert kernels == {"lvc_modes", "lvc_evolve", "lvc_price"}
        assert np.array_equal(got, want)


@pytest.mark.parametrize("shape,strike,precision", [
    ((40, 36, 5), 0.02, lvc.PRECISION_FP64), ((40, 36, 20), 0.02, lvc.PRECISION_FP64),
    ((40, 36, 20), 0.0998, lvc.PRECISION_FP64), ((40, 36, 20), 0.02, lvc.PRECISION_FP32)])
def test_the_index_read(shape, strike, precision):
    """The debugging report's index is problem 0's by whichever way it goes,
    the others another."""
    print(f"case: price index of {shape}, strike {strike}, precision {precision}", flush=True)
    p = {k: v * 3 for k, v in problem(*shape, strike).items()}
    p["numX"], p["numY"], p["strike"] = [shape[0], 64, 30], [shape[1], 20, 24], [strike, .01, .03]
    t, alpha = MARKET[1:3]
    with lvc.LocVolCalib(debugging=True) as ctx:
        ctx.main_batch(**p, precision=precision)
        assert ctx.price_index() == (18, int(40 / (20 * alpha * np.sqrt(t))))
        ctx.main_f64(3, 64, 20, shape[2], *MARKET)
        assert ctx.price_index() == (10, int(64 / (20 * alpha * np.sqrt(t))))


@pytest.mark.parametrize("market", [(0.0263, 2.2404, 0.2967, 0.4011, 0.4463),
                                    (0.0285, 1.9693, 0.247, 0.5365, 0.3156),
                                    (0.0219, 8.4294, 0.1329, 0.5501, 0.4267)])
def test_the_last_cell(market):
    """Strikes just below the grid's last node, whose price is small because the
    node is near and not because the strike is far: the f32 entry takes the modes."""
    print(f"case: strikes to the grid's end, {market}", flush=True)
    with lvc.LocVolCalib(profiling=True) as ctx:
        got, kernels = route(ctx, lambda: ctx.main(256, 256, 64, 12, *market))
    assert kernels == {"lvc_modes", "lvc_evolve", "lvc_price"}
    s0, t, alpha, nu, beta = (float(np.float32(v)) for v in market)
    dx = float(np.float32(20) * np.float32(alpha) * np.float32(s0) * np.sqrt(np.float32(t)) /
               np.float32(256))
    last = (255 - int(s0 / dx)) * dx + s0
    near = [int(1000 * last) - 1, int(1000 * last), int(1000 * last) + 1]
    strikes = (np.float32(0.001) * np.float32(near)).astype(np.float64)
    p = dict(zip(KEYS, [[v] * 3 for v in (256, 64, 12, s0)] + [strikes] +
                 [[v] * 3 for v in (t, alpha, nu, beta)]))
    ref = oracle.batch(*[p[k] for k in KEYS], dtype=np.float64, thomas=True, nthreads=8,
                       grid32=True)
    assert ref[1] > 0 and ref[2] == 0
    assert np.all(np.abs(got[near] - ref) <= 1e-6 * ref)
