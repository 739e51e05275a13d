"""The sweeps behind `main`, `main_f64`, the allocation-free entry and the FP64
batch, on a market that the price by separation of x does not take (an
elasticity below 0), and the modes at their sizes through `main_f64`, whose near
strikes always take them.  Which way a call goes is read from the profiling
report.

Tolerances, those of test_gpu_parity.py: FP64 1e-10 relative, FP32 with
refinement 1e-6, FP32 2e-5 (1e-4 on short runs); equal bits where two launches
run the same arithmetic.
"""
import numpy as np
import pytest

from oracle import oracle
import locvolcalib as lvc
from test_gpu_modes import SHAPES_T, SHAPES_WIDE, SHAPES_X, SHAPES_Y
from test_gpu_modes_route import KEYS, route
from test_gpu_tuning import BUILTIN
from test_zz_no_alloc import CALLS

pytestmark = pytest.mark.gpu

MARKET = (0.03, 5.0, 0.2, 0.6, -0.03)  # s0, t, alpha, nu, beta
SWEEPS = {"lvc_setup", "lvc_xsweep", "lvc_ysweep", "lvc_gather"}


def strikes_batch(nx, ny, nt, strikes, market=MARKET, dtype=np.float64):
    n = len(strikes)
    s0, t, alpha, nu, beta = (float(dtype(v)) for v in market)
    full = [np.full(n, v) for v in (nx, ny, nt, s0)] + [np.asarray(strikes, np.float64)]
    return dict(zip(KEYS, full + [np.full(n, v) for v in (t, alpha, nu, beta)]))


def oracle_batch(p, **kw):
    return oracle.batch(*[p[k] for k in KEYS], dtype=np.float64, thomas=True, nthreads=8, **kw)


def test_shared_factors():
    """x tiles shared by options that differ in the strike: main, main_f64 and
    FP64 batches with runs of such problems."""
    print("case: shared factors by the sweeps", flush=True)
    p = strikes_batch(64, 96, 7, np.linspace(0.0, 0.05, 20))
    p["nu"][5], p["numX"][11], p["numT"][15:] = 0.55, 32, 5
    out = {}
    for share in (1, 4, 16):
        with lvc.LocVolCalib(tuning={"lvc.xshare": share}, profiling=True) as ctx:
            runs = [lambda: ctx.main(24, 64, 64, 9, *MARKET),
                    lambda: ctx.main_f64(24, 64, 64, 9, *MARKET),
                    lambda: ctx.main_f64(24, 256, 256, 9, *MARKET),
                    lambda: ctx.main_batch(**p, precision=lvc.PRECISION_FP64)]
            out[share] = []
            for run in runs:
                got, kernels = route(ctx, run)
                assert kernels == SWEEPS
                out[share].append(got)
    for share in (4, 16):
        assert all(np.array_equal(a, b) for a, b in zip(out[1], out[share]))
    refs = [oracle_batch(strikes_batch(64, 64, 9, 0.001 * np.arange(24))),
            oracle_batch(strikes_batch(256, 256, 9, 0.001 * np.arange(24))), oracle_batch(p)]
    for got, ref in zip(out[16][1:], refs):
        assert np.max(np.abs(got - ref) / np.abs(ref)) < 1e-10


@pytest.mark.parametrize("precision,nx,ny,sx,sy",
                         [b for b in BUILTIN if b[0] == lvc.PRECISION_FP64])
def test_builtin_pair_fp64(precision, nx, ny, sx, sy):
    print(f"case: built-in pair, FP64 {nx}x{ny} by the sweeps", flush=True)
    p = strikes_batch(nx, ny, 12, np.linspace(0.0, 0.04, 6))
    p["alpha"] = np.linspace(0.15, 0.25, 6)
    with lvc.LocVolCalib(profiling=True) as ctx:
        got, kernels = route(ctx, lambda: ctx.main_batch(**p, precision=precision))
    assert kernels == SWEEPS
    with lvc.LocVolCalib(tuning={"lvc.seg_x": sx, "lvc.seg_y": sy}) as ctx:
        forced = ctx.main_batch(**p, precision=precision)
    with lvc.LocVolCalib(tuning={"lvc.seg_x": 16, "lvc.seg_y": 16}) as ctx:
        other = ctx.main_batch(**p, precision=precision)
    assert np.array_equal(got, forced) and not np.array_equal(got, other)
    ref = oracle_batch(p)
    assert np.max(np.abs(got - ref) / np.abs(ref)) < 1e-10


def test_plain_fp32():
    """FP32 without refinement: a batch of the former strikes of main, and main."""
    print("case: plain FP32 by the sweeps, 256x256x64", flush=True)
    p = strikes_batch(256, 256, 64, [0.0, 0.06, 0.127], market=(0.03, 5.0, 0.2, 0.6, 0.5))
    with lvc.LocVolCalib(precision=lvc.PRECISION_FP32, profiling=True) as ctx:
        got, kernels = route(ctx, lambda: ctx.main_batch(**p, precision=lvc.PRECISION_FP32))
        assert kernels == SWEEPS
        by_main, kernels = route(ctx, lambda: ctx.main(128, 256, 256, 64, *MARKET))
        assert kernels == SWEEPS
    ref = oracle_batch(p)
    assert np.max(np.abs(got - ref) / np.abs(ref)) < 2e-5
    near = [0, 30, 60]
    q = strikes_batch(256, 256, 64, (np.float32(0.001) * np.float32(near)).astype(np.float64),
                      dtype=np.float32)
    ref = oracle_batch(q, grid32=True)
    assert np.max(np.abs(by_main[near] - ref) / np.abs(ref)) < 2e-5


@pytest.mark.parametrize("precision", sorted(CALLS))
def test_noalloc_layout(precision):
    """The scratch's layout at real sizes, a smaller call behind a larger one."""
    with lvc.LocVolCalib(precision=precision) as ctx, \
            lvc.LocVolCalib(precision=precision, profiling=True) as main:
        for outer, nx, ny, nt in CALLS[precision]:
            print(f"case: main_noalloc({outer}, {nx}, {ny}, {nt}), precision {precision}",
                  flush=True)
            got = ctx.main_noalloc(outer, nx, ny, nt, *MARKET)
            want, kernels = route(main, lambda: main.main(outer, nx, ny, nt, *MARKET))
            assert kernels == SWEEPS and np.array_equal(got, want)


def test_graph_of_main():
    """lvc.graph: main's and main_f64's captured steps, replayed with eager work
    between."""
    print("case: graph replay of main by the sweeps", flush=True)
    with lvc.LocVolCalib() as eager, lvc.LocVolCalib(tuning={"lvc.graph": 1}) as ctx:
        want = eager.main(16, 64, 64, 9, *MARKET), eager.main_f64(5, 32, 300, 12, *MARKET)
        for _ in range(3):
            assert np.array_equal(ctx.main(16, 64, 64, 9, *MARKET), want[0])
            assert np.array_equal(ctx.main(16, 64, 64, 9, *MARKET), want[0])
            eager.main(4, 32, 32, 5, *MARKET)
            eager.sync()
            assert np.array_equal(ctx.main_f64(5, 32, 300, 12, *MARKET), want[1])


@pytest.mark.parametrize("shapes", [SHAPES_X, SHAPES_Y, SHAPES_T, SHAPES_WIDE],
                         ids=["x", "y", "t", "wide"])
def test_modes_at_their_sizes(shapes):
    with lvc.LocVolCalib(profiling=True) as ctx:
        for i, (nx, ny, nt) in enumerate(shapes):
            market = (0.03, 1.1 + 0.37 * i, 0.2, 0.4 + 0.02 * i, (0.0, 0.3, 0.5, 0.7)[i % 4])
            print(f"case: modes of {nx} x {ny} x {nt}, {market}", flush=True)
            got, kernels = route(ctx, lambda: ctx.main_f64(12, nx, ny, nt, *market))
            assert kernels == {"lvc_modes", "lvc_evolve", "lvc_price"}
            ref = oracle_batch(strikes_batch(nx, ny, nt, 0.001 * np.arange(12), market=market))
            assert np.max(np.abs(got - ref) / np.abs(ref)) < 1e-10
