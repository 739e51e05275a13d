"""Far strikes: prices that are a small part of the chord through the grid's
ends, of which the separated form takes its sum, by every entry that uses it,
each price by itself against the FP64 oracle.

Tolerance: the FP64 form's bar of 1e-10 relative, price by price (both sides
round relative to the local values: 1e-12 in the oracle's literal operator);
1e-6 for f32 prices, the bar of the refined form; no price below 0.
"""
import numpy as np
import pytest

from oracle import oracle
import locvolcalib as lvc

pytestmark = pytest.mark.gpu

KEYS = ("numX", "numY", "numT", "s0", "strike", "t", "alpha", "nu", "beta")
# lognormal and steeper markets with little volatility of the volatility, at
# the money to the grid's end; a small elasticity, whose grid is wide
MARKETS = [(256, 32, 32, 0.03, 1.0, 0.21, 0.1, 1.0), (256, 32, 128, 0.03, 1.0, 0.13, 0.02, 1.0),
           (256, 32, 64, 0.03, 1.0, 0.21, 0.1, 1.5), (128, 32, 32, 0.03, 1.0, 0.2, 0.2, 1.0),
           (64, 16, 12, 1.9, 1.1, 0.23, 0.02, 0.03), (100, 40, 20, 0.04, 3.0, 0.12, 0.15, 0.6),
           (40, 20, 30, 0.05, 6.0, 0.15, 0.5, 0.7)]


def market_strikes(m):
    nx, _, _, s0, t, alpha = m[:6]
    dx = 20 * alpha * s0 * np.sqrt(t) / nx
    last = (nx - 1 - int(s0 / dx)) * dx + s0
    return np.concatenate([[0.5 * s0, s0],
                           s0 + (last - s0) * np.array([.05, .15, .3, .45, .6, .8, .95])])


def batch_of():
    rows = [m[:4] + (k,) + m[4:] for m in MARKETS for k in market_strikes(m)]
    return {k: np.array(v) for k, v in zip(KEYS, zip(*rows))}


def oracle_batch(p, **kw):
    return oracle.batch(*[p[k] for k in KEYS], dtype=np.float64, thomas=True, nthreads=8, **kw)


def check(got, ref, bar):
    assert np.all(got >= 0)
    # below 1e-300 the oracle's own products leave the range of doubles
    far = ref > 1e-300
    assert np.max(np.abs(got[far] - ref[far]) / ref[far]) < bar


def test_batch(gpu_ctx):
    p = batch_of()
    print(f"case: far strikes, FP64 batch of {len(p['strike'])}", flush=True)
    got = gpu_ctx.main_batch(**p, precision=lvc.PRECISION_FP64)
    check(got, oracle_batch(p), 1e-10)
    alone = [gpu_ctx.main_batch(**{k: v[i:i + 1] for k, v in p.items()},
                                precision=lvc.PRECISION_FP64)[0] for i in range(0, len(got), 5)]
    assert np.array_equal(got[::5], alone)


@pytest.mark.parametrize("market", [MARKETS[0], MARKETS[2], MARKETS[5]],
                         ids=["lognormal", "steep", "flat"])
def test_main(gpu_ctx, market):
    """main's strikes, 0.001 i, from the grid's first node past its last: near
    ones, far ones and those worth exactly 0 in one call."""
    nx, ny, nt, s0, t, alpha, nu, beta = market
    n = int(1000 * 20 * alpha * s0 * np.sqrt(t)) + 4
    print(f"case: far strikes, main_f64 of {n}", flush=True)
    args = (nx, ny, nt, s0, t, alpha, nu, beta)
    got = gpu_ctx.main_f64(n, *args)
    ref = oracle.main(n, *args, dtype=np.float64, thomas=True, nthreads=8)
    assert ref[-1] == 0 and np.all(got[ref == 0] == 0)
    check(got, ref, 1e-10)
    # an option's price does not depend on how many there are
    for m in (1, n // 3, n // 2, n - 2):
        assert np.array_equal(gpu_ctx.main_f64(m, *args), got[:m])


@pytest.mark.parametrize("precision", [lvc.PRECISION_FP32_REFINE, lvc.PRECISION_FP64])
@pytest.mark.parametrize("market", [MARKETS[0], MARKETS[2]], ids=["lognormal", "steep"])
def test_main_f32(market, precision):
    """The f32 entry and its allocation-free form."""
    nx, ny, nt, s0, t, alpha, nu, beta = market
    args = (nx, ny, nt) + tuple(float(np.float32(v)) for v in (s0, t, alpha, nu, beta))
    n = int(1000 * 20 * alpha * s0 * np.sqrt(t)) + 2
    print(f"case: far strikes, main of {n}, precision {precision}", flush=True)
    strikes = (np.float32(0.001) * np.arange(n, dtype=np.float32)).astype(np.float64)
    p = dict(zip(KEYS, [np.full(n, v) for v in args[:4]] + [strikes] +
                 [np.full(n, v) for v in args[4:]]))
    ref = oracle_batch(p, grid32=True)
    with lvc.LocVolCalib(precision=precision) as ctx:
        got = ctx.main(n, *args)
        assert np.array_equal(got, ctx.main_noalloc(n, *args))
        assert np.array_equal(got[:n // 2], ctx.main_noalloc(n // 2, *args))
    normal = (ref == 0) | (ref > 1e-30)  # f32's range
    check(got[normal].astype(np.float64), ref[normal], 1e-6)


def test_side_by_side():
    """Calls that go both ways run their modes on the second stream beside the
    sweeps: the same bits as one after the other (with profiling), call after
    call on the memory of the one before, in two contexts in turn."""
    print("case: far strikes, modes beside sweeps", flush=True)
    p = batch_of()
    calls = [lambda c: c.main_f64(90, 256, 32, 32, 0.03, 5.0, 0.12, 0.1, 0.5),
             lambda c: c.main_batch(**p, precision=lvc.PRECISION_FP64),
             lambda c: c.main(260, 128, 40, 20, 0.03, 5.0, 0.2, 0.1, 1.0),
             lambda c: c.main_f64(40, 32, 16, 9, 0.03, 1.0, 0.1, 0.2, 0.7),
             lambda c: c.main_f64(3, 64, 64, 12, 0.03, 5.0, 0.2, 0.6, 0.9)]
    with lvc.LocVolCalib(profiling=True) as one:
        want = [call(one) for call in calls]
    with lvc.LocVolCalib() as first, lvc.LocVolCalib() as second:
        for ctx in (first, second, first):
            for _ in range(3):
                for call, ref in zip(calls, want):
                    assert np.array_equal(call(ctx), ref)


def test_side_by_side_with_graph():
    """The same under "lvc.graph", which captures the sweeps' steps."""
    print("case: far strikes, modes beside a captured graph", flush=True)
    p = batch_of()
    calls = [lambda c: c.main_f64(90, 256, 32, 32, 0.03, 5.0, 0.12, 0.1, 0.5),
             lambda c: c.main_batch(**p, precision=lvc.PRECISION_FP64),
             lambda c: c.main_f64(40, 32, 16, 9, 0.03, 1.0, 0.1, 0.2, 0.7)]
    with lvc.LocVolCalib() as eager, lvc.LocVolCalib(tuning={"lvc.graph": 1}) as ctx:
        want = [call(eager) for call in calls]
        for _ in range(3):
            for call, ref in zip(calls, want):
                assert np.array_equal(call(ctx), ref)
                eager.main(4, 32, 32, 5, 0.03, 5.0, 0.2, 0.6, 0.5)
                eager.sync()


def test_many_strikes(gpu_ctx):
    """Thousands of strikes within one grid, near and far."""
    args = (64, 16, 9, 1.5, 2.0, 0.2, 0.1, 0.5)
    print("case: far strikes, main_f64 of 9000", flush=True)
    got = gpu_ctx.main_f64(9000, *args)
    some = np.unique(np.linspace(0, 8999, 60).astype(int))
    p = dict(zip(KEYS, [np.full(len(some), v) for v in args[:4]] + [0.001 * some] +
                 [np.full(len(some), v) for v in args[4:]]))
    check(got[some], oracle_batch(p), 1e-10)
    assert np.array_equal(gpu_ctx.main_f64(2500, *args), got[:2500])
