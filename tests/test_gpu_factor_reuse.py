"""The column y sweep's factor table is kept from one step to the next while
the f32 time step stays the same number.

Timelines are chosen so that the step (numT - 1) / t lies half way between
two floats: FP64 rounding then moves dt between the two from step to step, and
the table is made again and again.  And a server slot passes from a request to
the next one of the same size: its prices are those of a fresh server, bit for
bit.  Bars as elsewhere: 1e-6 of the largest price with refinement, 1e-4
without, against the FP64 oracle.
"""
import numpy as np
import pytest

from oracle import oracle
import locvolcalib as lvc

pytestmark = pytest.mark.gpu

KEYS = ("numX", "numY", "numT", "s0", "strike", "t", "alpha", "nu", "beta")


def half_way(num_t, step):
    """t for which (num_t - 1) / t is half way between two floats near step."""
    f = np.float32(step)
    return (num_t - 1) / ((float(f) + float(np.nextafter(f, np.float32(np.inf)))) / 2)


def changes(t, num_t):
    k = np.arange(num_t - 1)
    dt = (1.0 / (t * (k + 1) / (num_t - 1.0) - t * k / (num_t - 1.0))).astype(np.float32)
    return int((dt[1:] != dt[:-1]).sum())


def problems():
    rng = np.random.default_rng(4)
    num_t = np.array([12, 20, 33, 12, 20, 33], np.int32)
    t = np.array([half_way(n, s) for n, s in zip(num_t, (2.0, 3.1, 7.3, 7.3, 2.0, 3.1))])
    assert sum(changes(a, b) > 2 for a, b in zip(t, num_t)) >= 4
    n = len(num_t)
    return dict(numX=np.array([40, 64, 33, 96, 128, 50], np.int32),
                numY=np.array([33, 64, 130, 40, 200, 70], np.int32), numT=num_t,
                s0=rng.uniform(0.02, 0.05, n), strike=rng.uniform(0.0, 0.05, n), t=t,
                alpha=rng.uniform(0.1, 0.3, n), nu=rng.uniform(0.4, 0.8, n),
                beta=rng.uniform(0.3, 0.7, n))


@pytest.mark.parametrize("precision,bar", [(lvc.PRECISION_FP32_REFINE, 1e-6),
                                           (lvc.PRECISION_FP32, 1e-4)])
@pytest.mark.parametrize("seg_y", [32, 64])
def test_steps_of_two_values(precision, bar, seg_y):
    print(f"precision {precision}, column segments of {seg_y}", flush=True)
    pr = problems()
    with lvc.LocVolCalib(tuning={"lvc.seg_y": seg_y}) as ctx:
        got = ctx.main_batch(**pr, precision=precision)
    ref = oracle.batch(*[pr[k] for k in KEYS], dtype=np.float64, thomas=True, nthreads=4)
    assert np.max(np.abs(got - ref)) / np.max(np.abs(ref)) < bar


def test_slot_passes_to_the_next_request():
    pr = problems()
    rows = [tuple(pr[k][i].item() for k in KEYS) for i in range(len(pr["t"]))]
    # the same grid and slot, other steps and volatilities
    rows = [(64, 64) + r[2:] for r in rows]
    fresh = []
    with lvc.LocVolCalib() as ctx:
        for r in rows:
            srv = lvc.Server(ctx, max_slots=1, precision=lvc.PRECISION_FP32_REFINE)
            i = srv.submit(*r)
            srv.drain()
            fresh.append(srv.poll(i))
            srv.free()
        srv = lvc.Server(ctx, max_slots=1, precision=lvc.PRECISION_FP32_REFINE)
        ids = [srv.submit(*r) for r in rows]
        srv.drain()
        got = [srv.poll(i) for i in ids]
        srv.free()
    assert got == fresh
