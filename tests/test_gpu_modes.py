"""Prices by separation of x (lvc_modes_kernels.hip) against the FP64 oracle,
at the sizes where the split of its work changes: blocks of 16 nodes and 4
modes per wavefront in x; 8, 12 or 16 rows per lane and 1 to 64 lanes per
mode in y; 64 steps per refill of the time factors.

Tolerance: the bar of the FP64 form, 1e-10 relative.  The FP64 oracle's
literal operator loses up to about 900 ulp per step to cancellation, 1e-13
per step and price; the modes' sums lose an ulp of the chord through the
grid's ends, at most 100 times the prices here.
"""
import numpy as np
import pytest

from oracle import oracle
import locvolcalib as lvc

pytestmark = pytest.mark.gpu

KEYS = ("numX", "numY", "numT", "s0", "strike", "t", "alpha", "nu", "beta")
# numX around the blocks of 16 nodes and the waves of 4 modes; numY around
# 8 lanes x 8 rows, the 12 and 16 row variants and the wider exchanges
SHAPES_X = [(nx, 12, 9) for nx in (3, 4, 5, 6, 7, 17, 18, 19, 34, 66)]
SHAPES_Y = [(9, ny, 7) for ny in (3, 8, 9, 16, 17, 64, 65, 128, 129, 192, 193, 256, 257,
                                  384, 385, 512, 513, 768, 769, 1024)]
SHAPES_T = [(8, 10, nt) for nt in (7, 64, 65, 66, 129, 200)]
SHAPES_WIDE = [(1024, 9, 8), (1023, 5, 7), (300, 40, 12)]


def problems(shapes, seed):
    rng = np.random.default_rng(seed)
    n = len(shapes)
    p = dict(zip(("numX", "numY", "numT"), np.array(shapes, np.int32).T))
    p.update(s0=rng.uniform(0.02, 0.05, n), strike=rng.uniform(0.0, 0.05, n),
             t=rng.uniform(1, 10, n), alpha=rng.uniform(0.1, 0.3, n),
             nu=rng.uniform(0.4, 0.8, n), beta=rng.uniform(0.0, 1.0, n))
    return p


def oracle_batch(p):
    return oracle.batch(*[p[k] for k in KEYS], dtype=np.float64, thomas=True, nthreads=8,
                        allow_nan=True)


@pytest.mark.parametrize("shapes", [SHAPES_X, SHAPES_Y, SHAPES_T, SHAPES_WIDE],
                         ids=["x", "y", "t", "wide"])
def test_shapes_vs_oracle(gpu_ctx, shapes):
    print(f"case: modes, {len(shapes)} shapes from {shapes[0]}", flush=True)
    p = problems(shapes, seed=len(shapes))
    got = gpu_ctx.main_batch(**p, precision=lvc.PRECISION_FP64)
    ref = oracle_batch(p)
    assert np.array_equal(np.isfinite(got), np.isfinite(ref))
    fin = np.isfinite(ref)
    # a strike above the grid's last node is worth exactly 0
    assert np.all(got[ref == 0] == 0)
    some = fin & (ref != 0)
    assert np.max(np.abs(got[some] - ref[some]) / np.abs(ref[some])) < 1e-10


def test_strikes_on_and_between_nodes(gpu_ctx):
    """Strikes at, between and beyond the grid's nodes, many on one grid: the
    payoff's kink at every place, no kink below the first and above the last
    node; and beta = 0, where every weight is the same."""
    print("case: modes, 60 strikes on one grid", flush=True)
    nx, s0, t, alpha = 24, 0.03, 5.0, 0.2
    dx = 20 * alpha * s0 * np.sqrt(t) / nx
    x = np.arange(nx) * dx - int(s0 / dx) * dx + s0
    strikes = np.concatenate([[-0.01, x[0] / 2, x[-1] + 1e-9, 1.0], x[:-3],
                              0.3 * x[:-4] + 0.7 * x[1:-3]])
    n = len(strikes)
    for beta in (0.0, 0.5):
        p = dict(numX=np.full(n, nx), numY=np.full(n, 20), numT=np.full(n, 30),
                 s0=np.full(n, s0), strike=strikes, t=np.full(n, t), alpha=np.full(n, alpha),
                 nu=np.full(n, 0.6), beta=np.full(n, beta))
        got = gpu_ctx.main_batch(**p, precision=lvc.PRECISION_FP64)
        ref = oracle_batch(p)
        # near the last nodes the price is a small part of the chord
        assert np.max(np.abs(got - ref)) < 1e-10 * np.max(np.abs(ref)) * 1e-2
        assert np.all(got[strikes > x[-1]] == 0.0)


def test_what_does_not_separate_takes_the_sweeps():
    """Few steps, a price node at the grid's edge and parameters outside the
    separated range give the oracle's prices or its NaN, mixed with separated
    problems in one batch."""
    print("case: modes and sweeps in one batch", flush=True)
    n = 6
    p = dict(numX=np.full(n, 40), numY=np.full(n, 24), numT=np.array([6, 7, 30, 30, 30, 12]),
             s0=np.full(n, 0.03), strike=np.full(n, 0.01), t=np.array([5, 5, 4.0, 5, 5, 5]),
             alpha=np.full(n, 0.2), nu=np.array([0.6, 0.6, 0.6, 0.6, 0.6, 0.6]),
             beta=np.array([0.5, 0.5, 0.5, -0.3, 6.0, 0.5]))
    ref = oracle_batch(p)
    with lvc.LocVolCalib() as ctx:
        got = ctx.main_batch(**p, precision=lvc.PRECISION_FP64)
        alone = [ctx.main_batch(**{k: v[i:i + 1] for k, v in p.items()},
                                precision=lvc.PRECISION_FP64)[0] for i in range(n)]
    assert np.array_equal(got, alone, equal_nan=True)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    fin = np.isfinite(ref)
    assert np.max(np.abs(got[fin] - ref[fin]) / np.abs(ref[fin])) < 1e-10
