"""OptionPricing's path kernels where they take another route than the
datasets do, against the oracle (f32 in the reference's order of operations,
mean in f64).

Routes of contract 3: a bridge whose live dates fit the slots in LDS (the
reference's left-first order), one that needs a slot per date (a chain), one
whose dates complete only at its end (right first), and prices that leave the
range of the log form (priced by the running product).  Of contracts 1 to 3:
several models that share a pass over the paths, or take more than one.

Tolerance: rtol 2e-5 as in test_gpu_optionpricing.py, where it is derived:
an ulp of the device's functions moves a payoff by a few ulps and, rarely, a
path over a barrier.  Models in one call against one call each: the arithmetic
of a path is the same, so the means are equal.
"""
import os

import numpy as np
import pytest

from conftest import GOLDEN
from oracle import oracle
from locvolcalib import futhark_values as fv
from locvolcalib import optionpricing as op

pytestmark = pytest.mark.gpu

RTOL = 2e-5
NAMES = {1: "small", 2: "medium", 3: "large"}


@pytest.fixture(scope="module")
def ctx():
    c = op.OptionPricing(device=0)
    yield c
    c.free()


def load(contract):
    path = os.path.join(GOLDEN, "OptionPricing-data", NAMES[contract] + ".in")
    return list(op.main_arguments(fv.load(path)))


def bridge(dates, order):
    """bb_inds, bb_data of a bridge over equal steps: the last date, then the
    others between built neighbours, "left" or "right" part first, or in a
    chain from the last date down."""
    t = np.arange(dates + 1) / 100.0
    steps = [(dates, 0, 0, np.sqrt(t[dates]), 0.0, 0.0)]
    if order == "chain":
        todo = [(0, hi, hi - 1) for hi in range(dates, 1, -1)]
    else:
        todo, stack = [], [(0, dates)]
        while stack:
            lo, hi = stack.pop()
            if hi - lo < 2:
                continue
            mid = (lo + hi) // 2
            todo.append((lo, hi, mid))
            parts = [(mid, hi), (lo, mid)]
            stack += parts if order == "left" else parts[::-1]
    for lo, hi, mid in todo:
        whole = t[hi] - t[lo]
        steps.append((mid, lo, hi, np.sqrt((t[mid] - t[lo]) * (t[hi] - t[mid]) / whole),
                      (t[hi] - t[mid]) / whole, (t[mid] - t[lo]) / whole))
    a = np.array(steps)
    return a[:, :3].T.astype(np.int32).copy(), a[:, 3:].T.astype(np.float32).copy()


def check(ctx, args):
    want = oracle.op_main(*args)
    assert np.all(np.isfinite(want))
    np.testing.assert_allclose(ctx.main(*args), want, rtol=RTOL)


@pytest.mark.parametrize("contract", [2, 3])
@pytest.mark.parametrize("order", ["left", "right", "chain"])
@pytest.mark.parametrize("paths", [65, 2111])
def test_bridge_orders(ctx, contract, order, paths):
    args = load(contract)
    args[1] = paths
    args[9], args[10] = bridge(args[9].shape[1], order)
    print(f"contract {contract}, {order}, {paths} paths", flush=True)
    check(ctx, args)


# (start prices' factor, volatilities' factor): starts outside the log form's
# 1e-4 .. 1e8, and returns that leave +-60
@pytest.mark.parametrize("contract", [2, 3])
@pytest.mark.parametrize("start,vol", [(1e-9, 1.0), (1e6, 1.0), (1.0, 0.0), (1.0, 40.0)])
def test_range_of_the_log_prices(ctx, contract, start, vol):
    args = load(contract)
    args[1] = 700
    args[6] = (args[6] * np.float32(start)).astype(np.float32)
    args[4] = (args[4] * np.float32(vol)).astype(np.float32)
    print(f"contract {contract}, starts x {start}, volatilities x {vol}", flush=True)
    check(ctx, args)


@pytest.mark.parametrize("contract", [1, 2, 3])
@pytest.mark.parametrize("models", [2, 4, 5])
def test_models_share_a_pass(ctx, contract, models):
    args = load(contract)
    args[1] = 1500
    rng = np.random.default_rng(models)
    for i in range(3, 9):
        args[i] = np.repeat(args[i], models, 0)
    for i in (4, 5, 6):
        factor = 1 + 0.05 * rng.standard_normal((models,) + (1,) * (args[i].ndim - 1))
        args[i] = (args[i] * factor).astype(np.float32)
    print(f"contract {contract}, {models} models", flush=True)
    got = ctx.main(*args)
    np.testing.assert_allclose(got, oracle.op_main(*args), rtol=RTOL)
    for m in range(models):
        one = args[:3] + [np.ascontiguousarray(a[m:m + 1]) for a in args[3:9]] + args[9:]
        np.testing.assert_array_equal(ctx.main(*one), got[m:m + 1])


@pytest.mark.parametrize("paths", [(1 << 15) + 3, 1 << 18])
def test_gaussian_tails(ctx, paths):
    """Sobol numbers down to 2^-19 of 0 and 1: beyond the polynomial's 2^-13."""
    args = load(1)
    args[1] = paths
    check(ctx, args)
