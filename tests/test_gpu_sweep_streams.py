"""A large FP32 batch steps as two independent halves on two streams.  Its
prices are the same bits as one stream's: the captured graph's (which steps
every problem on the context's stream), and those of small batches below the
rule's line.  Calls follow each other without a wait between, so that a call's
buffers are those the call before has just given back."""
import numpy as np
import pytest

import locvolcalib as lvc

pytestmark = pytest.mark.gpu

# (sizes drawn from, problems): several segment classes with odd sizes, small
# grids only, and rows and columns of the widest classes
MIXES = [((32, 37, 64, 100, 128, 255, 256, 300), 320), ((33, 64), 1100), ((512, 600, 70), 40)]


def problems(sizes, n, seed):
    rng = np.random.default_rng(seed)
    pr = dict(numX=rng.choice(sizes, n).astype(np.int32),
              numY=rng.choice(sizes, n).astype(np.int32),
              numT=rng.integers(9, 14, n).astype(np.int32),
              s0=rng.uniform(0.02, 0.05, n), strike=rng.uniform(0.0, 0.05, n),
              t=rng.uniform(1, 10, n), alpha=rng.uniform(0.1, 0.3, n),
              nu=rng.uniform(0.4, 0.8, n), beta=rng.uniform(0.3, 0.7, n))
    pr["numT"][n // 2] = 2                     # one step only
    # largest first, then one large and one small in turn
    order = np.argsort(-(pr["numX"].astype(np.int64) * pr["numY"]))
    half = n // 2
    order[half:] = np.stack([order[half:half + (n - half) // 2 * 2].reshape(2, -1)],
                            0)[0].T.reshape(-1).tolist() + order[half + (n - half) // 2 * 2:].tolist()
    return {k: v[order] for k, v in pr.items()}


@pytest.mark.parametrize("precision", [lvc.PRECISION_FP32, lvc.PRECISION_FP32_REFINE])
@pytest.mark.parametrize("sizes,n", MIXES)
def test_two_streams_keep_the_bits(sizes, n, precision):
    print(f"case: {n} problems of {sizes}, precision {precision}", flush=True)
    a, b = problems(sizes, n, 1), problems(sizes, n - 1, 2)
    with lvc.LocVolCalib(tuning={"lvc.graph": 1}) as ctx:
        want_a = ctx.main_batch(**a, precision=precision)
        want_b = ctx.main_batch(**b, precision=precision)
    with lvc.LocVolCalib() as ctx:
        for _ in range(3):
            assert np.array_equal(ctx.main_batch(**a, precision=precision), want_a)
            assert np.array_equal(ctx.main_batch(**b, precision=precision), want_b)
        some = np.arange(0, n, max(1, n // 12))
        few = {k: v[some] for k, v in a.items()}
        assert np.array_equal(ctx.main_batch(**few, precision=precision), want_a[some])
        # a shared run among the problems: one stream
        c = {k: np.concatenate([v, v[-2:-1], v[-2:-1]]) for k, v in a.items()}
        got = ctx.main_batch(**c, precision=precision)
    assert np.array_equal(got[:n], want_a)
    assert got[n] == want_a[n - 2] and got[n + 1] == want_a[n - 2]


@pytest.mark.parametrize("precision", [lvc.PRECISION_FP32, lvc.PRECISION_FP32_REFINE])
def test_equal_problems_apart_in_the_list(precision):
    """Equal problems with one of another segment class between them: they are
    neighbours in their class's list, and may come to lie on either stream."""
    print(f"case: equal problems in turn with others, precision {precision}", flush=True)
    one = problems((256,), 30, 3)
    pr = {k: np.repeat(v, 2) for k, v in one.items()}
    pr["numX"][1::2] = 600
    pr["numY"][1::2] = 40
    pr = {k: np.concatenate([np.tile(v[:2], 8), v]) for k, v in pr.items()}
    pr["strike"] = np.linspace(0.0, 0.04, len(pr["strike"]))
    with lvc.LocVolCalib(tuning={"lvc.graph": 1}) as ctx:
        want = ctx.main_batch(**pr, precision=precision)
    with lvc.LocVolCalib() as ctx:
        for _ in range(3):
            assert np.array_equal(ctx.main_batch(**pr, precision=precision), want)
        for i in (0, 1, 2, 15, len(want) - 1):
            alone = {k: v[i:i + 1] for k, v in pr.items()}
            assert ctx.main_batch(**alone, precision=precision)[0] == want[i]
