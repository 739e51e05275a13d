"""InterestCalib's evaluation with several virtual lanes on one physical lane:
a genome's prices are the same bits whether few genomes are evaluated (one
virtual lane each) or enough that the lanes are packed 2 or 4 to one, for
schedules around the powers of two of a lane's periods."""
import numpy as np
import pytest

from conftest import load_ic_dataset
from locvolcalib import interestcalib as icl

pytestmark = pytest.mark.gpu

# semi-annual schedules of 1 .. 128 periods: 12 * term / frequency
PERIODS = [1, 2, 3, 4, 5, 8, 9, 15, 16, 17, 18, 20, 30, 31, 32, 33, 40, 50, 60, 63, 64, 65, 96,
           127, 128]


@pytest.mark.parametrize("pop", [300, 700, 2500])
def test_prices_do_not_depend_on_the_packing(pop):
    print(f"case: {pop} genomes against 8 at a time", flush=True)
    data, *_ = load_ic_dataset("small")
    rng = np.random.default_rng(pop)
    sw = np.array([[1 + i % 7, 6.0, p / 2.0, 0.2 + 0.01 * i] for i, p in enumerate(PERIODS * 4)],
                  np.float32)
    g = np.stack([rng.uniform(0.05, 0.9, pop), rng.uniform(0.05, 0.9, pop),
                  rng.uniform(-0.9, 0.9, pop), rng.uniform(0.005, 0.19, pop),
                  rng.uniform(0.005, 0.19, pop)], 1).astype(np.float32)
    with icl.InterestCalib(device=0) as ctx:
        _, prices, logliks = ctx.eval_genomes(g, sw, data["herm_x"], data["herm_w"])
        for i in (0, 8, pop - 8):
            _, few, ll = ctx.eval_genomes(g[i:i + 8], sw, data["herm_x"], data["herm_w"])
            assert np.array_equal(prices[i:i + 8], few, equal_nan=True)
            assert np.array_equal(logliks[i:i + 8], ll, equal_nan=True)
