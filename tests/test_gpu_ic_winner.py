"""InterestCalib's winner, the left fold of :752-756 over the last population:
the first genome of the largest log-likelihood, for populations around the
lanes and the workgroup that fold it.  Without swaptions every log-likelihood
is the same (an empty sum) and genome 0 wins; with them the fold is restated
on the traced log-likelihoods."""
import numpy as np
import pytest

from conftest import load_ic_dataset
from locvolcalib import interestcalib as icl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pop", [1, 2, 63, 64, 65, 256, 257, 600])
@pytest.mark.parametrize("swaptions", [0, 3])
def test_first_of_the_largest(pop, swaptions):
    print(f"case: {pop} genomes, {swaptions} swaptions", flush=True)
    data, *_ = load_ic_dataset("small")
    sw = np.asarray(data["swaptions"], np.float32)[:swaptions].reshape(-1, 4)
    with icl.InterestCalib(device=0) as ctx:
        # one genome has no other to differ from: no moves (:700-712)
        tr = ctx.trace(pop, 3 if pop > 1 else 0, sw, data["herm_x"], data["herm_w"], data["dir_vct"])
    first, value = 0, np.float32(-np.inf)
    for i, v in enumerate(tr["logliks"][-1]):
        if value < v:
            first, value = i, v
    if swaptions == 0:
        assert first == 0
    g = tr["genomes"][-1][first]
    assert np.array_equal(tr["out"], np.array([g[0], g[1], g[4], g[3], g[2], value], np.float32))
