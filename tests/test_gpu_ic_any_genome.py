"""interestcalib_eval of genomes far outside the calibration's genes, where the
quotients' short form does not hold, against the oracle; and of ordinary ones
in a call with such a genome, which have the bits they have without it.

Tolerance: 1e-3 relative or 1e-7, the noise of f32 prices of 1e-5 .. 1 from sums
of terms of order 1 (the device's expf against the host's).
"""
import numpy as np
import pytest

from conftest import load_ic_dataset
from oracle import oracle
from locvolcalib import interestcalib

pytestmark = pytest.mark.gpu

# a, b, rho, nu, sigma: squares past 2^126, whose reciprocal is denormal
FAR = np.array([[1.5669239e+19, 2.4224730e+02, 9.5162493e-01, 8.0098639e+02, 4.5982154e+17],
                [1.8173155e+19, 4.7054498e+02, 5.6245834e-01, 4.2906191e+03, 3.4167942e+17],
                [9.6210423e+18, 3.4075101e+02, -2.7034441e-01, 5.0538095e+02, 8.4614374e+18]],
               np.float32)
ORDINARY = np.array([[0.02, 0.6, -0.5, 0.01, 0.05], [0.3, 0.01, 0.9, 0.15, 0.002]], np.float32)


def test_any_genome():
    print("case: interestcalib_eval, genomes outside the calibration's range", flush=True)
    args, _, _ = load_ic_dataset("small")
    rest = (args["swaptions"][:12], args["herm_x"], args["herm_w"])
    genomes = np.concatenate([FAR, ORDINARY])
    with interestcalib.InterestCalib() as ctx:
        _, prices, logliks = ctx.eval_genomes(genomes, *rest)
        _, alone, logliks_alone = ctx.eval_genomes(ORDINARY, *rest)
    for g, p in zip(genomes, prices):
        np.testing.assert_allclose(p, oracle.ic_eval(g, *rest)[1], rtol=1e-3, atol=1e-7)
    assert np.array_equal(prices[len(FAR):], alone)
    assert np.array_equal(logliks[len(FAR):], logliks_alone)
