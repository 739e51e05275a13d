"""OptionPricing's models in one pass over the paths where only some leave the
range of the log form: a model's mean is the one it has alone, bit for bit (its
paths' arithmetic is its own), and within rtol 2e-5 of the oracle as in
test_gpu_op_paths.py.
"""
import numpy as np
import pytest

from oracle import oracle
from locvolcalib import optionpricing as op
from test_gpu_op_paths import RTOL, load

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("contract", [1, 2, 3])
@pytest.mark.parametrize("outside", [[0], [1], [0, 2], [3], [0, 1, 2, 3]])
def test_a_model_outside_the_range(contract, outside):
    """`outside`: models whose start prices the log form does not take; the
    others' volatilities differ."""
    args, models = load(contract), 4
    args[1] = 193
    for i in range(3, 9):
        args[i] = np.repeat(args[i], models, 0)
    for m in range(models):
        args[4][m] *= np.float32(0.8 + 0.15 * m)
        if m in outside:
            args[6][m] *= np.float32(1e-9)
    print(f"contract {contract}, models {outside} outside", flush=True)
    with op.OptionPricing(device=0) as ctx:
        got = ctx.main(*args)
        np.testing.assert_allclose(got, oracle.op_main(*args), rtol=RTOL)
        for m in range(models):
            one = args[:3] + [np.ascontiguousarray(a[m:m + 1]) for a in args[3:9]] + args[9:]
            np.testing.assert_array_equal(ctx.main(*one), got[m:m + 1])
