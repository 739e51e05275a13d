"""The server's device lists: descriptors and tiles taken from pinned memory by
the setup launch, finished requests' tiles left in the list until half of it is
dead, prices written to pinned memory.  Requests of very different sizes and
lengths (2 steps of 3 x 3 to 30 steps of 130 x 200) pass through few or many
slots, by ticks with late submissions or by drain; every price is, bit for bit,
that of the request served alone.
"""
import numpy as np
import pytest

import locvolcalib as lvc

pytestmark = pytest.mark.gpu


def requests(n, seed):
    rng = np.random.default_rng(seed)
    sizes = [(3, 3), (130, 200), (32, 17), (64, 64), (5, 90), (200, 3)]
    return [sizes[i % len(sizes)] + (int(rng.integers(2, 31)), rng.uniform(0.02, 0.05),
                                     rng.uniform(0.0, 0.05), rng.uniform(1, 10),
                                     rng.uniform(0.1, 0.3), rng.uniform(0.4, 0.8),
                                     rng.uniform(0.3, 0.7)) for i in range(n)]


@pytest.fixture(scope="module")
def alone():
    prices = {}
    for precision in (lvc.PRECISION_FP32_REFINE, lvc.PRECISION_FP64):
        with lvc.LocVolCalib() as ctx:
            out = []
            for r in requests(40, 6):
                srv = lvc.Server(ctx, max_slots=1, precision=precision)
                i = srv.submit(*r)
                srv.drain()
                out.append(srv.poll(i))
                srv.free()
        prices[precision] = out
    return prices


@pytest.mark.parametrize("precision", [lvc.PRECISION_FP32_REFINE, lvc.PRECISION_FP64])
@pytest.mark.parametrize("slots", [1, 3, 64])
@pytest.mark.parametrize("late", [False, True])
def test_prices_do_not_depend_on_the_lists(alone, precision, slots, late):
    print(f"precision {precision}, {slots} slots, late submissions {late}", flush=True)
    rows = requests(40, 6)
    with lvc.LocVolCalib() as ctx:
        srv = lvc.Server(ctx, max_slots=slots, precision=precision)
        ids = []
        for r in rows:
            ids.append(srv.submit(*r))
            if late:
                srv.step()
        srv.drain()
        got = [srv.poll(i) for i in ids]
        srv.free()
    assert got == alone[precision]
