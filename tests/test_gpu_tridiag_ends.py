"""The staged tridiagonal solves with anything in the entries that no solve
reads, a[0] and c[m-1]: bit-exact against the oracle on the same systems with
zeros there, and no slower (the kernels leave the short divisions for the whole
wavefront, at four times the time, where the matrix leaves their range).
"""
import json

import numpy as np
import pytest

from oracle import oracle
import locvolcalib as lvc

pytestmark = pytest.mark.gpu


def systems(n, m, junk):
    rng = np.random.default_rng(n + m)
    a, c = (-rng.random((n, m)) for _ in range(2))
    b, y = 1 - a - c, rng.standard_normal((n, m))
    a[:, 0] = c[:, -1] = 0
    clean = [np.ascontiguousarray(v, np.float32) for v in (a, b, c, y)]
    dirty = [v.copy() for v in clean]
    dirty[0][:, 0] = dirty[2][:, -1] = np.float32(junk)
    return clean, dirty


@pytest.mark.parametrize("junk", [1e-30, 1e30, np.inf, np.nan])
@pytest.mark.parametrize("n,m", [(70, 1), (70, 2), (130, 5), (64, 16), (70, 31), (200, 33), (70, 115),
                                 (130, 128)])
def test_bits(n, m, junk):
    print(f"[{n}][{m}], {junk} in the unread entries", flush=True)
    clean, dirty = systems(n, m, junk)
    with lvc.LocVolCalib() as ctx:
        for seq, fn in ((True, oracle.tridag_seq), (False, oracle.tridag_par4)):
            ref = np.stack([fn(*(w[i] for w in clean)) for i in range(n)])
            assert np.array_equal(ctx.tridag_nested(*dirty, seq=seq), ref)


@pytest.mark.parametrize("junk", [1e-30, 1e30])
@pytest.mark.parametrize("m", [11, 60, 115, 128])
@pytest.mark.parametrize("seq", [True, False])
def test_time(m, seq, junk):
    print(f"[20000][{m}], seq {seq}, {junk} in the unread entries", flush=True)
    clean, dirty = systems(20000, m, junk)

    def fastest(ctx, v):
        times, total = [], 0.0
        for _ in range(8):
            ctx.tridag_nested(*v, seq=seq)
            now = sum(k["total_us"] for k in json.loads(ctx.report()).values()
                      if isinstance(k, dict))
            times.append(now - total)
            total = now
        return min(times)

    with lvc.LocVolCalib(profiling=True) as one, lvc.LocVolCalib(profiling=True) as two:
        assert fastest(two, dirty) < 1.7 * fastest(one, clean)
