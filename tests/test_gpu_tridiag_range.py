"""The staged tridiagonal solves where their divisions leave the range of the
short form: bit-exact against the oracle (IEEE division) on systems whose
pivots or numerators are zero, denormal, huge, tiny or infinite, alone or among
ordinary systems, and in a last workgroup that is not full."""
import numpy as np
import pytest

from oracle import oracle
import locvolcalib as lvc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with lvc.LocVolCalib() as c:
        yield c


def systems(kind, n, m):
    """Diagonally dominant rows, then what `kind` makes of some of them."""
    rng = np.random.default_rng(n * 1000 + m)
    a, c = (-rng.random((n, m)) for _ in range(2))
    a[:, 0] = c[:, -1] = 0
    b, y = 1 - a - c, rng.standard_normal((n, m))
    one = rng.integers(0, n)          # one system among ordinary ones
    if kind == "large":               # every coupling scaled up, pivots past 2^40
        a, b, c, y = a * 2.0 ** 50, b * 2.0 ** 50, c * 2.0 ** 50, y * 2.0 ** 50
    elif kind == "small":
        a, b, c, y = a * 2.0 ** -60, b * 2.0 ** -60, c * 2.0 ** -60, y * 2.0 ** -60
    elif kind == "tiny numerators":   # denormal couplings and right-hand sides
        a[one] *= 2.0 ** -130
        c[one] *= 2.0 ** -130
        y[one] *= 2.0 ** -140
    elif kind == "zeros":             # a zero pivot, zero couplings
        b[one, m // 2] = 0
        a[one, m // 2] = 0
        y[one] = 0
    elif kind == "infinite":
        y[one, m // 2] = np.inf
    elif kind == "nan":
        b[one, m // 2] = np.nan
    with np.errstate(over="ignore"):
        return [np.ascontiguousarray(v, np.float32) for v in (a, b, c, y)]


@pytest.mark.parametrize("kind", ["plain", "large", "small", "tiny numerators", "zeros",
                                  "infinite", "nan"])
@pytest.mark.parametrize("n,m", [(1, 5), (64, 16), (70, 115), (130, 128)])
def test_bits_beyond_the_short_division(ctx, kind, n, m):
    print(f"{kind}, [{n}][{m}]", flush=True)
    v = systems(kind, n, m)
    for seq, fn in ((True, oracle.tridag_seq), (False, oracle.tridag_par4)):
        got = ctx.tridag_nested(*v, seq=seq)
        ref = np.stack([fn(*(w[i] for w in v)) for i in range(n)])
        assert np.array_equal(got, ref, equal_nan=True)
