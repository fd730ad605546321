"""Column-split SW pairs of more than 4 symbols (compared codes): 5 to 8
symbols leave the 4-bit row tables where the maximum is kept, more than 8 keep it
whether asked to or not.  Bit-exact against the oracle where the byte tables' tests look: one
strip, rows filled up at the top of the reversed parts (whole waves, part of a
wave), strips with no column left or right of the cut, and the three
parts of pairs with more strips than CUs."""
import numpy as np
import pytest

import oracle as O
from gpumemefficient_amd import Job

pytestmark = pytest.mark.gpu

SHAPES = [(1024, 512), (1024, 513), (1030, 640), (1281, 1151), (1100, 9000), (4099, 4607), (7013, 3001), (5000, 129)]


def _pair(rng, n1, n2, k):
    """Symbols of any int32 value; the second sequence ends like the first."""
    names = np.array([0, 1, 2, 3, 4] if k == 5 else rng.choice(2**31 - 1, k, replace=False) - 2**30, dtype=np.int32)
    a = names[rng.integers(0, k, n1)]
    b = names[rng.integers(0, k, n2)]
    m = min(n1, n2) // 2
    keep = rng.random(m) >= 0.1
    b[n2 - m:][keep] = a[n1 - m:][keep]
    return a, b


def _check(ctx, a, b, k, nomax, parts):
    if a.size * b.size < 1e8:
        want = O.score("SW", a, b)
    else:
        want = O.blocked("SW", a, b, threads=8)
    p = ctx.plan([Job("SW", a, b, no_max=nomax)])
    d = p.describe()
    strips = -(-b.size // (64 * d["waves"] * d["rows_per_lane"]))
    assert d["tasks"] == parts * strips, d
    expect = (want[0], -1 if nomax and k <= 8 else want[1])
    for per_pair in (False, False, True):
        p.run(per_pair=per_pair)
        r = p.results()[0]
        assert r.status == 0 and (r.last, r.max_score) == expect, (d, per_pair)
    p.close()


@pytest.mark.parametrize("nomax", [False, True])
@pytest.mark.parametrize("k", [5, 8, 9, 20, 256])
@pytest.mark.parametrize("n1,n2", SHAPES)
def test_sw_codes_split(ctx, n1, n2, k, nomax):
    a, b = _pair(np.random.default_rng(n1 + 3 * n2 + k), n1, n2, k)
    _check(ctx, a, b, k, nomax, 1 if nomax and k <= 8 else 4)


@pytest.mark.parametrize("k", [7, 20])
def test_sw_codes_split_without_the_zero_boundary_part(ctx, k):
    a, b = _pair(np.random.default_rng(k), 16390, 86 * 512 + 129, k)
    _check(ctx, a, b, k, False, 3)
