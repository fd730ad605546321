"""The staircase cut of column-split SW pairs: strips of the left part and of
the reversed right part end at columns that fall by a strip lag (640 for
512-row strips), rows are filled up at the top of the reversed parts, and pairs
with more strips than CUs run without the part from a zero boundary, the
reversed parts keeping their own maxima.  Bit-exact against the oracle at the
cut's edges: one strip, strips with no column left or right of the cut (tall
pairs), row counts around waves and strips, alignments through the staircase's
rows, and pairs on either side of the limit of three or four parts (two or
three parts are taken from 16384 columns on, where 3 or 4 times the strips
exceed the CUs)."""
import numpy as np
import pytest

import oracle as O
from gpumemefficient_amd import Job, Tile

pytestmark = pytest.mark.gpu

THREE_FOUR = [(1024, 512), (1024, 513), (1024, 640), (1030, 1151), (1281, 1025), (1024, 5120), (1100, 9000),
              (2560, 2048), (4099, 4607), (6401, 5121), (5000, 255), (5000, 257), (5000, 129)]
TWO_THREE = [(16384, 86 * 512), (16390, 43521), (16447, 86 * 512 + 129)]


def _pair(rng, n1, n2, planted):
    a = rng.integers(0, 4, n1, dtype=np.int32)
    b = rng.integers(0, 4, n2, dtype=np.int32)
    if planted:  # a long alignment that ends near the corner, from a column near the middle
        k = min(n2, n1) // 2
        b[n2 - k:] = a[n1 - k:]
        hit = rng.random(k) < 0.1
        b[n2 - k:][hit] = (b[n2 - k:][hit] + 1) % 4
    return a, b


def _check(ctx, a, b, parts):
    want = O.score("SW", a, b) if a.size * b.size < 1e8 else O.blocked("SW", a, b, threads=8)
    for nm, n in zip((True, False), parts):
        p = ctx.plan([Job("SW", a, b, no_max=nm)])
        d = p.describe()
        strips = -(-b.size // (64 * d["waves"] * d["rows_per_lane"]))
        for _ in range(2):
            p.run()
            r = p.results()[0]
            assert r.status == 0 and (r.last, r.max_score) == (want[0], -1 if nm else want[1]), (nm, d)
        assert d["tasks"] == n * strips, d
        p.run(per_pair=True)
        r = p.results()[0]
        assert (r.last, r.max_score) == (want[0], -1 if nm else want[1]), ("per pair", nm, d)
        p.close()


@pytest.mark.parametrize("planted", [False, True])
@pytest.mark.parametrize("n1,n2", THREE_FOUR)
def test_sw_cut_three_and_four_parts(ctx, n1, n2, planted):
    _check(ctx, *_pair(np.random.default_rng(n1 + 3 * n2), n1, n2, planted), (3, 4))


@pytest.mark.parametrize("n1,n2", TWO_THREE)
def test_sw_cut_two_and_three_parts(ctx, n1, n2):
    a, b = _pair(np.random.default_rng(n1 + n2), n1, n2, True)
    want = (2 if 3 * -(-n2 // 512) > 256 else 3, 3 if 4 * -(-n2 // 512) > 256 else 4)
    _check(ctx, a, b, want)


def test_sw_cut_two_parts_graph_replays(ctx):
    a, b = _pair(np.random.default_rng(17), 16500, 86 * 512, True)
    p = ctx.plan([Job("SW", a, b)])
    p.run()
    first = p.results()[0]
    p.capture()
    for _ in range(3):
        p.run()
        r = p.results()[0]
        assert (r.last, r.max_score) == (first.last, first.max_score)
        x, y = _pair(np.random.default_rng(18), 1500, 700, False)
        assert ctx.align("SW", x, y, tile=Tile(no_max=True)).last == O.score("SW", x, y)[0]
    p.close()
