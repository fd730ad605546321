"""LCS and ED pairs cut along a staircase (staged bit-parallel engine, one wave
a strip): exact against the oracle where the cut can go wrong: one strip and
several, rows filled up at the top of the reversed half (part of a word, whole
words), pairs too narrow for the full lag (down to none), horizontal runs that
are no whole number of words, both ED boundaries, related and independent
sequences, the launch pair by pair and replayed from a graph."""
import numpy as np
import pytest

import oracle as O
from gpumemefficient_amd import Job

pytestmark = pytest.mark.gpu

SHAPES = [(1024, 2048), (1025, 2049), (1024, 4095), (1090, 6145), (1500, 20000), (4099, 2047), (5003, 4128),
          (8192, 8192), (9001, 10241), (1024, 2), (20011, 16385)]


def _pair(rng, n1, n2, k, related):
    a = rng.integers(0, k, n1, dtype=np.int32)
    b = rng.integers(0, k, n2, dtype=np.int32)
    m = min(n1, n2)
    keep = rng.random(m) >= 0.1
    if related == "head":
        b[:m][keep] = a[:m][keep]
    elif related == "tail":
        b[n2 - m:][keep] = a[n1 - m:][keep]
    return a, b


@pytest.mark.parametrize("related", ["", "head", "tail"])
@pytest.mark.parametrize("problem,textbook", [("LCS", False), ("ED", False), ("ED", True)])
@pytest.mark.parametrize("n1,n2", SHAPES)
def test_bitpar_staircase(ctx, n1, n2, problem, textbook, related):
    a, b = _pair(np.random.default_rng(n1 + 3 * n2), n1, n2, 4 if problem == "LCS" else 20, related)
    if n1 * n2 < 1e8:
        want = O.score(problem, a, b, textbook=textbook)[0]
    else:
        want = O.blocked(problem, a, b, textbook=textbook, threads=8)[0]
    p = ctx.plan([Job(problem, a, b, ed_textbook=textbook)])
    d = p.describe()
    assert d["engine"] == "bitpar_staged" and d["tasks"] == 2 * -(-n2 // 2048)
    for per_pair in (False, False, True):
        p.run(per_pair=per_pair)
        r = p.results()[0]
        assert r.status == 0 and r.last == want, (d, per_pair)
    p.close()


@pytest.mark.parametrize("problem,edge", [("ED", 576), ("LCS", 832)])
def test_bitpar_split_narrowest(ctx, problem, edge):
    """One column either side of the narrowest split pair, one strip and many
    (whose lag is then a few steps)."""
    rng = np.random.default_rng(edge)
    for n1, n2 in ((edge - 1, 900), (edge, 900), (edge, 30001), (edge + 1, 4097)):
        a, b = _pair(rng, n1, n2, 20 if problem == "ED" else 4, "head")
        p = ctx.plan([Job(problem, a, b)])
        assert p.describe()["tasks"] == (1 if n1 < edge else 2) * -(-n2 // 2048)
        p.run()
        assert p.results()[0].last == O.score(problem, a, b)[0]
        p.close()


def test_bitpar_staircase_graph_replays(ctx):
    rng = np.random.default_rng(5)
    jobs = [Job("ED", *_pair(rng, 3001, 7000, 20, "head")), Job("LCS", *_pair(rng, 700, 900, 4, "")),
            Job("LCS", *_pair(rng, 4000, 4097, 4, "tail"))]
    want = [O.score(j.problem, j.a, j.b)[0] for j in jobs]
    p = ctx.plan(jobs)
    p.capture()
    for _ in range(4):
        p.run()
        assert [r.last for r in p.results()] == want
        x, y = _pair(rng, 1500, 700, 4, "")
        assert ctx.align("LCS", x, y).last == O.score("LCS", x, y)[0]
    p.close()
