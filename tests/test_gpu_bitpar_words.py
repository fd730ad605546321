"""The staged bit-parallel engine's packed boundaries: lane 63's carries and
deltas travel 32 steps a word, from wave to wave and from strip to strip.
Exact against the oracle at column counts around words (32), chunks (64) and the
lanes' skew (63), over several strips, with one and two compute waves a strip."""
import numpy as np
import pytest

import oracle as O
from gpumemefficient_amd import Job, Tile

pytestmark = pytest.mark.gpu

N1 = [1, 2, 3, 30, 31, 32, 33, 34, 62, 63, 64, 65, 66, 95, 96, 97, 127, 128, 129, 130, 160, 191, 192, 193, 255, 257,
      1023, 1025, 1087, 1089]
N2 = [2048, 2049, 4097, 6200, 8193]


@pytest.mark.parametrize("strip_rows", [2048, 4096])
@pytest.mark.parametrize("prob,textbook", [("LCS", False), ("ED", False), ("ED", True)])
def test_packed_boundaries_match_oracle(ctx, prob, textbook, strip_rows):
    rng = np.random.default_rng(strip_rows + textbook)
    jobs, want = [], []
    for i, n1 in enumerate(N1):
        n2 = N2[i % len(N2)]
        a = rng.integers(0, 4, n1, dtype=np.int32)
        b = rng.integers(0, 4, n2, dtype=np.int32)
        if i % 2:  # long runs of matches: deltas of -1 and carries across the strips
            b[:] = a[np.arange(n2) % n1]
        jobs.append(Job(prob, a, b, ed_textbook=textbook))
        want.append(O.score(prob, a, b, textbook=textbook)[0])
    plan = ctx.plan(jobs, Tile(engine="bitpar_staged", strip_rows=strip_rows))
    assert plan.describe()["waves"] == strip_rows // 2048
    for rep in range(2):
        plan.run()
        got = [r.last for r in plan.results()]
        assert got == want, [(j.a.size, j.b.size, g, w) for j, g, w in zip(jobs, got, want) if g != w]
    plan.close()
