"""Server slots: requests with long strip chains (SW n1 + 1.5 n2 >= 65536, LCS
and ED n1 >= 49152) run alone while there are few, in the shared launches when
there are more, with one slot or per request.  Exact against the oracle, twice
on the same server (arenas outgrown and recycled), under a budget that leaves no
room for a split's rows too."""
import numpy as np
import pytest

import oracle as O
from gpumemefficient_amd import Job
from gpumemefficient_amd.server import Server

pytestmark = pytest.mark.gpu


def _want(j):
    if j.a.size * j.b.size < 1e8:
        last, mx = O.score(j.problem, j.a, j.b)[:2]
    else:
        last, mx = O.blocked(j.problem, j.a, j.b, threads=8)[:2]
    return last, mx


def _jobs(rng, sw, ed):
    def pair(k, n1, n2):
        return rng.integers(0, k, n1, dtype=np.int32), rng.integers(0, k, n2, dtype=np.int32)

    jobs = [Job("SW", *pair(4, int(rng.integers(40, 900)), int(rng.integers(40, 900)))) for _ in range(6)]
    jobs += [Job("ED", *pair(20, int(rng.integers(40, 900)), int(rng.integers(40, 900)))) for _ in range(6)]
    sizes = [(64001, 1001), (65536, 515), (20000, 30400), (66000, 257)]
    jobs += [Job("SW", *pair(20 if i == 1 else 4, *sizes[i])) for i in range(sw)]
    jobs += [Job("LCS" if i % 2 else "ED", *pair(4, 49152 + 7 * i, 300 + 700 * i)) for i in range(ed)]
    return [jobs[i] for i in rng.permutation(len(jobs))]


@pytest.mark.parametrize("sw,ed,kw", [(1, 0, {}), (3, 3, {}), (4, 7, {}), (2, 2, {"streams": 1}), (2, 2, {"streams": 2}),
                                      (1, 1, {"per_request": True}), (2, 2, {"hbm_budget": 16 << 20}),
                                      (2, 1, {"max_batch": 1})])
def test_server_long_requests(sw, ed, kw):
    jobs = _jobs(np.random.default_rng(10 * sw + ed), sw, ed)
    want = [_want(j) for j in jobs]
    with Server(0, **kw) as srv:
        for _ in range(2):
            tickets = [srv.submit(j) for j in jobs]
            srv.wait_idle(30.0)
            done = {c.ticket: c for c in srv.poll()}
            for j, t, (last, mx) in zip(jobs, tickets, want):
                c = done[t]
                assert c.status == 0 and c.last == last, (j.problem, j.a.size, j.b.size)
                if j.problem == "SW":
                    assert c.max_score == mx
        assert srv.stats()["hbm_used"] == 0
