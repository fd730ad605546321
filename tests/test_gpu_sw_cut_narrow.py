"""Narrow SW pairs with more strips than three or four parts have CUs for: two
parts (no maximum) or three, down to the narrowest width that is split and up to
the most strips that the chip holds, where most strips have no column on one side
of the cut.  Bit-exact against the oracle, the route on either side of each limit."""
import numpy as np
import pytest

import oracle as O
from gpumemefficient_amd import Job

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n1,strips,rem,k", [(1023, 65, 0, 4), (1024, 64, 0, 4), (1024, 65, 383, 4), (1025, 86, 1, 20),
                                             (1500, 170, 5, 4), (1100, 171, 500, 4), (2050, 171, 0, 20), (3000, 86, 129, 7),
                                             (1024, 256, 257, 4), (1030, 257, 511, 4), (16383, 65, 100, 4)])
def test_sw_cut_narrow(ctx, n1, strips, rem, k):
    n2 = strips * 512 - rem
    rng = np.random.default_rng(n1 + n2)
    a, b = rng.integers(0, k, n1, dtype=np.int32), rng.integers(0, k, n2, dtype=np.int32)
    a[:k] = np.arange(k)
    at = n2 // 2 - n1 // 2  # an alignment of all columns around the middle row, across the cut
    b[at:at + n1] = a
    want = O.blocked("SW", a, b, threads=8)
    for nm in ((False, True) if k == 4 else (False,)):
        parts = 3 if nm else 4
        if n1 < 1024:
            parts = 1
        elif parts * strips > 256 and not (nm and 3 * strips <= 512):
            parts = parts - 1 if (parts - 1) * strips <= 512 else 1
        p = ctx.plan([Job("SW", a, b, no_max=nm)])
        print(f"  {n1}x{n2} k={k} no_max={nm} parts={parts}", flush=True)
        assert p.describe()["tasks"] == parts * strips
        for per_pair in (False, False, True):
            p.run(per_pair=per_pair)
            r = p.results()[0]
            assert (r.status, r.last, r.max_score) == (0, want[0], -1 if nm else want[1])
        p.close()
