"""Single LCS and ED pairs of more than 32 symbols at sizes for which the shipped
autotune table names the bit-parallel engine, which takes at most 32."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prob,n1,n2,k", [("LCS", 2100, 4096, 33), ("LCS", 700, 32768, 200), ("ED", 900, 16384, 33),
                                          ("ED", 3001, 20011, 256)])
def test_large_alphabet_pairs(ctx, prob, n1, n2, k):
    rng = np.random.default_rng(n1 + n2)
    a, b = rng.integers(0, k, n1, dtype=np.int32), rng.integers(0, k, n2, dtype=np.int32)
    a[:k] = np.arange(k)
    print(f"  {prob} {n1}x{n2} {k} symbols", flush=True)
    r = ctx.align(prob, a, b)
    assert (r.status, r.last) == (0, O.score(prob, a, b)[0])
