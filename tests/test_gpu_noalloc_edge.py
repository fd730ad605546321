"""wf_align_noalloc at the largest LCS and ED pairs its scratch area takes, which
run unsplit there: the scores of wf_align, which splits them."""
import ctypes as C

import numpy as np
import pytest

from gpumemefficient_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prob,n1,n2", [("LCS", 5_583_000, 2049), ("ED", 5_583_000, 2049), ("ED", 5_500_000, 3000)])
def test_noalloc_unsplit_equals_split(ctx, prob, n1, n2):
    rng = np.random.default_rng(n1)
    a, b = rng.integers(0, 4, n1, dtype=np.int32), rng.integers(0, 4, n2, dtype=np.int32)
    want = ctx.align(prob, a, b)
    out = _lib.wf_result()
    pa, pb = (x.ctypes.data_as(C.POINTER(C.c_int32)) for x in (a, b))
    print(f"  {prob} {n1}x{n2}", flush=True)
    st = _lib.load().wf_align_noalloc(ctx._h, _lib.PROBLEMS[prob], pa, n1, pb, n2, None, C.byref(out))
    assert st == _lib.WF_OK and out.status == 0 and out.last == want.last
