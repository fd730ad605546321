"""SAT and SOR sweeps whose bottom rows go round their ring several times, back
to back with each other and with the engines that share the context's boundary
rows and launch tags: every cell against the oracle, several turns."""
import numpy as np
import pytest

import oracle as O
from gpumemefficient_amd import Context

pytestmark = pytest.mark.gpu


def _sweep(c, op, n1, n2, seed):
    from gpumemefficient_amd._hip import DeviceBuffer
    ld = (n1 + 6) // 4 * 4
    host = np.random.default_rng(seed).integers(-2 ** 31, 2 ** 31, size=(n2 + 2, ld), dtype=np.int64).astype(np.int32)
    dev = DeviceBuffer.from_array(host)
    print(f"  {op} {n1}x{n2}", flush=True)
    r = c.stencil_device(op, dev.ptr, n1, n2, ld)
    got = dev.to_array()
    dev.free()
    want = host.copy()
    want[:, :n1 + 3] = O.stencil(op, np.ascontiguousarray(host[:, :n1 + 3]))
    assert r.status == 0 and r.last == want[n2, n1]
    bad = np.argwhere(got != want)
    assert bad.size == 0, (op, n1, n2, bad.shape[0], tuple(bad[0]))


# More tile rows (strips) than the ring has: of one tile column with several
# turns, of four, of many with a ring of a few rows.
@pytest.mark.parametrize("op", ["SAT", "SOR"])
@pytest.mark.parametrize("n1,n2", [(1, 600_000), (7, 270_000), (2040, 60_000), (60_000, 2100)])
def test_ring_turns(ctx, op, n1, n2):
    _sweep(ctx, op, n1, n2, n1 + n2)


def test_sweeps_and_pairs_take_turns():
    rng = np.random.default_rng(3)
    a, b = rng.integers(0, 4, 2100, dtype=np.int32), rng.integers(0, 4, 2600, dtype=np.int32)
    want = O.score("SW", a, b)
    table = O.table("LCS", a[:600], b[:1500])[1:, 1:]
    with Context(0) as c:
        for turn in range(3):
            for n1, n2 in ((300, 6000), (1500, 2500), (20, 4000)):
                for op in ("SAT", "SOR"):
                    _sweep(c, op, n1, n2, turn)
                r = c.align("SW", a, b)
                assert (r.last, r.max_score) == tuple(want)
                _, t = c.align_table("LCS", a[:600], b[:1500])
                assert np.array_equal(t, table)


@pytest.mark.parametrize("op,n1,n2", [("SAT", 9000, 4000), ("SOR", 100, 0)])
def test_workgroups_claim_more_than_once(ctx, op, n1, n2):
    """More tiles (strips) than the launch has workgroups, so that some claim a
    second one."""
    from gpumemefficient_amd import _lib
    lib, cus = _lib.load(), ctx.info()["compute_units"]
    if op == "SAT":
        assert -(-n2 // 128) * -(-(n1 + 1) // 512) > lib.wf_sat_resident(cus)
    else:
        n2 = 64 * (lib.wf_stencil_resident(cus) + 300) + 7
    _sweep(ctx, op, n1, n2, 11)
