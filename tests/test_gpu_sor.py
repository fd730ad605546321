"""The SOR sweep's strips (wf_stencil.hip): 64 rows a strip, a window in step
order moved in chunks of 16 steps and turns of 6 chunks, 4-column vectors that
are skewed from row to row.  Every cell of the table, its boundary and its
padding columns, bit-exact against the oracle's row-major sweep at sizes around
those edges, among them pitches of exactly n1 + 3 (the last row's vectors then
reach the table's end)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = ([(n1, 130) for n1 in (1, 2, 3, 4, 5, 13, 16, 17, 18, 31, 33, 34, 35, 36, 37, 49, 65, 81, 93, 97, 98, 129, 130,
                                131, 132, 133, 189, 193, 225, 229)]
          + [(141, n2) for n2 in (1, 2, 62, 63, 64, 65, 66, 127, 128, 129, 191, 192, 193)]
          + [(5001, 67), (3, 3000), (2000, 2049), (1009, 4097)])


@pytest.mark.parametrize("pad", [0, 12])
@pytest.mark.parametrize("n1,n2", SHAPES)
def test_sor_strips_match_oracle(ctx, n1, n2, pad):
    from gpumemefficient_amd._hip import DeviceBuffer
    ld = (n1 + 6) // 4 * 4 + pad
    rng = np.random.default_rng(n1 * 137 + n2)
    host = rng.integers(-2 ** 31, 2 ** 31, size=(n2 + 2, ld), dtype=np.int64).astype(np.int32)
    dev = DeviceBuffer.from_array(host)
    r = ctx.stencil_device("SOR", dev.ptr, n1, n2, ld)
    got = dev.to_array()
    dev.free()
    want = host.copy()
    want[:, :n1 + 3] = O.stencil("SOR", np.ascontiguousarray(host[:, :n1 + 3]))
    assert r.status == 0 and r.last == want[n2, n1]
    bad = np.argwhere(got != want)
    assert bad.size == 0, (bad.shape[0], tuple(bad[0]))


def test_sor_wait_that_runs_out_is_reported():
    """Waits of at most 1 us: the strips below the first give up, the launch
    drains and reports the time-out; the next sweep is exact."""
    from gpumemefficient_amd import Context, WfError, _lib
    t = np.random.default_rng(9).integers(0, 1000, size=(602, 903), dtype=np.int32)
    with Context(0, timeout_s=1e-6) as c:
        with pytest.raises(WfError) as e:
            c.stencil("SOR", t)
        assert e.value.status == _lib.WF_ERR_TIMEOUT
    with Context(0, timeout_s=20.0) as c:
        assert np.array_equal(c.stencil("SOR", t)[1], O.stencil("SOR", t))
