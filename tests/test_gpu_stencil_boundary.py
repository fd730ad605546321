"""The boundary of a SAT or SOR table (row 0, row n2 + 1, columns 0, n1 + 1,
n1 + 2 and the padding) is never written, not with the same values either:
a sweep whose waits are given up (a limit of no time at all, so every tile and
strip below the first ones runs on with values that are not there yet) leaves
all of it as it was, and reports the timeout."""
import numpy as np
import pytest

from gpumemefficient_amd import Context, WfError, _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n1,n2", [(3, 9000), (600, 8000), (2045, 7000)])
@pytest.mark.parametrize("op", ["SAT", "SOR"])
def test_a_sweep_given_up_leaves_the_boundary(op, n1, n2):
    from gpumemefficient_amd._hip import DeviceBuffer
    ld = (n1 + 6) // 4 * 4
    host = np.random.default_rng(n1).integers(1, 2 ** 31, size=(n2 + 2, ld), dtype=np.int64).astype(np.int32)
    dev = DeviceBuffer.from_array(host)
    print(f"  {op} {n1}x{n2}", flush=True)
    with Context(0, timeout_s=1e-9) as c:
        with pytest.raises(WfError) as e:
            c.stencil_device(op, dev.ptr, n1, n2, ld)
    assert e.value.status == _lib.WF_ERR_TIMEOUT
    got = dev.to_array()
    dev.free()
    got[1:n2 + 1, 1:n1 + 1] = host[1:n2 + 1, 1:n1 + 1]
    bad = np.argwhere(got != host)
    assert bad.size == 0, (bad.shape[0], tuple(bad[0]))
