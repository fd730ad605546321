"""The tiled summed-area table (wf_sat.hip): tiles of 128 rows x 512 columns,
16 rows a wave, 4-column vectors.  Every cell of the table, its boundary and
its padding columns, bit-exact (int32 wrapping mod 2^32) against the oracle's
row-major sweep at sizes around those edges and with many tiles each way."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = ([(n1, 40) for n1 in (1, 2, 3, 4, 5, 508, 509, 510, 511, 512, 513, 514, 515, 1022, 1023, 1024, 1025)]
          + [(600, n2) for n2 in (1, 15, 16, 17, 112, 127, 128, 129, 143, 144, 145, 255, 256, 257)]
          + [(9000, 130), (40000, 3), (3, 9000), (520, 5000), (4100, 1300)])


@pytest.mark.parametrize("pad", [0, 8])
@pytest.mark.parametrize("n1,n2", SHAPES)
def test_sat_tiles_match_oracle(ctx, n1, n2, pad):
    from gpumemefficient_amd._hip import DeviceBuffer
    ld = (n1 + 6) // 4 * 4 + pad
    rng = np.random.default_rng(n1 * 131 + n2)
    host = rng.integers(-2 ** 31, 2 ** 31, size=(n2 + 2, ld), dtype=np.int64).astype(np.int32)
    dev = DeviceBuffer.from_array(host)
    r = ctx.stencil_device("SAT", dev.ptr, n1, n2, ld)
    got = dev.to_array()
    dev.free()
    want = host.copy()
    want[:, :n1 + 3] = O.stencil("SAT", np.ascontiguousarray(host[:, :n1 + 3]))
    assert r.status == 0 and r.last == want[n2, n1]
    bad = np.argwhere(got != want)
    assert bad.size == 0, (bad.shape[0], tuple(bad[0]))
