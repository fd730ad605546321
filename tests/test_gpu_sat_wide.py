"""SAT tables wider than a block of 64 tile columns (32768 table columns, column
0 among them): every cell against the oracle with one, two and many blocks, the
last of one tile, of a whole block and of something between; and the time per
cell of a very wide table, which must not grow with the width."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

BLOCK = 64 * 512


@pytest.mark.parametrize("n1,n2", [(BLOCK - 2, 20), (BLOCK - 1, 130), (BLOCK, 130), (BLOCK + 511, 20), (BLOCK + 512, 20),
                                   (2 * BLOCK - 1, 257), (2 * BLOCK, 17), (2 * BLOCK + 9000, 300), (700_001, 40)])
def test_sat_blocks_match_oracle(ctx, n1, n2):
    from gpumemefficient_amd._hip import DeviceBuffer
    ld = (n1 + 6) // 4 * 4
    host = np.random.default_rng(n1 + n2).integers(-2 ** 31, 2 ** 31, size=(n2 + 2, ld), dtype=np.int64).astype(np.int32)
    dev = DeviceBuffer.from_array(host)
    print(f"  SAT {n1}x{n2}", flush=True)
    r = ctx.stencil_device("SAT", dev.ptr, n1, n2, ld)
    got = dev.to_array()
    dev.free()
    want = host.copy()
    want[:, :n1 + 3] = O.stencil("SAT", np.ascontiguousarray(host[:, :n1 + 3]))
    assert r.status == 0 and r.last == want[n2, n1]
    bad = np.argwhere(got != want)
    assert bad.size == 0, (bad.shape[0], tuple(bad[0]))


def test_sat_time_per_cell_does_not_grow_with_the_width(ctx):
    """8 million columns x 128 rows against 32000 x 32768, a billion cells each:
    at most three times (1.2 measured).  Ten times as long where a tile read
    the row sums of every tile to its left."""
    from gpumemefficient_amd._hip import DeviceBuffer
    ms = []
    for n1, n2 in ((32000, 32768), (8_000_000, 128)):
        ld = (n1 + 6) // 4 * 4
        dev = DeviceBuffer((n2 + 2, ld))
        print(f"  SAT {n1}x{n2}", flush=True)
        ms.append(min(ctx.stencil_device("SAT", dev.ptr, n1, n2, ld).kernel_ms for _ in range(4)) / (n1 * n2))
        dev.free()
    assert ms[1] < 3 * ms[0], ms
