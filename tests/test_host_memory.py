"""Device memory that the host code asks for, on a HIP runtime without a GPU."""
import ctypes as C

import pytest

from gpumemefficient_amd import _lib

# (n1, n2): narrow, wide and square tables.
TABLES = [(1, 4_000_000), (13, 1_000_000), (100, 100_000), (511, 60_000), (512, 60_000), (600, 50_000), (4096, 65_536),
          (32_768, 32_768), (1_000_000, 6_000), (13_990_000, 4_900)]


@pytest.mark.parametrize("op", ["SAT", "SOR"])
@pytest.mark.parametrize("n1,n2", TABLES)
def test_sweep_memory_is_a_boundary_row_per_256_rows(fake, op, n1, n2):
    """A sweep keeps no more beside the table than a word a column for every 256
    rows, or 8 MiB, so that a table near the device's memory still runs."""
    lib = fake.c
    ctx, table = C.c_void_p(), C.c_void_p()
    assert lib.wf_ctx_create(0, C.byref(ctx)) == 0
    ld = (n1 + 6) // 4 * 4
    lib.fake_set_memory(1 << 40)
    assert lib.hipMalloc(C.byref(table), (n2 + 2) * ld * 4) == 0
    room = max((-(-n2 // 256) - 1) * (n1 + 1) * 8, 8 << 20) + 4096  # and a few small buffers
    lib.fake_set_memory(room)
    out = _lib.wf_result()
    st = lib.wf_stencil_device(ctx, _lib.STENCILS[op], n1, n2, table, ld, None, C.byref(out))
    lib.hipFree(table)
    lib.wf_ctx_destroy(ctx)
    lib.fake_set_memory(1 << 40)
    assert st == _lib.WF_OK
