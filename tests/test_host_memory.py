"""Device memory that the host code asks for, on a HIP runtime without a GPU."""
import ctypes as C

import numpy as np
import pytest

from fake_device import i32, pair
from gpumemefficient_amd import _lib, _server_abi

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


# (problem, n1, n2, symbols), the bytes that the pair needs unsplit and a little
# more (a column split takes twice the rows, or half the codes again).
SPLIT = [("SW", 20_000, 4000, 4, 7 * 20_000 * 8 + 300_000), ("SW", 20_000, 4000, 20, 7 * 20_000 * 8 + 300_000),
         ("SW", 20_000, 80_000, 4, 156 * 20_000 * 8 + 1_000_000), ("LCS", 2_000_000, 3000, 4, 3_200_000)]


@pytest.mark.parametrize("prob,n1,n2,k,room", SPLIT)
def test_a_split_that_does_not_fit_is_left_out(fake, prob, n1, n2, k, room):
    """A pair whose column split needs more memory than there is runs unsplit: a
    call, a plan and a server's request that the unsplit pair fits succeed."""
    lib = fake.c
    job = pair(prob, n1, n2, k)
    strips = -(-n2 // (512 if prob == "SW" else 2048))
    tasks = C.c_int64()
    for memory in (1 << 40, room):
        ctx = C.c_void_p()
        assert lib.wf_ctx_create(0, C.byref(ctx)) == 0
        lib.fake_set_memory(memory)
        out = _lib.wf_result()
        lib.fake_tasks()
        assert lib.wf_align_batch(ctx, fake.jobs([job]), 1, None, C.byref(out)) == _lib.WF_OK
        n = lib.fake_tasks()
        assert n == strips if memory == room else n > strips
        lib.wf_ctx_destroy(ctx)
        h = C.c_void_p()
        assert lib.wf_plan_create(fake.ctx, fake.jobs([job]), 1, None, C.byref(h)) == _lib.WF_OK
        lib.wf_plan_describe(h, None, None, None, None, C.byref(tasks), None)
        assert tasks.value == n
        lib.wf_plan_destroy(h)
        opts = _server_abi.wf_server_opts(hbm_budget=1 << 30)
        srv = C.c_void_p()
        assert lib.wf_server_create(0, C.byref(opts), C.byref(srv)) == 0
        assert lib.wf_server_submit(srv, fake.jobs([job]), None) == 0
        assert lib.wf_server_wait_idle(srv, 20.0) == 0
        done, got = (_server_abi.wf_completion * 1)(), C.c_int()
        assert lib.wf_server_poll(srv, done, 1, C.byref(got)) == 0
        lib.wf_server_destroy(srv)
        assert got.value == 1 and done[0].status == _lib.WF_OK
    lib.fake_set_memory(1 << 40)


@pytest.mark.parametrize("prob", ["ED", "LCS"])
def test_noalloc_takes_the_longest_pairs(fake, prob):
    """Pairs up to the size whose codes, and those of a half of their columns
    again, fill the 8 MiB of the scratch area: a half cut along a staircase is
    longer, and then the pair runs unsplit."""
    lib, n2 = fake.c, 2049

    def small(n1):  # descriptors, last columns, codes of a pair cut at its middle
        codes = sum((x + 15) // 16 * 16 for x in (n1, n2, n1 - n1 // 2, n2))
        return 256 * 6 + 2 * 2 * 64 * 8 + (codes + 255) // 256 * 256

    n1 = 5_000_000
    while small(n1 + 1) <= 8 << 20:
        n1 += 1
    for n in (n1, n1 - 1500, 4000):
        _, a, b, _ = pair(prob, n, n2)
        out = _lib.wf_result()
        st = lib.wf_align_noalloc(fake.ctx, _lib.PROBLEMS[prob], i32(a), a.size, i32(b), b.size, None, C.byref(out))
        assert st == _lib.WF_OK, n
    # (8 MiB of codes never fit.)
    a = np.zeros(8 << 20, np.int32)
    st = lib.wf_align_noalloc(fake.ctx, _lib.PROBLEMS[prob], i32(a), a.size, i32(b), b.size, None, C.byref(out))
    assert st == _lib.WF_ERR_SCRATCH
