"""The slot server's memory and scheduling, on a HIP runtime without a GPU."""
import time

import pytest

from fake_device import pair
from gpumemefficient_amd import _lib

OK = _lib.WF_OK


def _rows(n1, n2):
    return (-(-n2 // 512) - 1) * n1 * 8


def test_outgrown_arenas_count_against_the_budget(fake):
    """Memory that a slot has outgrown waits to be freed while another slot runs.
    It is part of the budget and of the statistics: a request for which it leaves
    no room waits for it to be freed."""
    lib = fake.c
    sizes = [(900, 20_000), (900, 30_000), (900, 40_000)]  # unsplit, each growing its slot
    outgrown = _rows(*sizes[0]) + _rows(*sizes[1])
    budget = 10 * outgrown
    srv = fake.server(streams=2, hbm_budget=budget)
    lib.fake_hold(1)
    fake.submit(srv, pair("SW", 300, 200))  # runs until it is released
    while fake.stats(srv).launches < 1:
        pass
    lib.fake_hold(0)
    for n1, n2 in sizes:
        fake.submit(srv, pair("SW", n1, n2))
        assert fake.done(srv, 1) == [OK]
    held = lib.fake_live()
    assert outgrown <= fake.stats(srv).hbm_used <= 2 * outgrown
    # All of the budget but half of what is outgrown.
    fake.submit(srv, pair("SW", 900, 512 * ((budget - outgrown // 2) // (900 * 8 + 520))))
    time.sleep(0.05)
    st = fake.stats(srv)
    assert st.pending == 1 and st.launches == 4
    lib.fake_release()
    assert fake.done(srv, 2) == [OK, OK]
    assert lib.wf_server_wait_idle(srv, 20.0) == OK
    assert fake.stats(srv).hbm_used == 0
    assert lib.fake_live() - held < budget - outgrown // 2
    lib.wf_server_destroy(srv)


def _launched(fake, srv, job):
    """Tasks of the launch that runs `job`, and hbm_used meanwhile."""
    lib = fake.c
    lib.fake_hold(1)
    lib.fake_tasks()
    before = fake.stats(srv).launches
    fake.submit(srv, job)
    end = time.monotonic() + 20
    while fake.stats(srv).launches == before and time.monotonic() < end:
        time.sleep(0.0005)
    tasks, used = lib.fake_tasks(), fake.stats(srv).hbm_used
    lib.fake_hold(0)
    lib.fake_release()
    assert fake.done(srv, 1) == [OK]
    assert lib.wf_server_wait_idle(srv, 20.0) == OK
    assert fake.stats(srv).hbm_used == 0
    return tasks, used


@pytest.mark.parametrize("n1,n2", [(64_001, 1001), (3000, 2000)])
def test_a_split_that_the_budget_has_no_room_for_is_left_out(fake, n1, n2):
    """The rows that a column split needs beyond the pair's own are part of the
    budget: charged while it runs, and without room for them the pair runs
    unsplit (a long one too, which has a launch of its own)."""
    job, strips, own = pair("SW", n1, n2), -(-n2 // 512), _rows(n1, n2) + n1 + n2
    for budget, parts in ((16 * own, 4), (own + 2000, 1)):
        srv = fake.server(streams=2, hbm_budget=budget)
        tasks, used = _launched(fake, srv, job)
        assert tasks == parts * strips
        assert own <= used <= budget
        assert used > 1.4 * own or parts == 1
        fake.c.wf_server_destroy(srv)


def test_long_bit_parallel_requests_are_charged_once(fake):
    """The rows of LCS and ED requests are a sixteenth of what they are charged,
    so a split of theirs charges nothing more."""
    srv = fake.server(streams=2, hbm_budget=1 << 30)
    tasks, used = _launched(fake, srv, pair("ED", 50_000, 10_000))
    assert tasks == 2 * 5
    assert used <= _rows(50_000, 10_000) + 100_000
    fake.c.wf_server_destroy(srv)


def test_completions_do_not_wait_for_outgrown_arenas_to_be_freed(fake):
    """Freeing what slots have outgrown waits for the device: the last launch's
    requests are done before it begins (and count no longer), and nothing is
    admitted until it has ended."""
    lib = fake.c
    srv = fake.server(streams=2, hbm_budget=1 << 30)
    lib.fake_hold(1)
    fake.submit(srv, pair("SW", 300, 200))
    while fake.stats(srv).launches < 1:
        pass
    lib.fake_hold(0)
    for n1, n2 in [(900, 20_000), (900, 40_000)]:
        fake.submit(srv, pair("SW", n1, n2))
        assert fake.done(srv, 1) == [OK]
    assert fake.stats(srv).hbm_used > _rows(900, 20_000)
    lib.fake_free_hold(1)
    lib.fake_release()
    assert fake.done(srv, 1, 5.0) == [OK]
    assert lib.wf_server_wait_idle(srv, 5.0) == OK
    assert fake.stats(srv).hbm_used == 0
    fake.submit(srv, pair("SW", 900, 700))
    time.sleep(0.05)
    assert fake.stats(srv).launches == 3
    lib.fake_free_hold(0)
    assert fake.done(srv, 1) == [OK]
    lib.wf_server_destroy(srv)
