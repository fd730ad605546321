"""The slot server's memory and scheduling, on a HIP runtime without a GPU."""
import time

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
