"""Plans and launches of the host code, on a HIP runtime without a GPU."""
import pytest

from fake_device import pair
from gpumemefficient_amd import _lib


@pytest.mark.parametrize("prob,n1,n2,k,parts", [("SW", 7013, 3001, 20, 4), ("SW", 7013, 3001, 7, 4),
                                                ("SW", 3000, 2000, 4, 4), ("SW", 65536, 65536, 4, 3),
                                                ("ED", 640, 640, 20, 2), ("LCS", 4000, 5000, 4, 2)])
def test_a_pairs_parts_share_its_launch(fake, prob, n1, n2, k, parts):
    """One launch per pair runs all parts of a column-split pair: in a launch each
    they would run one after another (7013 x 3001 then took twice the time of the
    unsplit pair)."""
    jobs = [pair(prob, n1, n2, k), pair(prob, 300, 200, k, 1)]
    for todo in (jobs[:1], jobs):
        st, plan, tasks = fake.plan(todo)
        assert st == 0
        if len(todo) == 1:
            assert tasks == parts * -(-n2 // (512 if prob == "SW" else 2048))
        fake.c.fake_tasks()
        before = fake.c.fake_launches()
        assert fake.c.wf_plan_run(plan, _lib.WF_RUN_PER_PAIR) == 0
        assert fake.c.fake_launches() - before == len(todo)
        assert fake.c.fake_tasks() == tasks
        assert fake.c.wf_plan_run(plan, _lib.WF_RUN_PERSISTENT) == 0
        assert fake.c.fake_launches() - before == len(todo) + 1
        assert fake.c.fake_tasks() == tasks
        fake.c.wf_plan_destroy(plan)


@pytest.mark.parametrize("prob,n1,n2", [("LCS", 3000, 4096), ("ED", 2000, 20_000), ("ED", 1000, 1000)])
def test_large_alphabets_beside_a_tuned_bit_parallel_entry(fake, tmp_path, prob, n1, n2):
    """A tuned entry is looked up by size: a pair of more symbols than its engine
    takes runs on the built-in choice, as a pair without an entry does."""
    table = tmp_path / "tune.txt"
    table.write_text("none 256 1 single 14 3 32 1 64 1.0\nnone 256 0 single 12 3 32 1 64 0.1\n"
                     "none 256 1 single 9 2 32 1 64 1.0\n")
    job = pair(prob, n1, n2, k=33)
    for _ in range(2):  # without the entries, with them
        st, plan, tasks = fake.plan([job])
        assert st == 0 and tasks == -(-n2 // 512)
        fake.c.wf_plan_destroy(plan)
        assert fake.c.wf_tune_load(str(table).encode()) == 0
    st, plan, tasks = fake.plan([pair(prob, n1, n2, k=32)])
    assert st == 0 and tasks <= 2 * -(-n2 // 2048)
    fake.c.wf_plan_destroy(plan)
    fake.c.wf_tune_clear()
