"""A batch's slots beyond one candidate's life: what a slot's next candidate finds in it."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("integer", [False, True])
def test_a_taken_slot_is_free_of_its_last_candidates_carries(gfe, integer):
    """Timed rounds square a slot whose candidate only waits for its read-back and leave carries
    pending in it; the candidate that takes the slot next starts from 1 all the same."""
    n, iters = 20, 64
    first, second = 1600000, 150000
    want = gfe.run_batch(n, [second], iters=iters)[0]
    bt = gfe.Batch(n, 1)
    if integer:
        bt.set_plan(bt.get_plan())
    seen = 0
    for _ in range(6):
        assert bt.submit(first, iters, 1) == 0
        bt.step()                     # the squarings
        bt.step()                     # the read-back, 4 MiB, is on its way
        if bt.active():
            seen += 1
            bt.time_rounds(3)
        while bt.active():
            bt.step()
        bt.poll()
        assert bt.submit(second, iters, 2) == 0
        while bt.active():
            bt.step()
        got = bt.poll()[0]
        for k in ("res64", "old64", "hash64"):
            assert got[k] == want[k], (k, got, want)
    assert seen, "no read-back was pending when the rounds were timed"
    bt.close()
