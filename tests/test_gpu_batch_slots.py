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


@pytest.mark.parametrize("n,count", [(12, 3), (15, 2)])
def test_the_tuner_finds_the_way_back_to_doubles(gfe, n, count):
    """After gfe_batch_set_plan too the tuner times the double-precision transform beside the integer
    plans (it takes half their time at these sizes)."""
    bases = [50000000 + 2 * i for i in range(count)]
    want = [r["res64"] for r in gfe.run_batch(n, bases, iters=300)]
    bt = gfe.Batch(n, count)
    bt.set_plan(bt.get_plan())
    for i, b in enumerate(bases):
        bt.submit(b, 300, i)
    bt.step()
    assert "in doubles" not in bt.info()
    bt.tune(1)
    assert "in doubles" in bt.info()
    got = {}
    while len(got) < count:
        bt.step()
        got.update((r["tag"], r["res64"]) for r in bt.poll())
    bt.close()
    assert [got[i] for i in range(count)] == want


@pytest.mark.parametrize("plan_at", [None, 0, 1])
@pytest.mark.parametrize("at", [10, 17, 24, 31])
def test_tuning_during_a_proofs_powers(gfe, plan_at, at):
    """gfe_batch_tune while power runs hold a multiplicand, in doubles (plan_at None, or the integer
    passes selected just before it: 1) or in the integer passes' form (selected at the start: 0): the
    plans are timed in their own passes, doubles are found to be faster, and the runs under way end in
    the transform that holds their multiplicand."""
    b, n, depth = 1026, 12, 3
    want = gfe.run_proof(b, n, depth)
    bt = gfe.Batch(n, 2, depth=depth)
    if plan_at == 0:
        bt.set_plan(bt.get_plan())
    for tag in (0, 1):
        bt.submit(b, 0, tag)
    got, steps, prp = [], 0, want["esize"] // 64
    while len(got) < 2:
        bt.step()
        steps += 1
        if steps == prp + at:
            if plan_at == 1:
                bt.set_plan(bt.get_plan())
            bt.tune(1)
            assert "in doubles" in bt.info()
        got += bt.poll()
    assert steps > prp + at
    bt.close()
    for r in got:
        assert (r["res64"], r["pkey"], r["mu_hash64"], r["gl_ok"]) == (want["res64"], want["pkey"], want["mu_hash64"], 1)
