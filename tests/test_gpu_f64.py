"""The double-precision limb transform (what an engine squares with unless gfe_set_plan selects the
integer passes) against the oracle, and its digits against the integer passes' own: at every n's
shape, at the bases where the prime count, the limb conversion or the rule changes, from extreme
digits, and through every use of the registers that has to apply its pending carries."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def canon(O, d, n, b):
    return O.unbalance(d, n, b)


def largest_two_prime_base(n):
    from test_f64 import bound
    lo, hi = 1 << 17, 1 << 25
    while hi - lo > 1:
        m = (lo + hi) // 2
        lo, hi = (m, hi) if bound(m, n, 2) else (lo, m)
    return lo


@pytest.mark.parametrize("n", range(12, 24))
def test_digits_equal_the_integer_passes(gfe, n):
    """Random and extreme digits, doubled or not: the digits read back are those of the integer
    passes, bit for bit, at the edges of the two- and three-prime ranges."""
    e = largest_two_prime_base(n)
    bases = [{21: 1148, 22: 1622, 23: 2292}.get(n, 1026), e - (e & 1), e + 2 - (e & 1), 15300000, 31987654, 32200000, 1999999998]
    for b in bases if n <= 17 else bases[::2]:
        t, u = gfe.Transform(b, n), gfe.Transform(b, n)
        u.set_plan(u.get_plan())
        assert "in doubles" in t.info() and "in doubles" not in u.info()
        rs = np.random.RandomState(n)
        N, h = 1 << n, b // 2 + 4
        for d in (rs.randint(-((b - 1) // 2), b // 2 + 1, N), np.full(N, -h), np.where(np.arange(N) % 2 == 0, h, -h)):
            for x in (t, u):
                x.set_digits(d.astype(np.int32))
                for dup in (1, 0, 1, 1):
                    x.square_dup(dup)
            got = t.get_digits()
            assert np.abs(got.astype(np.int64)).max() <= h
            assert np.array_equal(got, u.get_digits()), (b, n)
        t.close()
        u.close()


@pytest.mark.parametrize("b,n", [(1026, 12), (146950, 12), (1999999998, 12), (777777778, 13), (1999999266, 14),
                                 (1619951882, 15), (333333334, 17)])
def test_every_use_of_the_registers_matches_the_oracle(gfe, oracle, b, n):
    rs = np.random.RandomState(n)
    t, o = gfe.Transform(b, n), oracle.Engine(b, n)
    t.set(3); o.set(3)
    a = oracle.balance(rs.randint(0, b, 1 << n).astype(np.int32), n, b)
    t.set_digits(a, 1); o.set_digits(a, 1)
    for k in range(6):
        t.square_dup(k & 1); o.square_dup(k & 1)
    t.init_multiplicand(0); o.init_multiplicand(0)      # of register 0, its carries pending
    t.square_dup(True); o.square_dup(True)
    t.mul(); o.mul()
    t.copy(2, 0); o.copy(2, 0)
    t.mul(1); o.mul(1)                                   # another multiplicand
    t.square_mul(7); o.square_mul(7)
    plan = t.get_plan()
    t.square_dup(False); o.square_dup(False)
    t.set_plan(plan)                                     # the integer passes, carries pending
    t.square_dup(True); o.square_dup(True)
    t.mul(); o.mul()                                     # the multiplicand of the other transform
    t.rebase(b)                                          # back to doubles
    t.square_dup(False); o.square_dup(False)
    data = t.save_context(3)
    for r in (0, 1, 2):
        assert np.array_equal(canon(oracle, t.get_digits(r), n, b), canon(oracle, o.get_digits(r), n, b)), r
    u = gfe.Transform(b, n)
    assert u.read_context(data, 3)
    assert np.array_equal(canon(oracle, u.get_digits(0), n, b), canon(oracle, o.get_digits(0), n, b))
    t.time_squarings(3, 0b101)
    t.time_squarings(2, 0b1, per_kernel=True)
    for dup in (1, 0, 1, 1, 0, 0):
        o.square_dup(dup)
    assert np.array_equal(canon(oracle, t.get_digits(0), n, b), canon(oracle, o.get_digits(0), n, b))


def test_refused_bases_keep_the_integer_passes(gfe, oracle):
    """b = 1024 at n = 23 is outside the rule (the last piece may exceed the limb's size)."""
    n, b = 23, 1026
    t, o = gfe.Transform(b, n), oracle.Engine(b, n)
    assert "in doubles" not in t.info()
    d = np.full(1 << n, b // 2, dtype=np.int32)
    t.set_digits(d); o.set_digits(d, 0)
    t.square_dup(True); o.square_dup(True)
    assert np.array_equal(canon(oracle, t.get_digits(), n, b), canon(oracle, o.get_digits(0), n, b))


def run_batch(gfe, n, bases, iters, integer=False, graphs=True, mixed=False):
    bt = gfe.Batch(n, len(bases), mixed=mixed)
    assert "in doubles" in bt.info()
    bt.set_graphs(graphs)
    if integer:
        bt.set_plan(bt.get_plan()[:5] + (24,) if mixed else bt.get_plan())
        assert "in doubles" not in bt.info()
    for i, b in enumerate(bases):
        assert bt.submit(b, iters + 3 * i, i, n=12 + i % 2 if mixed else None) is not None
    got = []
    while len(got) < len(bases):
        bt.step()
        got += bt.poll()
    bt.close()
    return sorted((r["tag"], r["res64"], r["old64"], r["hash64"]) for r in got)


@pytest.mark.parametrize("n,count", [(12, 9), (12, 8), (12, 223), (12, 224), (13, 15), (13, 225), (14, 3), (14, 64), (14, 65),
                                     (15, 7), (17, 8), (18, 5), (19, 2), (20, 1)])
def test_batches_equal_the_integer_passes(gfe, n, count):
    """Slots spread over the XCDs or pinned to one each, two and three primes side by side, the primes one
    after the other in the column passes (past 2^19 limbs) and side by side, a slot's squaring in one
    workgroup (from 224 slots) or one a prime, slots that end rounds before others, graphs and single launches."""
    e = largest_two_prime_base(n)
    bases = [(1026, 1999999898, e & ~1, (e & ~1) + 2, 146950, 20204692)[i % 6] + 2 * (i // 6) for i in range(count)]
    want = run_batch(gfe, n, bases, 70, integer=True)
    assert run_batch(gfe, n, bases, 70) == want
    assert run_batch(gfe, n, bases, 70, graphs=False) == want


def test_mixed_batch_equals_the_integer_passes(gfe):
    bases = [1026, 1999999998, 146950, 20204692, 50000000, 4098, 999999618]
    assert run_batch(gfe, 13, bases, 70, mixed=True) == run_batch(gfe, 13, bases, 70, mixed=True, integer=True)


@pytest.mark.parametrize("at", [10, 17, 24, 31])
def test_plan_change_during_a_proofs_powers(gfe, at):
    """gfe_batch_set_plan while power runs hold their multiplicand in doubles: those runs end in
    doubles, what follows is in the integer passes, and the proof is the same."""
    b, n, depth = 1026, 12, 3
    want = gfe.run_proof(b, n, depth)
    bt = gfe.Batch(n, 2, depth=depth)
    for tag in (0, 1):
        bt.submit(b, 0, tag)
    got, steps, prp = [], 0, want["esize"] // 64
    while len(got) < 2:
        bt.step()
        steps += 1
        if steps == prp + at:
            bt.set_plan(bt.get_plan())
        got += bt.poll()
    assert steps > prp + at
    bt.close()
    for r in got:
        assert (r["res64"], r["pkey"], r["mu_hash64"], r["gl_ok"]) == (want["res64"], want["pkey"], want["mu_hash64"], 1)


@pytest.mark.parametrize("b,n", [(1026, 12), (1999999998, 13), (15300000, 14), (1999999998, 16)])
def test_noalloc_digits_equal_the_engines(gfe, b, n):
    """gfe_square_noalloc from extreme digits, one squaring and 65 (the doubling pattern's period and one)."""
    from test_zz_no_alloc import Hip
    h, hip, t = b // 2 + 4, Hip(), gfe.Transform(b, n)
    hip.ck(hip.h.hipSetDevice(0), "hipSetDevice")
    buf, got, dup = hip.malloc(4 << n), np.empty(1 << n, dtype=np.int32), 0x8000000000000003
    try:
        for d in (np.full(1 << n, -h), np.random.RandomState(n).randint(-h, h + 1, 1 << n)):
            for count in (1, 65):
                d = np.ascontiguousarray(d, dtype=np.int32)
                hip.to_device(buf, d)
                rc = gfe.lib().gfe_square_noalloc(b, n, 0, buf, count, dup, None)
                assert rc == 0, gfe.lib().gfe_last_error()
                hip.ck(hip.h.hipDeviceSynchronize(), "hipDeviceSynchronize")
                hip.to_host(got, buf)
                t.set_digits(d)
                for i in range(count):
                    t.square_dup((dup >> (i % 64)) & 1)
                assert np.array_equal(got, t.get_digits()), count
    finally:
        hip.h.hipFree(buf)


@pytest.mark.parametrize("n", range(19, 24))
def test_four_digit_limbs_equal_the_integer_passes(gfe, n):
    """At the edges of the rule of four-digit limbs and past them: extreme and random digits, products,
    copies and a change of base and back (to two-digit limbs between), against the integer passes."""
    from test_f64 import qbound, qedges
    lo, hi = qedges(max(n, 20))
    for b in (lo + (lo & 1), hi - (hi & 1), lo - 2 - (lo & 1), hi + 2 - (hi & 1)):
        t, u = gfe.Transform(b, n), gfe.Transform(b, n)
        u.set_plan(u.get_plan())
        assert ("four digits" in t.info()) == (qbound(b, n) is not None) and "in doubles" not in u.info()
        rs, N, h = np.random.RandomState(n), 1 << n, b // 2 + 4
        d = rs.randint(-((b - 1) // 2), b // 2 + 1, N).astype(np.int32)
        for x in (np.full(N, -h, np.int32), np.where(np.arange(N) % 2 == 0, h, -h).astype(np.int32), d):
            for e in (t, u):
                e.set_digits(x)
                for dup in (1, 0, 1):
                    e.square_dup(dup)
            got = t.get_digits()
            assert np.abs(got.astype(np.int64)).max() <= h
            assert np.array_equal(got, u.get_digits()), (b, n)
        for e in (t, u):
            e.set_digits(d, 1)
            e.init_multiplicand(1)
            e.square_dup(False)
            e.mul()
            e.copy(2, 0)                    # carries pending
            e.init_multiplicand(0)
            e.square_dup(True)
            e.mul()
            e.square_mul(7)
        assert np.array_equal(t.get_digits(0), u.get_digits(0)) and np.array_equal(t.get_digits(2), u.get_digits(2))
        t.rebase(hi + 2 + (hi & 1) if b > 2**25 else lo - 4 - (lo & 1))
        assert "two digits" in t.info()
        t.set(3)
        t.square_dup(True)
        t.rebase(b)
        u.copy(0, 1)
        t.set_digits(d, 0)
        for e in (t, u):
            e.square_dup(True)
        assert np.array_equal(t.get_digits(), u.get_digits())
        t.close()
        u.close()


def test_full_tests_in_a_batch_of_three_passes(gfe):
    """Whole tests at n = 14, with the Gerbicz-Li products (forward passes into the multiplicand and
    products of the active slots only) on slots of two and of three primes that reach them at
    different rounds; the residues are the single engine's."""
    n, e = 14, largest_two_prime_base(14)
    bases = [1026, (e & ~1) + 2, 4098]
    bt = gfe.Batch(n, len(bases))
    for i, b in enumerate(bases):
        assert bt.submit(b, 0, i) == i
    got = {}
    while len(got) < len(bases):
        bt.step()
        got.update((r["tag"], r) for r in bt.poll())
    bt.close()
    for i, b in enumerate(bases):
        w = gfe.run_quick(b, n)
        assert (got[i]["res64"], got[i]["old64"], got[i]["gl_ok"]) == (w["res64"], w["old64"], 1), b


def test_proofs_in_a_batch_of_three_passes(gfe):
    """The powers of a proof at n = 14: rows that square some slots and multiply others."""
    n, depth, bases = 14, 2, [1026, 4098]
    bt = gfe.Batch(n, len(bases), depth=depth)
    for i, b in enumerate(bases):
        assert bt.submit(b, 0, i) == i
    got = {}
    while len(got) < len(bases):
        bt.step()
        got.update((r["tag"], r) for r in bt.poll())
    bt.close()
    for i, b in enumerate(bases):
        w = gfe.run_proof(b, n, depth)
        assert (got[i]["res64"], got[i]["pkey"], got[i]["mu_hash64"], got[i]["gl_ok"]) == (w["res64"], w["pkey"], w["mu_hash64"], 1), b
