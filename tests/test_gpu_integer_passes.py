"""The integer passes where engines and batches square in doubles unless a plan is set: the
single-workgroup squaring in batches and mixed batches, proofs' powers, and a long run of the fused
limb plan, each on a plan set by hand and against the reference's fixtures or the passes in doubles."""
import json
import os

import pytest

from test_gpu_golden import canonical_sha256, golden, h

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))


def run(bt, cands, iters):
    for i, (n, b) in enumerate(cands):
        assert bt.submit(b, iters[i] if isinstance(iters, list) else iters, i, n=n) == i
    got = {}
    while len(got) < len(cands):
        bt.step()
        got.update((r["tag"], r) for r in bt.poll())
    bt.close()
    return [got[i] for i in range(len(cands))]


@pytest.mark.parametrize("n,count", [(12, 40), (13, 160)])
def test_single_workgroup_squaring_by_occupancy(gfe, n, count):
    """At n = 13 blocks of 128 or more active slots run it and blocks of fewer the four-step passes; at
    n = 12 every block runs it."""
    from genefer22_amd import workloads
    bases = workloads.seeded_bases(1300 + n, 1024, 2_000_000_000, count)
    iters = [200 + 3 * i for i in range(count)]
    bt = gfe.Batch(n, count)
    assert bt.get_plan()[5] & 16
    bt.set_plan(bt.get_plan())
    assert "in doubles" not in bt.info()
    got = run(bt, [(n, b) for b in bases], iters)
    want = run(gfe.Batch(n, count), [(n, b) for b in bases], iters)
    for b, g, w in zip(bases, got, want):
        assert (g["res64"], g["old64"], g["hash64"]) == (w["res64"], w["old64"], w["hash64"]), b


@pytest.mark.parametrize("few", [False, True])
def test_mixed_batch(gfe, few):
    """128 or more active slots of n = 13 beside slots of n = 12 in one launch; fewer on the four-step
    passes after it."""
    big, small = (5, 7) if few else (130, 10)
    cands = [(13, 1000000 + 14000000 * (k % 3) + 2 * k) for k in range(big)] + [(12, 5000000 + 2 * k) for k in range(small)]
    bt = gfe.Batch(13, len(cands), mixed=True)
    bt.set_plan(bt.get_plan()[:5] + (24,))
    assert "in doubles" not in bt.info()
    got = run(bt, cands, 256)
    want = run(gfe.Batch(13, len(cands), mixed=True), cands, 256)
    for c, g, w in zip(cands, got, want):
        assert (g["res64"], g["old64"], g["hash64"]) == (w["res64"], w["old64"], w["hash64"]), c


def test_full_tests_in_a_mixed_batch(gfe):
    rs = golden("ref_c1.json")[:3]
    bt = gfe.Batch(13, len(rs) + 1, mixed=True)
    bt.set_plan(bt.get_plan()[:5] + (24,))
    got = run(bt, [(12, r["b"]) for r in rs] + [(13, 1000000)], 0)
    for r, g in zip(rs, got):
        assert (h(g["res64"]), h(g["old64"]), g["gl_ok"]) == (r["res64"], r["old64"], 1), r["b"]
    assert (got[-1]["res64"], got[-1]["gl_ok"]) == (gfe.run_quick(1000000, 13)["res64"], 1)


def test_proofs_powers(gfe):
    """Squaring and multiplying rounds with the multiplicand in the integer passes' form."""
    fx = json.load(open(os.path.join(HERE, "golden", "pl_n12.json")))
    want = fx["proofs"]["3"]
    bt = gfe.Batch(fx["n"], 2, depth=3)
    bt.set_plan(bt.get_plan())
    for r in run(bt, [(fx["n"], fx["b"])] * 2, 0):
        assert (h(r["res64"]), h(r["old64"]), r["gl_ok"]) == (fx["res64"], fx["old64"], 1)
        assert [h(x) for x in r["mu_hash64"]] == want["mu_hash64"] and h(r["pkey"]) == want["pkey"]


def test_fused_limb_plan_at_the_top_of_its_range(gfe):
    """b = 35,000,000 at n = 22, where the limb CRT has the least slack: RES64 at every 2000th of the
    first 20,000 squarings, and the whole canonical residue there (SHA-256)."""
    for r in golden("ref_c4max.json"):
        b, n = r["b"], 22
        E = b  # the top bits of b^(2^n), 256 more than are used
        for _ in range(n):
            E *= E
            E >>= max(0, E.bit_length() - r["iters"] - 256)
        bits = [int(c) for c in bin(E)[2:2 + r["iters"]]]
        t = gfe.Transform(b, n)
        t.set_plan(t.get_plan())
        assert t.get_plan()[5] == 42 and "in doubles" not in t.info()
        t.set(1)
        for k in range(0, r["iters"], r["every"]):
            for bit in bits[k:k + r["every"]]:
                t.square_dup(bit)
            assert h(t.residue()["res64"]) == r["res64"][k // r["every"]], (b, k)
        assert canonical_sha256(gfe, t.get_digits(), n, b) == r["sha256"]
        t.close()
