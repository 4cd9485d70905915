"""What the squaring engine is timed on: the work that programs have it do through the package's
public entry points, over the range of n and b that the engine accepts (12 <= n <= 23, b up to 2e9).

Kinds of cases (each stands for a caller):

  prp      one candidate on one engine (Transform): a stretch of the PRP loop's squarings, some of
           them doubled as the exponent's bits ask, then the residue's digits read back -- a test
           running between two of its checkpoints, a server's lone request
  power    r0 = r1^e by square-and-multiply (set the multiplicand, then squarings and products):
           the Gerbicz-Li check and the Pietrzak-Li proof
  noalloc  squarings of digits the caller holds in device memory, on the caller's stream, with no
           allocation (gfe_square_noalloc): loops that are captured or must not allocate
  batch    many candidates of one n in shared launches (Batch): submit, step until all are done,
           poll; `mixed` holds candidates of n = 12 and 13 side by side
  request  one truncated test as a whole call (run_prp): engine set-up, squarings, residue

Bases are even, as the tests' candidates are; digits are balanced residues in the middle of a test
(every digit in use).  The seed decides digits, doublings, exponents and a batch's bases.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import genefer22_amd as G


def listed():
    return [
        # the smallest call: a candidate of n = 12 with a small base (two primes of 31 bits in the
        # reference's rule), a short stretch; launches and latency count
        dict(name="prp_n12_short", kind="prp", n=12, b=146950, count=64),
        # an ordinary candidate of n = 15 at the top of the base range, one per engine
        dict(name="prp_n15", kind="prp", n=15, b=1619951882, count=500),
        # an ordinary lone request of the serving mix
        dict(name="prp_n18", kind="prp", n=18, b=541873226, count=500),
        # n = 20 near the top of the serving mix's base range
        dict(name="prp_n20", kind="prp", n=20, b=54129870, count=500),
        # the headline: n = 22, about the range where candidates are being tested
        dict(name="prp_n22", kind="prp", n=22, b=20204692, count=1000),
        # the largest transform, at the small bases that are still untested there
        dict(name="prp_n23", kind="prp", n=23, b=150000, count=500),
        # the products of the Gerbicz-Li check and of proofs
        dict(name="power_n17", kind="power", n=17, b=333333334, count=301),
        # a caller that keeps its digits on the device and allocates nothing
        dict(name="noalloc_n16", kind="noalloc", n=16, b=1433042190, count=333),
        # many small candidates at once, an odd number of them
        dict(name="batch_n12", kind="batch", n=12, cap=301, lo=1024, hi=2_000_000_000, iters=2048, mixed=False),
        # 512 candidates of n = 15, the batched workload the engine is judged by
        dict(name="batch_n15", kind="batch", n=15, cap=512, lo=100_000_000, hi=2_000_000_000, iters=1024, mixed=False),
        # a server's pool of a few large candidates
        dict(name="batch_n18", kind="batch", n=18, cap=7, lo=1024, hi=1_000_000_000, iters=512, mixed=False),
        # a whole call for one truncated test, set-up included
        dict(name="request_n13", kind="request", n=13, b=777777778, iters=4096),
    ]


# largest base a drawn case takes at its n: what is in use there
_B_MAX = {12: 2_000_000_000, 13: 2_000_000_000, 14: 2_000_000_000, 15: 2_000_000_000, 16: 1_500_000_000,
          17: 1_000_000_000, 18: 1_000_000_000, 19: 400_000_000, 20: 150_000_000, 21: 80_000_000,
          22: 35_000_000, 23: 20_000_000}


def _even(rng, lo, hi):
    """An even base in [lo, hi], spread over its logarithm."""
    b = int(math.exp(rng.uniform(math.log(lo), math.log(hi)))) & ~1
    return min(max(b, lo + (lo & 1)), hi & ~1)


def draw(rng):
    kind = rng.choice(["prp", "prp", "prp", "power", "noalloc", "batch", "batch", "mixed", "request"])
    if kind in ("prp", "power"):
        n = rng.randint(12, 23)
        count = max(9, min(rng.randint(64, 600), int(2.0e9 / (1 << n))))
        return dict(kind=kind, n=n, b=_even(rng, 1024, _B_MAX[n]), count=count)
    if kind == "noalloc":
        n = rng.randint(12, 16)
        return dict(kind=kind, n=n, b=_even(rng, 1024, _B_MAX[n]), count=rng.randint(64, 600))
    if kind in ("batch", "mixed"):
        mixed = kind == "mixed"
        n = 13 if mixed else rng.randint(12, 20)
        top = max(2, min(400, (1 << 23) >> n))
        cap = max(1, int(math.exp(rng.uniform(0.0, math.log(top)))))
        lo, hi = sorted((_even(rng, 1024, _B_MAX[n]), _even(rng, 1024, _B_MAX[n])))
        return dict(kind="batch", n=n, cap=cap, lo=lo, hi=max(hi, lo + 64), iters=rng.randint(200, 1000), mixed=mixed)
    n = rng.randint(12, 18)
    return dict(kind="request", n=n, b=_even(rng, 1024, _B_MAX[n]), iters=rng.randint(200, 3000))


def _digits(rs, n, b):
    """A balanced residue in the middle of a test: digits uniform in (-b/2, b/2]."""
    return rs.randint(-((b - 1) // 2), b // 2 + 1, size=1 << n).astype(np.int32)


def _inputs(case, seed):
    rs = np.random.RandomState(seed % (1 << 32))
    kind = case["kind"]
    if kind == "prp":
        return _digits(rs, case["n"], case["b"]), [int(x) for x in rs.randint(0, 2, case["count"])]
    if kind == "power":
        return _digits(rs, case["n"], case["b"]), [1] + [int(x) for x in rs.randint(0, 2, case["count"] - 1)]
    if kind == "noalloc":
        return _digits(rs, case["n"], case["b"]), int(rs.randint(0, 1 << 32, dtype=np.int64)) << 32 | int(
            rs.randint(0, 1 << 32, dtype=np.int64))
    if kind == "batch":
        half = (case["hi"] - case["lo"]) // 2
        out = []
        for i, x in enumerate(rs.randint(0, half, size=4 * case["cap"])):
            b = case["lo"] + 2 * int(x)
            if b & (b - 1):
                out.append((12 + (i & 1) if case["mixed"] else case["n"], b))
        return out[:case["cap"]]
    # a request: another base near the case's, of the same prime set
    return case["b"] - 2 * int(rs.randint(0, max(1, case["b"] // 200)))


def prepare(case, seed):
    inp = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("prp", "power"):
        digits, bits = inp
        t = G.Transform(case["b"], case["n"], num_regs=3)
        t.set_digits(digits, 1)  # register 1: the residue a pass starts from
        return dict(kind=kind, t=t, bits=bits)
    if kind == "noalloc":
        digits, dup = inp
        dev = torch.device("cuda", 0)
        return dict(kind=kind, b=case["b"], n=case["n"], count=case["count"], dup=dup, stream=torch.cuda.Stream(dev),
                    start=torch.from_numpy(digits).to(dev))
    if kind == "batch":
        return dict(kind=kind, bt=G.Batch(case["n"], case["cap"], mixed=case["mixed"]), cands=inp, iters=case["iters"],
                    mixed=case["mixed"])
    return dict(kind=kind, b=max(inp, 1024), n=case["n"], iters=case["iters"])


def run(state):
    kind = state["kind"]
    if kind == "prp":
        t = state["t"]
        t.copy(0, 1)
        for bit in state["bits"]:
            t.square_dup(bit)
        return t.get_digits(0)
    if kind == "power":
        t = state["t"]
        t.init_multiplicand(1)
        t.set(1)
        for bit in state["bits"]:
            t.square_dup(False)
            if bit:
                t.mul()
        return t.get_digits(0)
    if kind == "noalloc":
        stream = state["stream"]
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            d = state["start"].clone()
            rc = G.lib().gfe_square_noalloc(state["b"], state["n"], 0, ctypes.c_void_p(d.data_ptr()), state["count"],
                                            state["dup"], ctypes.c_void_p(stream.cuda_stream))
        if rc != 0:
            raise G.GfeError(f"gfe error {rc}: {G.lib().gfe_last_error().decode(errors='replace')}")
        torch.cuda.current_stream().wait_stream(stream)
        d.record_stream(torch.cuda.current_stream())
        return d
    if kind == "batch":
        bt, cands = state["bt"], state["cands"]
        for i, (n, b) in enumerate(cands):
            bt.submit(b, state["iters"], i, n=n if state["mixed"] else None)
        done = []
        while len(done) < len(cands):
            bt.step()
            done += bt.poll()
        done.sort(key=lambda r: r["tag"])
        return [np.array([r[k] for r in done], dtype=np.uint64).view(np.int64)
                for k in ("n", "b", "iters", "res64", "old64", "hash64")]
    r = G.run_prp(state["b"], state["n"], iters=state["iters"], b_gl=-1, digits=True)
    return [r["digits"], np.array([r["res64"], r["old64"], r["hash64"]], dtype=np.uint64).view(np.int64)]


def work(case):
    """The digits a pass starts from read once and those it returns written once, and for every
    squaring the 5 N log2 N operations of a floating-point convolution of N real values (two
    transforms)."""
    kind, n = case["kind"], case["n"]
    if kind == "batch":
        sizes = [12 + (i & 1) for i in range(case["cap"])] if case["mixed"] else [n] * case["cap"]
        sq = [(m, case["iters"]) for m in sizes]
        moved = sum(4 << m for m in sizes)  # the residues' digits, read for their hashes
    elif kind == "request":
        sq, moved = [(n, case["iters"])], 4 << n
    else:
        sq, moved = [(n, case["count"] * 3 // 2 if kind == "power" else case["count"])], 8 << n
    return {"bytes": moved, "flops": sum(c * 5 * m * (1 << m) for m, c in sq)}


def _balanced(v, n, b):
    """Balanced digits of the residue v mod b^(2^n) + 1."""
    N = 1 << n
    pw = [b]
    while len(pw) < n:
        pw.append(pw[-1] * pw[-1])
    out = np.zeros(N, dtype=np.int64)

    def split(x, lo, k):
        if k == 0:
            out[lo] = x
            return
        hi, rest = divmod(x, pw[k - 1])
        split(rest, lo, k - 1)
        split(hi, lo + (1 << (k - 1)), k - 1)

    sign = 1
    if v == b ** N:
        v, sign = 1, -1
    split(v, 0, n)
    d = [sign * int(x) for x in out]
    half, c, i = b // 2, 0, 0
    while i < N or c:
        x = d[i % N] + c
        c = 0
        while x > half:
            x, c = x - b, c + 1
        while x < -((b - 1) // 2):
            x, c = x + b, c - 1
        d[i % N] = x
        i += 1
        if i % N == 0:
            c = -c
        if i >= N and c == 0:
            break
    return np.array(d, dtype=np.int32)


def exact(case, seed):
    """The residue by Python's integers, where that takes seconds (one candidate, n = 12)."""
    if case["kind"] not in ("prp", "noalloc") or case["n"] > 12 or case["count"] > 100:
        return None
    n, b, N = case["n"], case["b"], 1 << case["n"]
    digits, dup = _inputs(case, seed)
    bits = dup if case["kind"] == "prp" else [(dup >> (i % 64)) & 1 for i in range(case["count"])]
    parts, base = [int(x) for x in digits], b
    while len(parts) > 1:
        parts = [parts[i] + parts[i + 1] * base for i in range(0, len(parts), 2)]
        base *= base
    F = b ** N + 1
    v = parts[0] % F
    for bit in bits:
        v = v * v
        if bit:
            v += v
        hi, lo = divmod(v, F - 1)  # b^N = -1
        v = (lo - hi) % F
    return _balanced(v, n, b)
