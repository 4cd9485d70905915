"""The double-precision limb transform's arithmetic (genefer22_amd/csrc/gfe_f64.h), emulated with
Python floats (IEEE doubles; fma and the exact steps through Fraction) against integers: the modular
product and its size bound, and the CRT with the digit split at the edges of the host's rule for
every prime count.  The kernels themselves run in tests/test_gpu_f64.py."""
import random
from fractions import Fraction

import pytest

P = [562949869535233, 562949517213697, 562949282332673]
G = [5, 10, 3]


def fma(a, b, c):
    return float(Fraction(a) * Fraction(b) + Fraction(c))


def rint(x):
    return float(round(x))  # ties to even, as v_rndne_f64


def mul(a, w, p, pinv):
    h = a * w
    l = fma(a, w, -h)
    q = rint(h * pinv)
    return fma(-q, float(p), h) + l


def bal(v, p):
    v %= p
    return float(v - p if v > p // 2 else v)


def test_primes():
    for p, g in zip(P, G):
        assert p < 2**49 and (p - 1) % 2**24 == 0
        assert pow(g, p - 1, p) == 1 and pow(g, (p - 1) // 2, p) == p - 1
        assert all(p % d for d in range(3, 100000, 2))


@pytest.mark.parametrize("k", range(3))
def test_product_is_exact_and_bounded(k):
    """r = a w mod p for |a| up to 15 p, |w| up to 0.51 p: congruent, and at most 0.52 + 0.096 |a| / p."""
    p, pinv, rng = P[k], 1.0 / P[k], random.Random(k)
    for i in range(3000):
        B = rng.choice([0.5, 1.0, 2.0, 4.0, 8.0, 12.0, 14.9])
        a = float(rng.choice([-1, 1]) * (int(B * p) - rng.randrange(1000 if i % 2 else int(B * p))))
        w = float(rng.choice([-1, 1]) * (int(0.51 * p) - rng.randrange(1000 if i % 3 else int(0.51 * p))))
        r = mul(a, w, p, pinv)
        assert (int(r) - int(a) * int(w)) % p == 0
        assert abs(r) <= (0.52 + 0.096 * abs(a) / p) * p


def bound(b, n, K):
    """The host's rule restated: the largest doubled coefficient, or None where (b, n) is refused."""
    M, L = 2 ** (n - 1), (b / 2 + 4) * (b + 1)
    g = M / 2 + 4
    for _ in range(64):
        L0, L1 = (b + 5) + b * (1.05 * b + 6 + g / b + 2), L + g + 2
        X = 2 * (M / 16) * (L0 * L0 + L1 * L1 + 14 * L * L)
        if X / b**4 + 4 <= g:
            break
        g = (X / b**4 + 4) * 1.001
        if g > b * b or g > 1e8:
            return None
    prod = P[0] * P[1] * (P[2] if K == 3 else 1)
    return X if g <= b * b and g <= 1e8 and X < (0.3 if K == 3 else 0.1) * prod else None


def split(x, b, pieces):
    out = []
    for i in range(pieces - 1):
        r = x % b
        if r > b // 2:
            r -= b
        out.append(r)
        x = (x - r) // b
    return out + [x]


def lo32(v):
    return int(v) & 0xFFFFFFFF


def s32(v):
    v &= 0xFFFFFFFF
    return v - (1 << 32) if v >> 31 else v


def pieces(x, b, n, K, dup, rng):
    """f64_crt_pieces on raw residues of any representative up to 15 p."""
    pinv = [1.0 / p for p in P]
    raw, sc = [], []
    for k in range(K):
        p = P[k]
        s = pow(pow(2, n - 3, p), -1, p)
        v = (x // (2 if dup else 1)) * pow(s, -1, p) % p
        raw.append(float(v + p * rng.randrange(-15, 15)))
        sc.append(bal(s * (2 if dup else 1), p))
    binv = 1.0 / b
    v1 = mul(raw[0], sc[0], P[0], pinv[0])
    v2 = mul(mul(raw[1], sc[1], P[1], pinv[1]) - v1, bal(pow(P[0], -1, P[1]), P[1]), P[1], pinv[1])
    vs = [(v1, [1, 0, 0, 0, 0]), (v2, split(P[0], b, 3) + [0, 0] if K == 3 else split(P[0], b, 5))]
    if K == 3:
        t = mul(raw[2], sc[2], P[2], pinv[2]) - v1
        t = mul(t, bal(pow(P[0], -1, P[2]), P[2]), P[2], pinv[2]) - v2
        v3 = mul(t, bal(pow(P[1], -1, P[2]), P[2]), P[2], pinv[2])
        vs.append((v3, split(P[0] * P[1], b, 5)))
    g, q, ql = [], 0.0, 0
    for i in range(5):
        S, Sl = q, ql
        for v, w in vs:
            if w[i]:
                S = v if w[i] == 1 and i == 0 and v is v1 else fma(v, float(w[i]), S)
                Sl += lo32(v) * (w[i] & 0xFFFFFFFF)
        if i == 4:
            g.append(s32(Sl))
        else:
            q = rint(S * binv)
            assert abs(q) < 2**51
            ql = lo32(q)
            g.append(s32(Sl - ql * b))
    return g


# (b, n, K): the ends of the rule -- the smallest and largest base of two primes, the smallest and the
# largest of three, at the smallest and the largest n
EDGES = []
for _n in (12, 17, 23):
    for _K in (2, 3):
        ok = [b for e in range(10, 31) for b in (2**e + 2, 2**e + 2**(e - 1), 2**(e + 1) - 2) if b <= 2_000_000_000 and
              (_K == 2 or b >= 2**17) and bound(b, _n, _K)] + ([2_000_000_000] if _K == 3 else [])
        EDGES += [(ok[0], _n, _K), (ok[-1], _n, _K)]


@pytest.mark.parametrize("b,n,K", EDGES)
def test_crt_pieces_at_the_rules_edges(b, n, K):
    X = bound(b, n, K)
    assert X is not None
    rng = random.Random(b + n)
    X = int(X)
    xs = [0, 1, -1, X, -X, X - 1, b**4 if b**4 < X else X // 2]
    xs += [rng.choice([-1, 1]) * rng.randrange(1 << rng.randrange(1, X.bit_length())) for _ in range(300)]
    xs += [rng.randrange(-X, X) for _ in range(300)]
    for x in xs:
        for dup in (0, 1):
            v = x - (x & 1) if dup else x
            if abs(v) > X:
                continue
            g = pieces(v, b, n, K, dup, rng)
            assert sum(gi * b**i for i, gi in enumerate(g)) == v
            assert all(abs(gi) <= 0.65 * b for gi in g[:4]) and abs(g[3]) <= 0.55 * b
            assert abs(g[4]) <= X / b**4 + 4 and abs(g[2]) + abs(g[4]) < 2**31


def test_digit_quotient_is_balanced():
    """rint(fma(D, 1/b, -1/(4b))) leaves a remainder in (-b/2, b/2], ties down, for every sum D."""
    rng = random.Random(7)
    for b in (1024, 1025, 146950, 33554434, 1999999998, 2_000_000_000):
        binv, lo, hi = 1.0 / b, -((b - 1) // 2), b // 2
        for _ in range(2000):
            D = rng.choice([rng.randrange(-2**33, 2**33), rng.randrange(-3, 4) * b + rng.choice([lo, hi, lo - 1, hi + 1, 0])])
            q = rint(fma(float(D), binv, -(0.25 * binv)))
            assert lo <= D - int(q) * b <= hi


def test_rule_covers_the_range_in_use():
    """b = 2e9 at n = 23 needs three primes and fits; C1's and the largest n's small bases need two."""
    assert bound(2_000_000_000, 23, 3) and not bound(2_000_000_000, 23, 2)
    assert bound(2_000_000, 12, 2) and bound(150_000, 23, 2) and bound(1024, 12, 2)
    for n in range(12, 21):  # every base
        for b in list(range(1024, 5000, 7)) + [int(1024 * 1.05**i) for i in range(298)] + [2_000_000_000]:
            assert bound(b, n, 2) or (b >= 2**17 and bound(b, n, 3)), (b, n)
    for n, b in ((21, 1148), (22, 1622), (23, 2292)):  # the first base covered
        assert bound(b, n, 2) and not bound(b - 2, n, 2)


# Limbs of four digits over five 45.5-bit primes (gfe_f64q.h)
Q = [49757816881153, 49757632331777, 49757078683649, 49756457926657, 49756323708929]
QPROD = Q[0] * Q[1] * Q[2] * Q[3] * Q[4]


def qbound(b, n):
    """The host's rule restated: the largest doubled coefficient, or None where (b, n) is refused."""
    if not 20 <= n <= 23 or b < 2**20 or b * b > 1.5 * 2**52:
        return None
    M, up = 2 ** (n - 2), (b + 1) * (b * b + 1)
    half = Fraction(b, 2)
    L, g = (half + 4) * up, min(M, half) - 4
    X = 2 * (M // 16) * (((Fraction(106, 100) * b + g + 8) * up) ** 2 + (L + g) ** 2 + 14 * L * L)
    return X if 10 * X < 3 * QPROD and X / b**8 + 4 < g else None


def qedges(n):
    """Smallest and largest base of the rule at n."""
    lo, hi = 2**20 - 1, 2**23
    while hi - lo > 1:
        m = (lo + hi) // 2
        lo, hi = (lo, m) if qbound(m, n) else (m, hi)
    lo2, hi2 = 2**23, 2**27
    while hi2 - lo2 > 1:
        m = (lo2 + hi2) // 2
        lo2, hi2 = (m, hi2) if qbound(m, n) else (lo2, m)
    return hi, lo2


def base_pieces(x, b, count):
    out = []
    for _ in range(count):
        r = x % b
        if r > b // 2:
            r -= b
        out.append(r)
        x = (x - r) // b
    return out


def qpieces(x, b, n, dup, rng):
    """f64q_crt_pieces on raw residues of any representative up to 64 p (8 p into the last chunk of three levels); every sum has to be exact."""
    v = []
    for k, p in enumerate(Q):
        pinv, s = 1.0 / p, pow(pow(2, n - 4, p), -1, p)
        raw = float((x // (2 if dup else 1)) * pow(s, -1, p) % p + p * rng.randrange(-64, 64))
        t = mul(raw, bal(s * (2 if dup else 1), p), p, pinv)
        for j in range(k):
            t = mul(t - v[j], bal(pow(Q[j], -1, p), p), p, pinv)
        v.append(t)
    hi = [rint(t * 2.0**-23) for t in v]
    lo = [fma(-h, 2.0**23, t) for h, t in zip(hi, v)]
    prod, w, u = 1, [], []
    for j in range(4):
        prod *= Q[j]
        w.append(base_pieces(prod, b, 9))
        u.append(base_pieces(prod << 23, b, 9))
        assert not any(w[j][2 * j + 3:]) and (j >= 2 or not any(u[j][2 * j + 4:]))  # what the kernel leaves out
    g, S = [], v[0]
    for i in range(9):
        exact = int(S) + sum(int(lo[j + 1]) * w[j][i] + int(hi[j + 1]) * u[j][i] for j in range(4))
        for j in range(4):
            S = fma(lo[j + 1], float(w[j][i]), S)
            S = fma(hi[j + 1], float(u[j][i]), S)
        assert int(S) == exact
        q = rint(S * (1.0 / b))
        g.append(int(fma(-q, float(b), S)))
        assert g[-1] == exact - int(q) * b
        S = q
    return g


def test_four_digit_primes():
    for p, gen in zip(Q, (7, 5, 3, 5, 3)):
        assert p < 2**45.5 and (p - 1) % 2**24 == 0
        assert pow(gen, p - 1, p) == 1 and pow(gen, (p - 1) // 2, p) == p - 1
        assert all(p % d for d in range(3, 100000, 2))


def test_four_digit_product_is_bounded():
    """|r| <= 0.52 + 0.0085 B by a constant, 0.5 + 0.0167 B B' (and 0.02 of slack) by a residue."""
    rng = random.Random(5)
    for i in range(6000):
        p = Q[i % 5]
        B, C = rng.choice([(1.0, 0.5), (14.0, 0.5), (146.0, 0.5), (14.0, 14.0), (28.0, 14.0), (4.0, 8.0)])
        a, w = (float(rng.choice([-1, 1]) * (int(x * p) - rng.randrange(1000 if i % 2 else int(x * p)))) for x in (B, C))
        r = mul(a, w, p, 1.0 / p)
        assert (int(r) - int(a) * int(w)) % p == 0
        assert abs(r) <= (0.52 + 0.0085 * abs(a) / p if C == 0.5 else 0.52 + 0.0167 * abs(a * w) / p / p) * p


@pytest.mark.parametrize("n", range(20, 24))
def test_four_digit_pieces_at_the_rules_edges(n):
    for b in (*qedges(n), 2**23 + 2):
        X, rng = int(qbound(b, n)), random.Random(b)
        assert b * b * 1.07 < 2**53 and 1.07 * b * b < 146 * min(Q)
        xs = [0, 1, -1, X, -X, b**8, -b**8 // 2] + [rng.randrange(-X, X) for _ in range(150)]
        xs += [rng.choice([-1, 1]) * rng.randrange(1 << rng.randrange(1, X.bit_length() - 1)) for _ in range(150)]
        for x in xs:
            for dup in (0, 1):
                x2 = x - (x & 1) if dup else x
                g = qpieces(x2, b, n, dup, rng)
                assert sum(gi * b**i for i, gi in enumerate(g)) == x2
                assert all(abs(gi) <= 0.55 * b for gi in g)
