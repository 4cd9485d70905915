// gfe_f64q.h -- the double-precision transform with limbs of four digits over five 45.5-bit primes.
//
// b^N + 1 = B^M + 1 with B = b^4, M = N / 4.  Against limbs of two digits over three 49-bit primes
// (gfe_f64.h, whose passes these are) that is 5/4 N instead of 3/2 N residues and one level fewer, so
// a sixth less to move and a fifth fewer instructions; and with 2^53 > 180 p the passes hardly reduce:
// forward levels and the pointwise products run unreduced (at most 14 p), inverse chunks reduce few
// elements.  Exact for b from 2^20 to about 2^25.8 at n = 22 (f64q_ok), and faster from n = 20 on; us a
// squaring, limbs of two digits and of four on one machine: n = 20 33.9 and 30.6, 21 45.7 and 41.6,
// 22 80.2 and 70.6 (76.9 and 65.5 on a cooler one), 23 152.5 and 139.0.
// A pass takes about the sum of its moves and its arithmetic.  At n = 22: forward 9.6 of moves and 6 of
// arithmetic, rows 12.6 and 18, inverse 8.5 and 13.  A column pass's 256 workgroups are all resident at
// once, two waves a SIMD, and load, compute and store together; the row pass's 1280 of 8 waves are four
// a CU and a quarter of a layer more.
//
// CRT: as in gfe_f64.h, mixed-radix digits v1..v5 of the coefficient (v5 the centred one) and the
// base-b pieces of p1, p1 p2, .., here modulo b^9: nine pieces g0..g8 of at most 0.51 b, the last
// the coefficient's quotient by b^8, which the rule keeps below b / 2.
#pragma once

#include "gfe_f64.h"

namespace gfe {

constexpr int F64Q_PRIMES = 5;
constexpr uint32_t F64Q_MIN_N = 20;
constexpr int F64Q_COL_MIN = 6, F64Q_SPLIT_MAX = 7, F64Q_COL_MAX = 8, F64Q_ROW_MIN = 12, F64Q_ROW_MAX = 13;  // instantiated shapes
// p = k 2^24 + 1 below 2^45.5 with their least primitive roots
constexpr uint64_t F64Q_P[F64Q_PRIMES] = {49757816881153ull, 49757632331777ull, 49757078683649ull, 49756457926657ull,
                                          49756323708929ull};
constexpr uint32_t F64Q_G[F64Q_PRIMES] = {7, 5, 3, 5, 3};

// In units of p (2^53 > 181 p): a product by a constant is at most 0.52 + 0.0085 B, one of two
// residues 0.5 + 0.0167 B B'.  Limbs enter at 2.3 p (f64q_limb), 19 levels later they are below 14 p;
// a coefficient of the pointwise square, three products of those, is below 18 p.
struct F64Slim {
    static constexpr double lim = 170.0, start = 18.0, keep = 8.0, slope = 0.0085;
    static constexpr bool reduce = false;
};

struct F64QCrt {
    double p[5], pinv[5];
    double s[2][5];              // scale of prime k's raw output mod p_k, doubled for dup
    double inv[5][4];            // inv[k][j] = p_j^-1 mod p_k, j < k
    double sq[5];                // b^2 mod p_k
    double w[4][9], u[4][9];     // p1 .. p_(j+1) and 2^23 times it in base b, modulo b^9
    double bd, binv, qb;         // b, 1 / b, 1 / (4 b)
};
typedef const F64QCrt GFE_AS4 *F64QCrtP;

// The limb y0 + b^2 y1 of two digit pairs mod p: |y0|, |y1| < 146 p.
__device__ __forceinline__ double f64q_limb(const F64Mod &md, double y0, double y1, double sq) {
    return md.mul(y1, sq) + md.red(y0);
}

// The group's digits with the range carries of the last normalisation added: the carry into range
// k C / 16 + blk is (u0, u1, u2, u3), on the digits of limb 0, then (v, ..), on digit 0 of limb 1.
template <int LOGE, int LOGG>
__device__ __forceinline__ void f64q_load_digits(int4 (&d)[1 << LOGE], const int32_t *__restrict__ src,
                                                 const int4 *__restrict__ ls, uint32_t C, unsigned blk, uint32_t t) {
    constexpr int E = 1 << LOGE, YL = LOGG - LOGE;
    const uint32_t q = t & 15u, s = t >> 4;
    const int4 *g = reinterpret_cast<const int4 *>(src) + (size_t)s * C + blk * 16 + q;
#pragma unroll
    for (int rr = 0; rr < E; ++rr) d[rr] = g[((size_t)rr << YL) * C];
    if (ls && q < 2) {
        const int4 *c = ls + (size_t)s * (C / 8) + blk * 2 + q;
        int4 e[E];
#pragma unroll
        for (int rr = 0; rr < E; ++rr) e[rr] = c[((size_t)rr << YL) * (C / 8)];
#pragma unroll
        for (int rr = 0; rr < E; ++rr) {
            d[rr].x += e[rr].x;
            d[rr].y += q == 0 ? e[rr].y : 0;
            d[rr].z += q == 0 ? e[rr].z : 0;
            d[rr].w += q == 0 ? e[rr].w : 0;
        }
    }
}

// Pieces of p1 .. p_(j+1) and 2^23 times it in base b >= 2^20 (45.5 (j + 1) and 23 more bits).
constexpr int f64q_w_pieces(int j) { return 2 * j + 3; }
constexpr int f64q_u_pieces(int j) { return j >= 2 ? 9 : 2 * j + 4; }

// Base-b pieces g[0..8] of the coefficient with raw residues r[0..4].  Each v but the first is taken in
// halves of 23 bits, whose products with base-b pieces (2^26 at most) add up exactly in 53 bits.
__device__ __forceinline__ void f64q_crt_pieces(F64QCrtP c, const double (&r)[5], int dup, double (&g)[9]) {
    const double binv = c->binv, bd = c->bd;
    double v[5], lo[5], hi[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        const F64Mod md{c->p[k], c->pinv[k]};
        double t = md.mul(r[k], c->s[dup][k]);
#pragma unroll
        for (int j = 0; j < k; ++j) t = md.mul(t - v[j], c->inv[k][j]);
        v[k] = t;
        hi[k] = rint(t * 0x1p-23);
        lo[k] = fma(-hi[k], 0x1p23, t);
    }
    double S = v[0];
#pragma unroll
    for (int i = 0; i < 9; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (i < f64q_w_pieces(j)) S = fma(lo[j + 1], c->w[j][i], S);
            if (i < f64q_u_pieces(j)) S = fma(hi[j + 1], c->u[j][i], S);
        }
        const double q = rint(S * binv);
        g[i] = fma(-q, bd, S);
        S = q;
    }
}

// Limb of lane q (16 lanes = 16 consecutive limbs): four digits, balanced but for the carry of the lane
// below (at most 2) added to the first; lane 15's share of the next range's first two limbs in
// u = (g4 + g8 of lane 14 + carry, g5, g6, g7) and g[8].
__device__ __forceinline__ int4 f64q_limb_digits(F64QCrtP c, const double (&g)[9], int4 &u) {
    const double bd = c->bd, binv = c->binv, qb = c->qb;
    const int32_t h[4] = {(int32_t)g[4] + f64_lane_below<1>((int32_t)g[8]), (int32_t)g[5], (int32_t)g[6], (int32_t)g[7]};
    int32_t D[4];
    double q = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const double X = g[i] + (double)f64_lane_below<1>(h[i]) + q;
        q = rint(fma(X, binv, -qb));
        D[i] = (int32_t)fma(-q, bd, X);
    }
    const int32_t cr = (int32_t)q;
    u = make_int4(h[0] + cr, h[1], h[2], h[3]);
    return make_int4(D[0] + f64_lane_below<1>(cr), D[1], D[2], D[3]);
}

// Digits of limb i from its raw residues, stored with the carry into the next range of 16.
__device__ __forceinline__ void f64q_norm_limb(F64QCrtP c, const double (&r)[5], int dup, uint32_t i, uint32_t M,
                                               int32_t *__restrict__ dst, int4 *__restrict__ slots) {
    double g[9];
    f64q_crt_pieces(c, r, dup, g);
    int4 u;
    reinterpret_cast<int4 *>(dst)[i] = f64q_limb_digits(c, g, u);
    if ((i & 15u) == 15u) {
        uint32_t w = (i >> 4) + 1;
        int32_t v = (int32_t)g[8];
        if (w == M / 16) { w = 0; u = make_int4(-u.x, -u.y, -u.z, -u.w); v = -v; }  // B^M = -1
        slots[2 * w] = u;
        slots[2 * w + 1] = make_int4(v, 0, 0, 0);
    }
}

// As f64_flush_range for range w of 64 digits.
template <bool STORE = true>
__device__ __forceinline__ int32_t f64q_flush_range(const int32_t *src, int32_t *dst, const int4 *slots, uint32_t b, uint32_t w) {
    const double bd = (double)b, binv = 1.0 / bd, qb = 0.25 * binv;
    const int4 u = slots[2 * w], v = slots[2 * w + 1];
    const int4 *p = reinterpret_cast<const int4 *>(src + (size_t)w * 64);
    int4 *o = reinterpret_cast<int4 *>(dst + (size_t)w * 64);
    int4 in[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) in[i] = p[i];
    double c = 0.0;
    auto digit = [&](int32_t d, int32_t e) -> int32_t {
        const double D = (double)d + (double)e + c;
        c = rint(fma(D, binv, -qb));
        return (int32_t)fma(-c, bd, D);
    };
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        int4 x = in[i];
        x.x = digit(x.x, i == 0 ? u.x : i == 1 ? v.x : 0);
        x.y = digit(x.y, i == 0 ? u.y : 0);
        x.z = digit(x.z, i == 0 ? u.z : 0);
        x.w = digit(x.w, i == 0 ? u.w : 0);
        if constexpr (STORE) o[i] = x;
    }
    return (int32_t)c;
}

// As f64_flush_body; the carry out stays in slots[2 w + 1].w.
__device__ __forceinline__ void f64q_flush_body(int32_t *dst, int4 *slots, uint32_t b, uint32_t w) {
    const int32_t c = f64q_flush_range(dst, dst, slots, b, w);
    slots[2 * w] = make_int4(0, 0, 0, 0);
    slots[2 * w + 1] = make_int4(0, 0, 0, c);
}

}  // namespace gfe
