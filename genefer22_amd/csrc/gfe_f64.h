// gfe_f64.h -- the two-digit-limb transform in double precision: exact modular arithmetic over two
// or three 49-bit primes on the fp64 vector units.
//
// b^N + 1 = B^M + 1 with B = b^2, M = N / 2: the register's digits pair into M limbs d_2j + b d_2j+1
// and a squaring is a negacyclic convolution of the limbs (as in gfe_limb.h).  A residue is an
// integer-valued double of either sign, not necessarily reduced: |x| < 2^53 is all that its
// exactness needs.  A product a w mod p takes six full-rate instructions,
//     h = a w,  l = fma(a, w, -h),  q = rint(h / p),  r = fma(-q, p, h) + l,
// each step after h exact (h + l = a w; h - q p is an integer below 2^53), and leaves |r| a little
// above p / 2; additions and subtractions are not reduced at all.  A butterfly is therefore eight
// instructions for 49 bits; in 32-bit integer arithmetic it is twelve for 31.  fp64 multiplies,
// additions and fma issue at the rate of 32-bit integer multiplies on gfx950 (measured: 50-57
// lane-operations per clock and CU for v_fma_f64, v_add_f64, v_mul_f64 and v_rndne_f64, 54-58 for
// v_mul_lo_u32 and v_mul_hi_u32), so a squaring needs about half the instructions.
//
// Sizes in units of p (p < 2^49, so 2^53 > 16 p).  The rounding of q costs at most
// 3 2^-53 |a w| / p <= 0.094 B for |a| = B p, |w| <= 0.51 p, so a product is below 0.52 + 0.096 B
// (F64Wide).  Forward levels add one product per level, so they run unreduced from 2 p through a
// whole column pass and, from a reduced start, through a whole row pass.  The inverse sums double
// per level: its reductions are placed at compile time from the same bounds (InvSched).
//
// The row pass stops two levels early: a row's last two levels would split X^4 - w; instead four
// residues a0..a3 are squared (or multiplied) as a polynomial modulo X^4 - w, in the thread that
// holds them.  That costs 22 instructions per residue against 25 for the two levels both ways and the
// square, and the twiddle table shrinks to a quarter (M / 4 entries per prime).
//
// CRT (crt_pieces).  v1, v2, v3 are mixed-radix digits of the coefficient x = v1 + p1 v2 + p1 p2 v3,
// any representatives of v1 and v2 and the centred one of v3 (|x| < 0.3 P puts it well inside).  With
// p1 and p1 p2 split into base-b pieces on the host, x = g0 + g1 b + g2 b^2 + g3 b^3 + g4 b^4 follows
// digit by digit: a sum S known as a double and mod 2^32, the quotient q = rint(S / b) within 0.75
// of S / b, the piece S - q b exact in 32 bits.  Every piece but the last is at most 0.75 b in size, the
// last at most a coefficient over b^4 (f64_bound's G, range carries included: 0.3 N for large bases, never
// over b^2 or 1e8).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "gfe_device.h"

namespace gfe {

constexpr int F64_PRIMES = 3;
// p = k 2^24 + 1 below 2^49 with their least primitive roots
constexpr uint64_t F64_P[F64_PRIMES] = {562949869535233ull, 562949517213697ull, 562949282332673ull};
constexpr uint32_t F64_G[F64_PRIMES] = {5, 10, 3};
constexpr int F64_ROW_MIN = 8, F64_ROW_BATCH = 12, F64_ROW_MAX = 14;  // the longest rows of a batch (n <= 20) and of all
constexpr int F64_COL_MIN = 5, F64_COL_MAX = 8, F64_SPLIT_MAX = 7;
constexpr int F64_WHOLE_MIN = 11, F64_WHOLE_MAX = 12;           // log2 limbs of a one-workgroup transform
constexpr uint32_t F64_NORM_T = 64;  // limbs per workgroup of its normalisation
constexpr int F64_COL_E = 3;     // log2 of the residues per thread in the column passes

// Constants of one candidate, read with scalar loads.
struct F64Crt {
    double p[3], pinv[3];
    double s[2][3];              // scale of prime k's raw output mod p_k, doubled for dup
    double i12, i13, i23;        // p1^-1 mod p2, p1^-1 mod p3, p2^-1 mod p3
    double w1[5], w2[5];         // p1 and p1 p2 in base b: balanced pieces, the last takes the rest
    double bd, binv, qb;         // b, 1 / b, 1 / (4 b)
    uint32_t w1l[5], w2l[5];     // their low words
    uint32_t b;
    int32_t big;                 // limbs that enter a pass unreduced: 0 all of them (below p / 2), 1 those
                                 // of a column pass (below 2 p), 2 none
    int32_t n, K;                // the candidate's n and primes
};

#define GFE_AS4 __attribute__((address_space(4)))
typedef const F64Crt GFE_AS4 *F64CrtP;
typedef const double GFE_AS4 *F64ConstP;

struct F64Mod {
    double p, pinv;
    __device__ __forceinline__ double mul(double a, double w) const {
        const double h = a * w, l = fma(a, w, -h), q = rint(h * pinv);
        return fma(-q, p, h) + l;
    }
    __device__ __forceinline__ double red(double x) const { return fma(-rint(x * pinv), p, x); }
};

template <int I, int END, class F>
__device__ __forceinline__ void f64_for(const F &f) {
    if constexpr (I < END) {
        f(std::integral_constant<int, I>{});
        f64_for<I + 1, END>(f);
    }
}
template <int I, int END, class F>
__device__ __forceinline__ void f64_for_down(const F &f) {
    if constexpr (I < END) {
        f(std::integral_constant<int, END - 1>{});
        f64_for_down<I, END - 1>(f);
    }
}

// ---------------------------------------------------------------------------------------------
// Bounds and chunks

// Bounds of a prime size, in units of p: lim the largest operand a butterfly may form, start what the
// inverse transform starts from, keep what an inverse chunk leaves, a product of B p by a constant
// at most 0.52 + slope B; reduce: rows reduce on the way in and before the pointwise products.
struct F64Wide {  // p < 2^49
    static constexpr double lim = 15.0, start = 1.8, keep = 1.8, slope = 0.096;
    static constexpr bool reduce = true;
};

// Where the inverse chunk of NE levels on 2^LOGE elements, all at most B0 p, reduces: pre[mu] bit i
// before level mu, post bit i after the last.
template <class SZ, int LOGE, int NE>
struct InvSched {
    uint32_t pre[NE > 0 ? NE : 1] = {};
    uint32_t post = 0;
    constexpr explicit InvSched(double B0) {
        constexpr int E = 1 << LOGE;
        double B[E] = {};
        for (int i = 0; i < E; ++i) B[i] = B0;
        for (int mu = NE - 1; mu >= 0; --mu) {
            const int h = E >> (mu + 1);
            for (int bi = 0; bi < (1 << mu); ++bi)
                for (int i = 0; i < h; ++i) {
                    const int i0 = bi * 2 * h + i, i1 = i0 + h;
                    if (B[i0] + B[i1] > SZ::lim) {
                        if (B[i0] > SZ::keep) { pre[mu] |= 1u << i0; B[i0] = 0.51; }
                        if (B[i1] > SZ::keep) { pre[mu] |= 1u << i1; B[i1] = 0.51; }
                    }
                    const double s = B[i0] + B[i1];
                    B[i0] = s;
                    B[i1] = 0.52 + SZ::slope * s;
                }
        }
        for (int i = 0; i < E; ++i)
            if (B[i] > SZ::keep) post |= 1u << i;
    }
};

// Forward levels 0..NE-1 of the chunk in x[], twiddle of level mu, block bi at w[2^mu + bi].
template <int LOGE, int NE, class W>
__device__ __forceinline__ void f64_fwd_chunk(const F64Mod &md, double (&x)[1 << LOGE], const W &w) {
    constexpr int E = 1 << LOGE;
#pragma unroll
    for (int mu = 0; mu < NE; ++mu) {
        const int h = E >> (mu + 1);
#pragma unroll
        for (int bi = 0; bi < (1 << mu); ++bi) {
            const double wv = w[(1 << mu) + bi];
#pragma unroll
            for (int i = 0; i < h; ++i) {
                const int i0 = bi * 2 * h + i, i1 = i0 + h;
                const double u = x[i0], v = md.mul(x[i1], wv);
                x[i0] = u + v;
                x[i1] = u - v;
            }
        }
    }
}

// Inverse levels NE-1..0: the twiddle of block bi, level mu is -1 / w[2^mu + bi]'s mirror (f64_inv_tw),
// so the difference enters as v - u.  FIRST: of the inverse transform; POST: bring every element back to
// SZ::keep.
template <class SZ, int LOGE, int NE, bool FIRST, bool POST, class W>
__device__ __forceinline__ void f64_inv_chunk(const F64Mod &md, double (&x)[1 << LOGE], const W &w) {
    constexpr int E = 1 << LOGE;
    constexpr InvSched<SZ, LOGE, NE> S{FIRST ? SZ::start : SZ::keep};
#pragma unroll
    for (int mu = NE - 1; mu >= 0; --mu) {
        const int h = E >> (mu + 1);
#pragma unroll
        for (int i = 0; i < E; ++i)
            if ((S.pre[mu] >> i) & 1u) x[i] = md.red(x[i]);
#pragma unroll
        for (int bi = 0; bi < (1 << mu); ++bi) {
            const double wv = w[(1 << mu) + bi];
#pragma unroll
            for (int i = 0; i < h; ++i) {
                const int i0 = bi * 2 * h + i, i1 = i0 + h;
                const double u = x[i0], v = x[i1];
                x[i0] = u + v;
                x[i1] = md.mul(v - u, wv);
            }
        }
    }
    if constexpr (POST) {
#pragma unroll
        for (int i = 0; i < E; ++i)
            if ((S.post >> i) & 1u) x[i] = md.red(x[i]);
    }
}

// Twiddles of a chunk whose first level is lam and whose sub-transform is block J of that level
// (table Psi[m + j] = psi^bitrev(m + j), m = 2^level): w[2^mu + bi] = Psi[2^(lam+mu) + J 2^mu + bi],
// inverse Psi[2 2^(lam+mu) - 1 - J 2^mu - bi] (= -1 / Psi of the forward one).  UNI: lam and J are
// the same in the whole wave and the loads are scalar.
template <int LOGE, bool UNI>
__device__ __forceinline__ void f64_fwd_tw(double (&w)[1 << LOGE], const double *tw, uint32_t lam, uint32_t J, int NE) {
#pragma unroll
    for (int mu = 0; mu < NE; ++mu) {
        const uint32_t at = (1u << (lam + mu)) + (J << mu);
        if constexpr (UNI) {
            const F64ConstP q = (F64ConstP)(tw + __builtin_amdgcn_readfirstlane(at));
#pragma unroll
            for (int bi = 0; bi < (1 << mu); ++bi) w[(1 << mu) + bi] = q[bi];
        } else {
#pragma unroll
            for (int bi = 0; bi < (1 << mu); ++bi) w[(1 << mu) + bi] = tw[at + bi];
        }
    }
}
template <int LOGE, bool UNI>
__device__ __forceinline__ void f64_inv_tw(double (&w)[1 << LOGE], const double *tw, uint32_t lam, uint32_t J, int NE) {
#pragma unroll
    for (int mu = 0; mu < NE; ++mu) {
        const uint32_t at = (2u << (lam + mu)) - (J << mu) - (1u << mu);
        if constexpr (UNI) {
            const F64ConstP q = (F64ConstP)(tw + __builtin_amdgcn_readfirstlane(at));
#pragma unroll
            for (int bi = 0; bi < (1 << mu); ++bi) w[(1 << mu) + bi] = q[(1 << mu) - 1 - bi];
        } else {
#pragma unroll
            for (int bi = 0; bi < (1 << mu); ++bi) w[(1 << mu) + bi] = tw[at + (1u << mu) - 1u - bi];
        }
    }
}

// Chunks of a LOGG-level pass in steps of LOGE levels, the first one partial (as Geo in gfe_pass.h).
template <int LOGG, int LOGE>
struct F64Geo {
    static_assert(LOGG >= LOGE, "a pass spans at least one chunk");
    static constexpr int R = LOGG % LOGE;
    static constexpr int NCH = (LOGG + LOGE - 1) / LOGE;
    static constexpr int lam0(int ci) { return R == 0 ? ci * LOGE : (ci == 0 ? 0 : R + (ci - 1) * LOGE); }
    static constexpr int ne(int ci) { return (R != 0 && ci == 0) ? R : LOGE; }
    static constexpr int ylog(int ci) { return LOGG - lam0(ci) - LOGE; }
};

// ---------------------------------------------------------------------------------------------
// Row pass: rows of 2^LOGG contiguous residues, 2^LOGE per thread, thread s of a row.  Exchanges through
// LDS at k + (k >> LOGE) (64-bit accesses of 16 consecutive lanes fall in distinct banks in every
// chunk with 16 residues per thread, and with 8 but for one lane of 16).  MODE as in gfe_kernels.h: square, product by zp, or forward only.

// F64_EITHER: a square, or the product where `mul` (uniform over the workgroup): rounds of batched powers.

enum { F64_SQUARE = 0, F64_MUL = 1, F64_FWD = 2, F64_EITHER = 3 };

// 8 residues a thread, 16 from 2^13 on (where 8 would be 1024 threads and gain nothing).  Twice the waves
// outweigh one exchange more: us per round or squaring with 16 and with 8 a thread, 8 slots of n = 12
// 9.1 and 7.7, 301 19.7 and 19.0, 1024 47.4 and 45.5; n = 13 64 slots 12.9 and 12.0, 301 32.9 and
// 32.3; n = 15 64 slots 38.0 and 35.7, 512 226 and 222; 7 of n = 18 41.2 and 39.1; one candidate of
// n = 18 19.1 and 16.4.
__host__ __device__ constexpr int f64_row_loge(int logg) { return logg <= 12 ? 3 : 4; }
__host__ __device__ constexpr uint32_t f64_row_words(int logg) { return (1u << logg) + (1u << (logg - f64_row_loge(logg))); }

// Between the LDS writes of a chunk and the next chunk's reads, YL the larger of their strides' logs: up
// to 6 the elements of a wave's 64 threads are the same run of residues in both chunks, and a
// wave's own accesses stay in order; beyond that the workgroup's threads meet.  (A thread writes
// back the very elements it has read, so nothing is needed between its reads and its writes.)
template <int YL>
__device__ __forceinline__ void f64_exchange() {
    if constexpr (YL <= 6) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    } else {
        __syncthreads();
    }
}

template <int LOGE>
__device__ __forceinline__ constexpr uint32_t f64_off(uint32_t rr, int YL) { return (rr << YL) + ((rr << YL) >> LOGE); }

// (a0..a3)^2 mod X^4 - w, operands reduced; results below 1.8 p.
__device__ __forceinline__ void f64_quad_square(const F64Mod &md, double &a0, double &a1, double &a2, double &a3, double w) {
    const double e0 = a0 + a0, e1 = a1 + a1, e2 = a2 + a2;
    const double t0 = md.mul(e1, a3) + md.mul(a2, a2);
    const double t1 = md.mul(e2, a3);
    const double t2 = md.mul(a3, a3);
    const double c0 = md.mul(a0, a0) + md.mul(t0, w);
    const double c1 = md.mul(e0, a1) + md.mul(t1, w);
    const double c2 = md.mul(e0, a2) + md.mul(a1, a1) + md.mul(t2, w);
    const double c3 = md.mul(e0, a3) + md.mul(e1, a2);
    a0 = c0; a1 = c1; a2 = c2; a3 = c3;
}

__device__ __forceinline__ void f64_quad_mul(const F64Mod &md, double &a0, double &a1, double &a2, double &a3,
                                             double z0, double z1, double z2, double z3, double w) {
    const double t0 = md.mul(a1, z3) + md.mul(a2, z2) + md.mul(a3, z1);
    const double t1 = md.mul(a2, z3) + md.mul(a3, z2);
    const double t2 = md.mul(a3, z3);
    const double c0 = md.mul(a0, z0) + md.mul(t0, w);
    const double c1 = md.mul(a0, z1) + md.mul(a1, z0) + md.mul(t1, w);
    const double c2 = md.mul(a0, z2) + md.mul(a1, z1) + md.mul(a2, z0) + md.mul(t2, w);
    const double c3 = md.mul(a0, z3) + md.mul(a1, z2) + (md.mul(a2, z1) + md.mul(a3, z0));
    a0 = c0; a1 = c1; a2 = c2; a3 = c3;
}

// The store of a row's result to `data`.
template <int E>
struct F64Store {
    double *data;
    template <class YL>
    __device__ __forceinline__ void operator()(const double (&x)[E], uint32_t base, YL) const {
#pragma unroll
        for (int rr = 0; rr < E; ++rr) data[base + ((uint32_t)rr << YL::value)] = x[rr];
    }
};

// load(x, base, YL): the first chunk's elements base + rr 2^YL, at most 0.52 p; store(x, base, YL): the same
// elements of the result (F64_FWD writes `data`).  `data` / `zp` at the
// row's first residue, `row` its index among the 2^a rows, L its LDS words.
template <class SZ, int LOGG, int LOGE, int MODE, class LD, class ST>
__device__ __forceinline__ void f64_row_pass(const F64Mod &md, const LD &load, const ST &store, double *__restrict__ data,
                                             const double *__restrict__ zp, const double *__restrict__ tw, int a,
                                             uint32_t row, uint32_t s, double *L, bool mul) {
    using GM = F64Geo<LOGG, LOGE>;
    constexpr int E = 1 << LOGE, LAST = GM::NCH - 1;
    static_assert(GM::NCH >= 2, "two chunks at least");
    // With 8 residues per thread a pass is bound by latency: a chunk's twiddles are on their way while the
    // chunk before it is computed (with 16 the registers go to more waves).
    constexpr bool AHEAD = LOGE <= 3;
    double x[E], w[E], wn[E];
    const auto twiddles = [&](auto cc, auto inv, double (&v)[E]) {
        constexpr int ci = decltype(cc)::value;
        constexpr int lam0 = GM::lam0(ci), NE = ci == LAST ? LOGE - 2 : GM::ne(ci), YL = GM::ylog(ci);
        // a wave's 64 threads lie in one sub-transform of this level (and in one row)
        constexpr bool UNI = YL >= 6;
        const uint32_t J = (row << lam0) + (s >> YL);
        if constexpr (decltype(inv)::value) f64_inv_tw<LOGE, UNI>(v, tw, (uint32_t)(a + lam0), J, NE);
        else f64_fwd_tw<LOGE, UNI>(v, tw, (uint32_t)(a + lam0), J, NE);
    };
    const auto next = [&]() {
#pragma unroll
        for (int i = 0; i < E; ++i) w[i] = wn[i];
    };
    if constexpr (AHEAD) twiddles(std::integral_constant<int, 0>{}, std::false_type{}, w);
    f64_for<0, GM::NCH>([&](auto cc) {
        constexpr int ci = decltype(cc)::value;
        constexpr int lam0 = GM::lam0(ci), NE = ci == LAST ? LOGE - 2 : GM::ne(ci), YL = GM::ylog(ci);
        const uint32_t hi = s >> YL, base = (hi << (LOGG - lam0)) + (s & ((1u << YL) - 1u));
        if constexpr (!AHEAD) twiddles(cc, std::false_type{}, w);
        else if constexpr (ci != LAST) twiddles(std::integral_constant<int, ci + 1>{}, std::false_type{}, wn);
        else twiddles(cc, std::true_type{}, wn);
        if constexpr (ci == 0) {
            load(x, base, std::integral_constant<int, YL>{});
        } else {
            f64_exchange<GM::ylog(ci - 1)>();
            const double *p = L + base + (base >> LOGE);
#pragma unroll
            for (int rr = 0; rr < E; ++rr) x[rr] = p[f64_off<LOGE>(rr, YL)];
        }
        f64_fwd_chunk<LOGE, NE>(md, x, w);
        if constexpr (ci != LAST) {
            double *p = L + base + (base >> LOGE);
#pragma unroll
            for (int rr = 0; rr < E; ++rr) p[f64_off<LOGE>(rr, YL)] = x[rr];
            if constexpr (AHEAD) next();
        }
    });
    if constexpr (SZ::reduce || MODE == F64_FWD) {
#pragma unroll
        for (int rr = 0; rr < E; ++rr) x[rr] = md.red(x[rr]);
    }
    const uint32_t base_last = s << LOGE;
    if constexpr (MODE == F64_FWD) {
#pragma unroll
        for (int rr = 0; rr < E; rr += 2)
            *reinterpret_cast<double2 *>(data + base_last + rr) = make_double2(x[rr], x[rr + 1]);
        return;
    } else {
        if (MODE == F64_SQUARE || (MODE == F64_EITHER && !mul)) {
#pragma unroll
            for (int i = 0; i < E / 4; ++i)
                f64_quad_square(md, x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3], (i & 1) ? -w[E / 8 + i / 2] : w[E / 8 + i / 2]);
        } else {
            const double2 *z = reinterpret_cast<const double2 *>(zp + base_last);
#pragma unroll
            for (int i = 0; i < E / 4; ++i) {
                const double2 za = z[2 * i], zb = z[2 * i + 1];
                f64_quad_mul(md, x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3], za.x, za.y, zb.x, zb.y,
                             (i & 1) ? -w[E / 8 + i / 2] : w[E / 8 + i / 2]);
            }
            // a product's coefficients reach 2.4 p
            if constexpr (SZ::reduce) {
#pragma unroll
                for (int rr = 0; rr < E; ++rr) x[rr] = md.red(x[rr]);
            }
        }
        f64_for_down<0, GM::NCH>([&](auto cc) {
            constexpr int ci = decltype(cc)::value;
            constexpr int lam0 = GM::lam0(ci), NE = ci == LAST ? LOGE - 2 : GM::ne(ci), YL = GM::ylog(ci);
            const uint32_t hi = s >> YL, base = (hi << (LOGG - lam0)) + (s & ((1u << YL) - 1u));
            if constexpr (!AHEAD) twiddles(cc, std::true_type{}, w);
            else {
                next();
                if constexpr (ci > 0) twiddles(std::integral_constant<int, ci - 1>{}, std::true_type{}, wn);
            }
            if constexpr (ci != LAST) {
                f64_exchange<YL>();
                const double *p = L + base + (base >> LOGE);
#pragma unroll
                for (int rr = 0; rr < E; ++rr) x[rr] = p[f64_off<LOGE>(rr, YL)];
            }
            f64_inv_chunk<SZ, LOGE, NE, ci == LAST, true>(md, x, w);
            if constexpr (ci == 0) {
                store(x, base, std::integral_constant<int, YL>{});
            } else {
                double *p = L + base + (base >> LOGE);
#pragma unroll
                for (int rr = 0; rr < E; ++rr) p[f64_off<LOGE>(rr, YL)] = x[rr];
            }
        });
    }
}

// ---------------------------------------------------------------------------------------------
// Column passes: 16 adjacent columns of the 2^LOGG x C matrix of limbs per workgroup, thread t ->
// column q = t mod 16 and sub-transform s = t / 16 of 2^LOGE residues; LDS element (k, q) at
// 16 k + q (conflict-free).

// Limb mod p: as it is, or reduced to 0.52 p.
__device__ __forceinline__ double f64_limb(const F64Mod &md, int32_t d0, int32_t d1, double bd, bool reduce) {
    const double e0 = (double)d0, e1 = (double)d1;
    if (!reduce) return fma(e1, bd, e0);
    const double h = e1 * bd, l = fma(e1, bd, -h);
    return fma(-rint(h * md.pinv), md.p, h) + (l + e0);
}

// The group's digit pairs with the range carries of the last normalisation added (ls: the carry
// into range k C / 16 + blk is (u0, u1, v): (u0, u1) on the digits of limb 0, v on digit 0 of limb 1).
template <int LOGE, int LOGG>
__device__ __forceinline__ void f64_load_digits(int2 (&d)[1 << LOGE], const int32_t *__restrict__ src,
                                                const int4 *__restrict__ ls, uint32_t C, unsigned blk, uint32_t t) {
    constexpr int E = 1 << LOGE, YL = LOGG - LOGE;
    const uint32_t q = t & 15u, s = t >> 4;
    const int2 *g = reinterpret_cast<const int2 *>(src) + (size_t)blk * 16 + q;
#pragma unroll
    for (int rr = 0; rr < E; ++rr) d[rr] = g[(size_t)(s + ((uint32_t)rr << YL)) * C];
    if (ls && q < 2) {
        const int2 *c = reinterpret_cast<const int2 *>(ls + blk) + q;
        int2 e[E];
#pragma unroll
        for (int rr = 0; rr < E; ++rr) e[rr] = c[(size_t)(s + ((uint32_t)rr << YL)) * (C / 8)];
#pragma unroll
        for (int rr = 0; rr < E; ++rr) {
            d[rr].x += e[rr].x;
            d[rr].y += q == 0 ? e[rr].y : 0;
        }
    }
}

// limb(rr): residue of the limb in row s + rr 2^(LOGG - LOGE).
template <int LOGE, int LOGG, class LD>
__device__ __forceinline__ void f64_col_fwd(const F64Mod &md, const LD &limb, double *__restrict__ dst,
                                            const double *__restrict__ tw, uint32_t C, unsigned blk, uint32_t t,
                                            double *lds) {
    using GM = F64Geo<LOGG, LOGE>;
    constexpr int E = 1 << LOGE;
    const uint32_t q = t & 15u, s = t >> 4;
    double x[E], w[E], wn[E];
    const auto twiddles = [&](auto cc, double (&v)[E]) {
        constexpr int ci = decltype(cc)::value;
        constexpr bool UNI = GM::ylog(ci) >= 2;  // a wave holds four consecutive s
        f64_fwd_tw<LOGE, UNI>(v, tw, (uint32_t)GM::lam0(ci), s >> GM::ylog(ci), GM::ne(ci));
    };
    twiddles(std::integral_constant<int, 0>{}, w);
    f64_for<0, GM::NCH>([&](auto cc) {
        constexpr int ci = decltype(cc)::value;
        constexpr int lam0 = GM::lam0(ci), NE = GM::ne(ci), YL = GM::ylog(ci);
        const uint32_t hi = s >> YL, base = (hi << (LOGG - lam0)) + (s & ((1u << YL) - 1u));
        if constexpr (ci + 1 < GM::NCH) twiddles(std::integral_constant<int, ci + 1>{}, wn);
        if constexpr (ci == 0) {
#pragma unroll
            for (int rr = 0; rr < E; ++rr) x[rr] = limb(rr);
        } else {
            __syncthreads();
            const double *p = lds + base * 16 + q;
#pragma unroll
            for (int rr = 0; rr < E; ++rr) x[rr] = p[(uint32_t)rr << (YL + 4)];
        }
        f64_fwd_chunk<LOGE, NE>(md, x, w);
        if constexpr (ci == GM::NCH - 1) {
            double *o = dst + (size_t)blk * 16 + q;
#pragma unroll
            for (int rr = 0; rr < E; ++rr) o[(size_t)(base + ((uint32_t)rr << YL)) * C] = x[rr];
        } else {
            if constexpr (ci == 0) __syncthreads();  // the previous prime's last reads
            double *p = lds + base * 16 + q;
#pragma unroll
            for (int rr = 0; rr < E; ++rr) p[(uint32_t)rr << (YL + 4)] = x[rr];
#pragma unroll
            for (int i = 0; i < E; ++i) w[i] = wn[i];
        }
    });
}

// Loads a column group's residues in the layout of the first inverse chunk (the last forward one).
template <int LOGE, int LOGG>
__device__ __forceinline__ void f64_col_load(double (&x)[1 << LOGE], const double *__restrict__ ws, uint32_t C,
                                             unsigned blk, uint32_t t) {
    constexpr int E = 1 << LOGE;
    const uint32_t q = t & 15u, s = t >> 4;
    const double *g = ws + (size_t)blk * 16 + q;
#pragma unroll
    for (int rr = 0; rr < E; ++rr) x[rr] = g[(size_t)((s << LOGE) + rr) * C];
}

// Inverse column levels on x (f64_col_load's layout in, the first forward chunk's out: rows
// s + rr 2^(LOGG - LOGE)).
template <class SZ, int LOGE, int LOGG>
__device__ __forceinline__ void f64_col_inv(const F64Mod &md, double (&x)[1 << LOGE], const double *__restrict__ tw,
                                            uint32_t t, double *lds) {
    using GM = F64Geo<LOGG, LOGE>;
    constexpr int E = 1 << LOGE;
    const uint32_t q = t & 15u, s = t >> 4;
    double w[E], wn[E];
    const auto twiddles = [&](auto cc, double (&v)[E]) {
        constexpr int ci = decltype(cc)::value;
        f64_inv_tw<LOGE, (GM::ylog(ci) >= 2)>(v, tw, (uint32_t)GM::lam0(ci), s >> GM::ylog(ci), GM::ne(ci));
    };
    twiddles(std::integral_constant<int, GM::NCH - 1>{}, w);
    f64_for_down<0, GM::NCH>([&](auto cc) {
        constexpr int ci = decltype(cc)::value;
        constexpr int lam0 = GM::lam0(ci), NE = GM::ne(ci), YL = GM::ylog(ci);
        const uint32_t hi = s >> YL, base = (hi << (LOGG - lam0)) + (s & ((1u << YL) - 1u));
        if constexpr (ci > 0) twiddles(std::integral_constant<int, ci - 1>{}, wn);
        if constexpr (ci != GM::NCH - 1) {
            __syncthreads();
            const double *p = lds + base * 16 + q;
#pragma unroll
            for (int rr = 0; rr < E; ++rr) x[rr] = p[(uint32_t)rr << (YL + 4)];
        }
        f64_inv_chunk<SZ, LOGE, NE, false, (ci != 0)>(md, x, w);
        if constexpr (ci != 0) {
            if constexpr (ci == GM::NCH - 1) __syncthreads();  // the previous prime's last reads
            double *p = lds + base * 16 + q;
#pragma unroll
            for (int rr = 0; rr < E; ++rr) p[(uint32_t)rr << (YL + 4)] = x[rr];
#pragma unroll
            for (int i = 0; i < E; ++i) w[i] = wn[i];
        }
    });
}

template <bool FIRST, class T>
__device__ __forceinline__ T &f64_either(T &a, T &b) {
    if constexpr (FIRST) return a;
    else return b;
}

// f64_col_load and f64_col_inv on x[k] of prime k, mod(k), for K primes as a pipeline: step d runs chunk
// NCH - 1 - i of prime d - i for every i, from LDS buffer (prime mod NCH), and one barrier ends
// the step.  (A buffer's last reads, in a prime's last chunk, are a step before the writes of
// the prime that takes it over.)  K + NCH - 2 barriers instead of 2 K (NCH - 1), and up to NCH
// independent chains between them; residues at ws + k M, twiddles at tw + k tws.  The first chunk's twiddles
// differ within a wave and are vector loads, each prime's before its residues': a wait for them
// would else include the residues of all.
template <class SZ, int K, int LOGE, int LOGG, class MD>
__device__ __forceinline__ void f64_cols_inv(const MD &mod, double (&x)[K][1 << LOGE], const double *__restrict__ ws,
                                             size_t M, const double *__restrict__ tw, size_t tws, uint32_t C,
                                             unsigned blk, uint32_t t, double *lds) {
    using GM = F64Geo<LOGG, LOGE>;
    constexpr int E = 1 << LOGE, NCH = GM::NCH;
    const uint32_t q = t & 15u, s = t >> 4;
    double wl[K][E];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        f64_inv_tw<LOGE, false>(wl[k], tw + k * tws, (uint32_t)GM::lam0(NCH - 1), s, GM::ne(NCH - 1));
        f64_col_load<LOGE, LOGG>(x[k], ws + k * M, C, blk, t);
    }
    f64_for<0, K + NCH - 1>([&](auto dd) {
        constexpr int d = decltype(dd)::value;
        f64_for<0, NCH>([&](auto cc) {
            constexpr int ci = decltype(cc)::value, k = d - (NCH - 1 - ci);
            if constexpr (k >= 0 && k < K) {
                constexpr int lam0 = GM::lam0(ci), NE = GM::ne(ci), YL = GM::ylog(ci);
                const uint32_t hi = s >> YL, base = (hi << (LOGG - lam0)) + (s & ((1u << YL) - 1u));
                double v[E], *p = lds + (k % NCH) * (16u << LOGG) + base * 16 + q;
                constexpr bool UNI = YL >= 2;
                if constexpr (UNI) {
                    f64_inv_tw<LOGE, UNI>(v, tw + k * tws, (uint32_t)lam0, hi, NE);
                }
                auto &w = f64_either<UNI>(v, wl[k]);
                if constexpr (ci != NCH - 1) {
#pragma unroll
                    for (int rr = 0; rr < E; ++rr) x[k][rr] = p[(uint32_t)rr << (YL + 4)];
                }
                f64_inv_chunk<SZ, LOGE, NE, false, (ci != 0)>(mod(k), x[k], w);
                if constexpr (ci != 0) {
#pragma unroll
                    for (int rr = 0; rr < E; ++rr) p[(uint32_t)rr << (YL + 4)] = x[k][rr];
                }
            }
        });
        if constexpr (d < K + NCH - 2) __syncthreads();
    });
}

// ---------------------------------------------------------------------------------------------
// CRT and carry

// The low 32 bits of the integer-valued double v, |v| < 2^51.
__device__ __forceinline__ uint32_t f64_lo(double v) {
    return (uint32_t)__double2loint(v + 0x1.8p52);
}

// One base-b digit of the exact sum known as the double S and mod 2^32: the piece S - q b, and the
// quotient in q / ql.
__device__ __forceinline__ int32_t f64_piece(double S, uint32_t Sl, const double binv, const uint32_t b, double &q,
                                             uint32_t &ql) {
    q = rint(S * binv);
    ql = f64_lo(q);
    return (int32_t)(Sl - ql * b);
}

// Base-b pieces g[0..4] of the coefficient with raw residues r[0..K-1].
template <int K>
__device__ __forceinline__ void f64_crt_pieces(F64CrtP c, const double (&r)[K], int dup, int32_t (&g)[5]) {
    const F64Mod m0{c->p[0], c->pinv[0]}, m1{c->p[1], c->pinv[1]};
    const double binv = c->binv;
    const uint32_t b = c->b;
    const double v1 = m0.mul(r[0], c->s[dup][0]);
    const double v2 = m1.mul(m1.mul(r[1], c->s[dup][1]) - v1, c->i12);
    const uint32_t v1l = f64_lo(v1), v2l = f64_lo(v2);
    double q;
    uint32_t ql;
    if constexpr (K == 2) {
        g[0] = f64_piece(fma(v2, c->w1[0], v1), v1l + v2l * c->w1l[0], binv, b, q, ql);
#pragma unroll
        for (int i = 1; i < 4; ++i) g[i] = f64_piece(fma(v2, c->w1[i], q), ql + v2l * c->w1l[i], binv, b, q, ql);
        g[4] = (int32_t)(ql + v2l * c->w1l[4]);
    } else {
        const F64Mod m2{c->p[2], c->pinv[2]};
        const double v3 = m2.mul(m2.mul(m2.mul(r[2], c->s[dup][2]) - v1, c->i13) - v2, c->i23);
        const uint32_t v3l = f64_lo(v3);
        g[0] = f64_piece(fma(v3, c->w2[0], fma(v2, c->w1[0], v1)), v1l + v2l * c->w1l[0] + v3l * c->w2l[0], binv, b, q, ql);
#pragma unroll
        for (int i = 1; i < 3; ++i)  // p1 has three pieces: b^3 > 2^49 wherever three primes are needed
            g[i] = f64_piece(fma(v3, c->w2[i], fma(v2, c->w1[i], q)), ql + v2l * c->w1l[i] + v3l * c->w2l[i], binv, b, q, ql);
        g[3] = f64_piece(fma(v3, c->w2[3], q), ql + v3l * c->w2l[3], binv, b, q, ql);
        g[4] = (int32_t)(ql + v3l * c->w2l[4]);
    }
}

// The value of the lane D below within its row of 16 lanes (0 past the row's start).
template <int D>
__device__ __forceinline__ int32_t f64_lane_below(int32_t v) {
    return __builtin_amdgcn_update_dpp(0, v, 0x110 + D, 0xF, 0xF, false);
}

// Limb of lane q (16 lanes = 16 consecutive limbs) from its pieces and those of the two limbs
// below: two digits, balanced but for the carry of the lane below (at most 4) added to the first,
// and in lane 15 what goes on to the next range: (g2 + g4 of lane 14 + carry, g3, g4).
__device__ __forceinline__ int2 f64_limb_digits(F64CrtP c, const int32_t (&g)[5], int4 &out) {
    const double bd = c->bd, binv = c->binv, qb = c->qb;
    const int32_t g4b = f64_lane_below<1>(g[4]);
    const double D0 = (double)g[0] + (double)(f64_lane_below<1>(g[2]) + f64_lane_below<1>(g4b));
    const double q0 = rint(fma(D0, binv, -qb));  // balanced: ties go down (D - 1/4 is no tie)
    const double d0 = fma(-q0, bd, D0);
    const double D1 = (double)g[1] + (double)f64_lane_below<1>(g[3]) + q0;
    const double q1 = rint(fma(D1, binv, -qb));
    const double d1 = fma(-q1, bd, D1);
    const int32_t cr = (int32_t)q1;
    out = make_int4(g[2] + g4b + cr, g[3], g[4], 0);
    return make_int2((int32_t)d0 + f64_lane_below<1>(cr), (int32_t)d1);
}

// Digits of limb i (lane i mod 16 of its range of 16) from its raw residues, stored with the carry into
// the next range.
template <int K>
__device__ __forceinline__ void f64_norm_limb(F64CrtP c, const double (&r)[K], int dup, uint32_t i, uint32_t M,
                                              int32_t *__restrict__ dst, int4 *__restrict__ slots) {
    int32_t g[5];
    f64_crt_pieces<K>(c, r, dup, g);
    int4 u;
    reinterpret_cast<int2 *>(dst)[i] = f64_limb_digits(c, g, u);
    if ((i & 15u) == 15u) {
        // within b / 2: the digit sums of the next pass stay below 2^31
        const double U = (double)u.x, a = rint(fma(U, c->binv, -c->qb));
        u.x = (int32_t)fma(-a, c->bd, U);
        u.y += (int32_t)a;
        uint32_t w = (i >> 4) + 1;
        if (w == M / 16) { w = 0; u.x = -u.x; u.y = -u.y; u.z = -u.z; }  // B^M = -1
        slots[w] = u;
    }
}

// A column workgroup's limbs: thread t holds rows s + rr 2^YL, column q of its 16 columns.
template <int K, int LOGE, int LOGG>
__device__ __forceinline__ void f64_norm_store(F64CrtP c, const double (&x)[K][1 << LOGE], uint32_t C, unsigned blk,
                                               uint32_t t, int dup, int32_t *__restrict__ dst, int4 *__restrict__ slots) {
    constexpr int E = 1 << LOGE, YL = LOGG - LOGE;
    const uint32_t q = t & 15u, s = t >> 4;
#pragma unroll
    for (int rr = 0; rr < E; ++rr) {
        double r[K];
#pragma unroll
        for (int i = 0; i < K; ++i) r[i] = x[i][rr];
        f64_norm_limb<K>(c, r, dup, (s + ((uint32_t)rr << YL)) * C + blk * 16 + q, C << LOGG, dst, slots);
    }
}

// Digits of range w (32 digits from 32 w of src) with their range carry, balanced, to the same place of
// dst (STORE); returns the carry out.  All are loaded before the first is stored: in turn (src may be
// dst) each load waited for memory by itself: a squaring and a copy out 14.3 us at n = 14, not 13.1, 81.2
// at n = 22, not 79.8.
template <bool STORE = true>
__device__ __forceinline__ int32_t f64_flush_range(const int32_t *src, int32_t *dst, const int4 *slots, uint32_t b, uint32_t w) {
    const double bd = (double)b, binv = 1.0 / bd, qb = 0.25 * binv;
    const int4 v = slots[w];
    const int4 *p = reinterpret_cast<const int4 *>(src + (size_t)w * 32);
    int4 *o = reinterpret_cast<int4 *>(dst + (size_t)w * 32);
    int4 in[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) in[i] = p[i];
    double c = 0.0;
    auto digit = [&](int32_t d, int32_t e) -> int32_t {
        const double D = (double)d + (double)e + c;
        c = rint(fma(D, binv, -qb));
        return (int32_t)fma(-c, bd, D);
    };
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        int4 x = in[i];
        x.x = digit(x.x, i == 0 ? v.x : 0);
        x.y = digit(x.y, i == 0 ? v.y : 0);
        x.z = digit(x.z, i == 0 ? v.z : 0);
        x.w = digit(x.w, 0);
        if constexpr (STORE) o[i] = x;
    }
    return (int32_t)c;
}

// In place: the carry out stays in slots[w].w (which no pass reads) for f64_carry_body, which adds it to
// the range above once every range is done; the range carry is cleared.
__device__ __forceinline__ void f64_flush_body(int32_t *dst, int4 *slots, uint32_t b, uint32_t w) {
    slots[w] = make_int4(0, 0, 0, f64_flush_range(dst, dst, slots, b, w));
}

// A carry c into balanced digits p[0..N-1], N digits of a range.
template <int N>
__device__ __forceinline__ void f64_carry_digits(int32_t *p, int32_t c, uint32_t b) {
    if (c == 0) return;
    const int32_t hi = (int32_t)(b / 2), lo = -(int32_t)((b - 1) / 2);
    for (int i = 0; i < N - 1 && c != 0; ++i) {
        int32_t d = p[i] + c;
        c = (d > hi) - (d < lo);
        p[i] = d - c * (int32_t)b;
    }
    if (c) p[N - 1] += c;
}

// Register 0 with its pending range carries, balanced, to dst, in one launch; the register and its carries
// stay as they are.  F64_FLUSH_R ranges of N digits a workgroup, range(std::bool_constant<STORE>, w) one of
// them; a wave of its own works out the carry out of the range below again.
constexpr uint32_t F64_FLUSH_R = 64;
template <int N, class R>
__device__ __forceinline__ void f64_flush_to_body(const R &range, int32_t *dst, uint32_t nrange, uint32_t b) {
    __shared__ int32_t cs[F64_FLUSH_R + 1];
    const uint32_t t = threadIdx.x, w0 = blockIdx.x * F64_FLUSH_R, w = w0 + t;
    if (t < F64_FLUSH_R) {
        cs[t + 1] = range(std::true_type{}, w);
    } else if (t == F64_FLUSH_R) {
        const int32_t c = range(std::false_type{}, w0 == 0 ? nrange - 1 : w0 - 1);
        cs[0] = w0 == 0 ? -c : c;  // B^M = -1
    }
    __syncthreads();
    if (t < F64_FLUSH_R) f64_carry_digits<N>(dst + (size_t)w * N, cs[t], b);
}

__device__ __forceinline__ void f64_carry_body(int32_t *dst, const int4 *slots, uint32_t nrange, uint32_t b, uint32_t w) {
    f64_carry_digits<32>(dst + (size_t)w * 32, w == 0 ? -slots[nrange - 1].w : slots[w - 1].w, b);
}

}  // namespace gfe
