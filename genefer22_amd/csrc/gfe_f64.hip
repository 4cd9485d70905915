// gfe_f64.hip -- kernels and host constants of the double-precision limb transform (gfe_f64.h).
//
// One squaring is three launches: forward column pass (digits -> residues of every prime), row pass
// (forward, square, inverse), inverse column pass with the CRT and the carry; or, up to 2^12 limbs,
// two: the whole transform of each prime, then the CRT and the carry.
#include "gfe_f64_host.h"

#include <cstring>
#include <mutex>

namespace gfe {

// Work of workgroup blockIdx.x of a launch of `per` workgroups a slot: slot and index within it.  Slots
// follow each other, or with pin slot s takes workgroups of XCD s mod 8 only (workgroups go to the 8
// XCDs in turn).
struct F64Job {
    uint32_t slot, w;
    F64CrtP c;
    int K;
    bool run;
};
__device__ __forceinline__ F64Job f64_job(const F64Args &A, uint32_t per) {
    F64Job J;
    const uint32_t id = blockIdx.x;
    if (A.K) {
        J.slot = 0; J.w = id; J.c = (F64CrtP)A.crt; J.K = A.K; J.run = true;
        return J;
    }
    if (A.pin) {
        const uint32_t i = id >> 3, g = i / per;
        J.slot = (g << 3) + (id & 7u);
        J.w = i - g * per;
    } else {
        J.slot = id / per;
        J.w = id - J.slot * per;
    }
    J.run = J.slot < A.nslots && !(A.active && !A.active[J.slot]);
    J.c = (F64CrtP)A.crt + (J.run ? J.slot : 0);
    J.K = J.c->K;
    return J;
}
// Column block of index x of nb (XCD by XCD, unless the slot is on one).
__device__ __forceinline__ unsigned f64_block(const F64Args &A, unsigned x, unsigned nb) { return A.pin ? x : xcd_block(x, nb); }

// C / 16 workgroups a slot, or with `split` one per column block and prime: 16 columns for all primes
// from one read of the digits, or for one.
template <int LOGG>
__global__ void __launch_bounds__(16 << (LOGG - F64_COL_E)) k64_col_fwd(F64Args A, int split) {
    extern __shared__ double lds64[];
    constexpr int LOGE = F64_COL_E;
    const uint32_t M = 1u << A.tn, C = M >> LOGG, nb = C / 16, t = threadIdx.x;
    const F64Job J = f64_job(A, split ? 3 * nb : nb);
    if (!J.run) return;
    const F64CrtP c = J.c;
    const int K = J.K, k0 = split ? (int)(J.w / nb) : 0, k1 = split ? k0 + 1 : K;
    if (k0 >= K) return;
    const unsigned blk = f64_block(A, split ? J.w - k0 * nb : J.w, nb);
    int2 d[1 << LOGE];
    f64_load_digits<LOGE, LOGG>(d, A.regs + J.slot * A.reg_stride + (size_t)A.src_reg * (2u << A.tn),
                                A.absorb ? A.slots + J.slot * A.slot_stride : nullptr, C, blk, t);
    const double bd = c->bd;
    const bool reduce = c->big == 2;
    double *ws = A.ws + J.slot * A.ws_stride;
#pragma unroll 1
    for (int k = k0; k < k1; ++k) {
        const F64Mod md{c->p[k], c->pinv[k]};
        const auto limb = [&](int rr) { return f64_limb(md, d[rr].x, d[rr].y, bd, reduce); };
        f64_col_fwd<LOGE, LOGG>(md, limb, ws + (size_t)k * M, A.tw + (size_t)k * A.tws, C, blk, t, lds64);
    }
}

constexpr int f64_row_threads(int logg) { return logg > 11 ? 1 << (logg - f64_row_loge(logg)) : 256; }

// 3 2^a / ng workgroups a slot.
template <int LOGG, int MODE>
__global__ void __launch_bounds__(f64_row_threads(LOGG)) k64_row(F64Args A) {
    extern __shared__ double lds64[];
    constexpr int LOGE = f64_row_loge(LOGG);
    constexpr uint32_t SPR = 1u << (LOGG - LOGE);
    const uint32_t nb = (1u << A.a) / (uint32_t)A.ng;
    const F64Job J = f64_job(A, 3 * nb);
    const int k = (int)(J.w / nb);
    if (!J.run || k >= J.K) return;
    const uint32_t t = threadIdx.x, q = t / SPR, s = t % SPR;
    uint32_t row = (J.w - (uint32_t)k * nb) * (uint32_t)A.ng + q;
    if constexpr (SPR >= 64) row = __builtin_amdgcn_readfirstlane(row);
    const size_t at = J.slot * A.ws_stride + ((size_t)k << A.tn) + ((size_t)row << LOGG);
    const F64Mod md{J.c->p[k], J.c->pinv[k]};
    double *data = A.ws + at;
    const auto load = [&](double (&x)[1 << LOGE], uint32_t base, auto yl) {
#pragma unroll
        for (int rr = 0; rr < 1 << LOGE; ++rr) x[rr] = data[base + ((uint32_t)rr << decltype(yl)::value)];
#pragma unroll
        for (int rr = 0; rr < 1 << LOGE; ++rr) x[rr] = md.red(x[rr]);
    };
    f64_row_pass<F64Wide, LOGG, LOGE, MODE>(md, load, F64Store<1 << LOGE>{data}, data, A.zp + at, A.tw + (size_t)k * A.tws, A.a, row, s,
                                            lds64 + q * f64_row_words(LOGG),
                                            MODE == F64_EITHER && A.mulf && A.mulf[J.slot]);
}

// A prime's whole transform, from the digits, in one workgroup; thread s of
// 2^(LOGG - f64_row_loge(LOGG)).
template <int LOGG, int MODE>
__device__ __forceinline__ void f64_whole_body(const F64Args &A, const F64Job &J, int k, uint32_t s, double *lds) {
    constexpr int LOGE = f64_row_loge(LOGG), E = 1 << LOGE;
    const F64CrtP c = J.c;
    const F64Mod md{c->p[k], c->pinv[k]};
    const double bd = c->bd;
    const bool reduce = c->big != 0;
    const int2 *src = reinterpret_cast<const int2 *>(A.regs + J.slot * A.reg_stride + (size_t)A.src_reg * (2u << LOGG));
    const int4 *ls = A.absorb ? A.slots + J.slot * A.slot_stride : nullptr;
    const size_t at = J.slot * A.ws_stride + ((size_t)k << LOGG);
    const auto load = [&](double (&x)[E], uint32_t base, auto yl) {
        constexpr int YL = decltype(yl)::value;
        int2 d[E];
#pragma unroll
        for (int rr = 0; rr < E; ++rr) d[rr] = src[base + ((uint32_t)rr << YL)];
        if (ls && (base & 15u) < 2) {  // as f64_load_digits
            const uint32_t q = base & 1u;
            int2 e[E];
#pragma unroll
            for (int rr = 0; rr < E; ++rr) e[rr] = reinterpret_cast<const int2 *>(ls + ((base + ((uint32_t)rr << YL)) >> 4))[q];
#pragma unroll
            for (int rr = 0; rr < E; ++rr) {
                d[rr].x += e[rr].x;
                d[rr].y += q == 0 ? e[rr].y : 0;
            }
        }
#pragma unroll
        for (int rr = 0; rr < E; ++rr) x[rr] = f64_limb(md, d[rr].x, d[rr].y, bd, reduce);
    };
    f64_row_pass<F64Wide, LOGG, LOGE, MODE>(md, load, F64Store<E>{A.ws + at}, A.ws + at, A.zp + at, A.tw + (size_t)k * A.tws, 0, 0, s, lds,
                                            MODE == F64_EITHER && A.mulf && A.mulf[J.slot]);
}

// 3 workgroups a slot.
template <int LOGG, int MODE>
__global__ void __launch_bounds__(1 << (LOGG - f64_row_loge(LOGG))) k64_whole(F64Args A) {
    extern __shared__ double lds64[];
    const F64Job J = f64_job(A, 3);
    if (J.run && (int)J.w < J.K) f64_whole_body<LOGG, MODE>(A, J, (int)J.w, threadIdx.x, lds64);
}

// A mixed batch: each workgroup at its slot's n, 12 or 13 (of the 512 threads n = 12 takes four whole
// waves; the others end before any barrier).
template <int MODE>
__global__ void __launch_bounds__(512) k64_whole_mixed(F64Args A) {
    extern __shared__ double lds64[];
    const F64Job J = f64_job(A, 3);
    if (!J.run || (int)J.w >= J.K) return;
    if (J.c->n == 13) f64_whole_body<12, MODE>(A, J, (int)J.w, threadIdx.x, lds64);
    else if (threadIdx.x < 256) f64_whole_body<11, MODE>(A, J, (int)J.w, threadIdx.x, lds64);
}

// A slot's whole squaring in one workgroup: the primes one after the other, each thread keeping its limbs'
// residues, then the CRT and the carry (the digits and range carries are read by every thread before the
// first exchange's barrier, so before any is written).
template <int K, int LOGG>
__device__ __forceinline__ void f64_all_body(const F64Args &A, const F64Job &J, double *lds) {
    constexpr int LOGE = f64_row_loge(LOGG), E = 1 << LOGE, YL = LOGG - LOGE;
    const F64CrtP c = J.c;
    const uint32_t s = threadIdx.x;
    const double bd = c->bd;
    const bool reduce = c->big != 0;
    int32_t *regs = A.regs + J.slot * A.reg_stride;
    int4 *slots = A.slots + J.slot * A.slot_stride;
    int2 d[E];
#pragma unroll
    for (int rr = 0; rr < E; ++rr) d[rr] = reinterpret_cast<const int2 *>(regs)[s + ((uint32_t)rr << YL)];
    if ((s & 15u) < 2) {  // as f64_load_digits
        const uint32_t q = s & 1u;
        int2 e[E];
#pragma unroll
        for (int rr = 0; rr < E; ++rr) e[rr] = reinterpret_cast<const int2 *>(slots + ((s + ((uint32_t)rr << YL)) >> 4))[q];
#pragma unroll
        for (int rr = 0; rr < E; ++rr) {
            d[rr].x += e[rr].x;
            d[rr].y += q == 0 ? e[rr].y : 0;
        }
    }
    double x[K][E];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const F64Mod md{c->p[k], c->pinv[k]};
        const auto load = [&](double (&y)[E], uint32_t, auto) {
#pragma unroll
            for (int rr = 0; rr < E; ++rr) y[rr] = f64_limb(md, d[rr].x, d[rr].y, bd, reduce);
        };
        const auto store = [&](const double (&y)[E], uint32_t, auto) {
#pragma unroll
            for (int rr = 0; rr < E; ++rr) x[k][rr] = y[rr];
        };
        if (k) __syncthreads();  // the last prime's reads of lds
        f64_row_pass<F64Wide, LOGG, LOGE, F64_SQUARE>(md, load, store, nullptr, nullptr, A.tw + (size_t)k * A.tws, 0, 0, s,
                                                      lds, false);
    }
    const int dup = A.dupf ? (A.dupf[J.slot] != 0) : A.dup;
#pragma unroll
    for (int rr = 0; rr < E; ++rr) {
        double r[K];
#pragma unroll
        for (int k = 0; k < K; ++k) r[k] = x[k][rr];
        f64_norm_limb<K>(c, r, dup, s + ((uint32_t)rr << YL), 1u << LOGG, regs, slots);
    }
}

// One workgroup a slot.
template <int LOGG>
__global__ void __launch_bounds__(1 << (LOGG - f64_row_loge(LOGG))) k64_all(F64Args A) {
    extern __shared__ double lds64[];
    const F64Job J = f64_job(A, 1);
    if (!J.run) return;
    if (J.K == 2) f64_all_body<2, LOGG>(A, J, lds64);
    else f64_all_body<3, LOGG>(A, J, lds64);
}

template <int K, int LOGG>
__device__ __forceinline__ void f64_inv_body(const F64Args &A, const F64Job &J, int dup, double *lds) {
    constexpr int LOGE = F64_COL_E;
    const uint32_t M = 1u << A.tn, C = M >> LOGG, t = threadIdx.x;
    const unsigned blk = f64_block(A, J.w, C / 16);
    const double *ws = A.ws + J.slot * A.ws_stride;
    double x[K][1 << LOGE];
#pragma unroll
    for (int k = 0; k < K; ++k) f64_col_load<LOGE, LOGG>(x[k], ws + (size_t)k * M, C, blk, t);
#pragma unroll
    for (int k = 0; k < K; ++k)
        f64_col_inv<F64Wide, LOGE, LOGG>(F64Mod{J.c->p[k], J.c->pinv[k]}, x[k], A.tw + (size_t)k * A.tws, t, lds);
    f64_norm_store<K, LOGE, LOGG>(J.c, x, C, blk, t, dup, A.regs + J.slot * A.reg_stride,
                                  A.slots + J.slot * A.slot_stride);
}

// C / 16 workgroups a slot.
template <int LOGG>
__global__ void __launch_bounds__(16 << (LOGG - F64_COL_E)) k64_col_inv(F64Args A) {
    extern __shared__ double lds64[];
    const F64Job J = f64_job(A, (1u << A.tn) >> (LOGG + 4));
    if (!J.run) return;
    const int dup = A.dupf ? (A.dupf[J.slot] != 0) : A.dup;
    if (J.K == 2) f64_inv_body<2, LOGG>(A, J, dup, lds64);
    else f64_inv_body<3, LOGG>(A, J, dup, lds64);
}

// The inverse column pass with a candidate's primes side by side: K groups of 16 2^(LOGG - LOGE) threads,
// one prime each, then all threads over the limbs.  C / 16 workgroups a slot; a slot of two primes ends
// the third group before any barrier.
template <int K, int LOGG>
__device__ __forceinline__ void f64_inv_split_body(const F64Args &A, const F64Job &J, int dup, double *lds) {
    constexpr int LOGE = F64_COL_E, E = 1 << LOGE;
    constexpr uint32_t T = 16u << (LOGG - LOGE), LIMBS = 16u << LOGG;
    const F64CrtP c = J.c;
    const uint32_t M = 1u << A.tn, C = M >> LOGG;
    const int k = __builtin_amdgcn_readfirstlane(threadIdx.x / T);
    if (k >= K) return;
    const uint32_t t = threadIdx.x % T;
    const unsigned blk = f64_block(A, J.w, C / 16);
    double x[E], *L = lds + k * LIMBS;
    f64_col_load<LOGE, LOGG>(x, A.ws + J.slot * A.ws_stride + (size_t)k * M, C, blk, t);
    f64_col_inv<F64Wide, LOGE, LOGG>(F64Mod{c->p[k], c->pinv[k]}, x, A.tw + (size_t)k * A.tws, t, L);
#pragma unroll
    for (int rr = 0; rr < E; ++rr) L[((t >> 4) + ((uint32_t)rr << (LOGG - LOGE))) * 16 + (t & 15u)] = x[rr];
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < (LIMBS + K * T - 1) / (K * T); ++j) {
        const uint32_t i = threadIdx.x + j * K * T;
        if (i >= LIMBS) break;  // whole waves
        double r[K];
#pragma unroll
        for (int m = 0; m < K; ++m) r[m] = lds[m * LIMBS + i];
        f64_norm_limb<K>(c, r, dup, (i >> 4) * C + blk * 16 + (i & 15u), M, A.regs + J.slot * A.reg_stride,
                         A.slots + J.slot * A.slot_stride);
    }
}

// K: one candidate's primes (0.15 us a launch less than by the slot), or 0.
template <int K, int LOGG>
__global__ void __launch_bounds__(3 * (16 << (LOGG - F64_COL_E))) k64_col_inv_split(F64Args A) {
    extern __shared__ double lds64[];
    if constexpr (K != 0) {
        const F64Job J{0, blockIdx.x, (F64CrtP)A.crt, K, true};
        f64_inv_split_body<K, LOGG>(A, J, A.dup, lds64);
    } else {
        const F64Job J = f64_job(A, (1u << A.tn) >> (LOGG + 4));
        if (!J.run) return;
        const int dup = A.dupf ? (A.dupf[J.slot] != 0) : A.dup;
        if (J.K == 2) f64_inv_split_body<2, LOGG>(A, J, dup, lds64);
        else f64_inv_split_body<3, LOGG>(A, J, dup, lds64);
    }
}

template <int K>
__device__ __forceinline__ void f64_norm_body(const F64Args &A, const F64Job &J, uint32_t M, int dup) {
    const uint32_t i = J.w * F64_NORM_T + threadIdx.x;
    const double *ws = A.ws + J.slot * A.ws_stride;
    double r[K];
#pragma unroll
    for (int k = 0; k < K; ++k) r[k] = ws[(size_t)k * M + i];
    f64_norm_limb<K>(J.c, r, dup, i, M, A.regs + J.slot * A.reg_stride, A.slots + J.slot * A.slot_stride);
}

// The normalisation after k64_whole: M / F64_NORM_T workgroups a slot (a mixed batch's slots of the
// smaller n leave the rest idle).
__global__ void __launch_bounds__(F64_NORM_T) k64_norm(F64Args A) {
    const F64Job J = f64_job(A, (1u << A.tn) / F64_NORM_T);
    if (!J.run) return;
    const uint32_t M = A.K ? 1u << A.tn : 1u << (J.c->n - 1);
    if (J.w * F64_NORM_T >= M) return;
    const int dup = A.dupf ? (A.dupf[J.slot] != 0) : A.dup;
    if (J.K == 2) f64_norm_body<2>(A, J, M, dup);
    else f64_norm_body<3>(A, J, M, dup);
}

// Register 0 of the slots in grid.y with its pending range carries, balanced (f64_flush_body).
__global__ void __launch_bounds__(256) k64_flush(F64Args A) {
    const uint32_t s = blockIdx.y, w = blockIdx.x * 256u + threadIdx.x;
    if (A.active && !A.active[s]) return;
    const F64CrtP c = (F64CrtP)A.crt + s;
    if (c->n == 0 || w >= (1u << c->n) / 32) return;
    f64_flush_body(A.regs + s * A.reg_stride, A.slots + s * A.slot_stride, c->b, w);
}

__global__ void __launch_bounds__(256) k64_carry(F64Args A) {
    const uint32_t s = blockIdx.y, w = blockIdx.x * 256u + threadIdx.x;
    if (A.active && !A.active[s]) return;
    const F64CrtP c = (F64CrtP)A.crt + s;
    if (c->n == 0 || w >= (1u << c->n) / 32) return;
    f64_carry_body(A.regs + s * A.reg_stride, A.slots + s * A.slot_stride, (1u << c->n) / 32, c->b, w);
}

// One candidate's register 0 with its pending range carries, balanced, to dst: M / 16 / F64_FLUSH_R
// workgroups.  Copies, scalar products, waits and read-outs take it so: flushing in place takes two launches
// (a range's carry out may only be added once the range above it is done), which at n <= 16 was more
// than the squaring had gained on the integer passes.  us a squaring and the operation, flushed in place,
// here, and in integers, at n = 14: copy out 20.2, 13.1, 17.3; wait 28.0, 24.5, 26.9; scalar product 23.2,
// 19.2, 20.4; the Gerbicz-Li update (a product and three copies) 55.8, 36.1, 48.4.
__global__ void __launch_bounds__(2 * F64_FLUSH_R) k64_flush_to(F64Args A, uint32_t b, int32_t *dst) {
    const auto range = [&](auto st, uint32_t w) { return f64_flush_range<decltype(st)::value>(A.regs, dst, A.slots, b, w); };
    f64_flush_to_body<32>(range, dst, (1u << A.tn) / 16, b);
}

struct F64TwArgs {
    double *tw;
    uint32_t words;                       // per prime
    int bits;                             // log2 M
    double p[F64Q_PRIMES], pinv[F64Q_PRIMES];
    double pw[F64Q_PRIMES][22];           // psi^(2^i)
};

// Psi[j] = psi^bitrev(j): bit i of j contributes psi^(2^(bits - 1 - i)).
__global__ void __launch_bounds__(256) k64_twiddles(F64TwArgs A) {
    const uint32_t j = blockIdx.x * 256u + threadIdx.x;
    const int k = blockIdx.y;
    if (j >= A.words) return;
    const F64Mod md{A.p[k], A.pinv[k]};
    double w = 1.0;
    for (int i = 0; i < A.bits; ++i)
        if ((j >> i) & 1u) w = md.mul(w, A.pw[k][A.bits - 1 - i]);
    A.tw[(size_t)k * A.words + j] = w;
}

// ------------------------------------------------------------------------------------------------
// Host constants

static uint64_t mul64(uint64_t a, uint64_t b, uint64_t p) { return (uint64_t)((unsigned __int128)a * b % p); }
static uint64_t pow64(uint64_t a, uint64_t e, uint64_t p) {
    uint64_t r = 1;
    for (; e; e >>= 1, a = mul64(a, a, p))
        if (e & 1) r = mul64(r, a, p);
    return r;
}
uint64_t f64_inv_mod(uint64_t a, uint64_t p) { return pow64(a % p, p - 2, p); }
uint64_t f64_inv_pow2(int k, uint64_t p) {
    uint64_t s = 1;
    while (k-- > 0) s = ((s & 1) ? s + p : s) / 2;
    return s;
}
double f64_balanced(uint64_t a, uint64_t p) { return a > p / 2 ? -(double)(p - a) : (double)a; }

// Largest doubled coefficient against the primes' product.  Limbs are at most L = (b/2 + 4)(b + 1),
// but for the first two of a range of 16, which enter with the range carry added: the first's
// digits take |u0| <= b/2 and |u1| <= 0.55 b + G / b + 2, the second's low digit v <= G + 2, where
// G >= |g4| is the largest coefficient over b^4.  By Cauchy-Schwarz a doubled coefficient is at most
// X = 2 (M / 16)(L0^2 + L1^2 + 14 L^2), which gives G in turn: the pair is settled by iteration.
// Three primes need X < 0.3 P (the mixed-radix digit v3 is then the centred one, whatever the
// rounding of its quotient); with two the last digit's quotient has the larger rounding: 0.1 P.
static bool f64_bound(uint32_t b, uint32_t n, int K) {
    const long double bb = b, M = (long double)((uint64_t)1 << (n - 1));
    long double P = 1;
    for (int k = 0; k < K; ++k) P *= (long double)F64_P[k];
    const long double L = (bb / 2 + 4) * (bb + 1);
    long double G = M / 2 + 4, X = 0;
    for (int it = 0; it < 64; ++it) {
        const long double L0 = (bb + 5) + bb * (1.05L * bb + 6 + G / bb + 2), L1 = L + G + 2;
        X = 2 * (M / 16) * (L0 * L0 + L1 * L1 + 14 * L * L);
        const long double g = X / (bb * bb * bb * bb) + 4;
        if (g <= G) break;
        G = g * 1.001L;
        if (G > bb * bb || G > 1.0e8L) return false;
    }
    return G <= bb * bb && G <= 1.0e8L && X < (K == 3 ? 0.3L : 0.1L) * P;
}

int f64_primes(uint32_t b, uint32_t n) {
    if (n < 12 || n > 23 || b < 1024) return 0;
    if (f64_bound(b, n, 2)) return 2;
    // three primes: p1 in three base-b pieces
    return (b >= (1u << 17) && f64_bound(b, n, 3)) ? 3 : 0;
}

F64Crt make_f64_crt(uint32_t n, uint32_t b, int K) {
    F64Crt c;
    memset(&c, 0, sizeof(c));
    for (int k = 0; k < 3; ++k) {
        const uint64_t p = F64_P[k];
        c.p[k] = (double)p;
        c.pinv[k] = 1.0 / (double)p;
        // n - 3 of the transform's n - 1 levels are run and undone: 2^(n-3) comes out of the inverse
        const uint64_t s = f64_inv_pow2((int)n - 3, p);
        c.s[0][k] = f64_balanced(s, p);
        c.s[1][k] = f64_balanced(mul64(s, 2, p), p);
    }
    // the primes' inverses once: made with every base's constants they took 3 us, and 7 in make_f64q_crt, of a
    // rebase or submission
    static const double i12 = f64_balanced(f64_inv_mod(F64_P[0], F64_P[1]), F64_P[1]);
    static const double i13 = f64_balanced(f64_inv_mod(F64_P[0], F64_P[2]), F64_P[2]);
    static const double i23 = f64_balanced(f64_inv_mod(F64_P[1], F64_P[2]), F64_P[2]);
    c.i12 = i12; c.i13 = i13; c.i23 = i23;
    auto split = [&](__int128 x, int pieces, double *w, uint32_t *wl) {
        for (int i = 0; i < pieces; ++i) {
            __int128 r = x;
            if (i < pieces - 1) {
                r = x % b;
                if (r > b / 2) r -= b;
                x = (x - r) / b;
            }
            w[i] = (double)(int64_t)r;
            wl[i] = (uint32_t)(int64_t)r;
        }
    };
    split((__int128)F64_P[0], K == 3 ? 3 : 5, c.w1, c.w1l);
    if (K == 3) split((__int128)F64_P[0] * F64_P[1], 5, c.w2, c.w2l);
    c.bd = (double)b;
    c.binv = 1.0 / (double)b;
    c.qb = 0.25 * c.binv;
    c.b = b;
    const double limb = 1.1 * (double)b * (double)b + (double)((uint64_t)1 << n);  // range carry included
    c.big = limb > 0x1p50 ? 2 : limb > 0x1p48 ? 1 : 0;
    c.n = (int32_t)n;
    c.K = K;
    return c;
}

static int build_twiddles(const uint64_t *primes, const uint32_t *gen, int K, int bits, double *tw, hipStream_t stream) {
    F64TwArgs A;
    memset(&A, 0, sizeof(A));
    A.tw = tw;
    A.words = 1u << (bits - 2);
    A.bits = bits;
    for (int k = 0; k < K; ++k) {
        const uint64_t p = primes[k];
        A.p[k] = (double)p;
        A.pinv[k] = 1.0 / (double)p;
        uint64_t w = pow64(gen[k], (p - 1) >> (bits + 1), p);  // a primitive 2M-th root, M = 2^bits
        for (int i = 0; i < A.bits; ++i, w = mul64(w, w, p)) A.pw[k][i] = f64_balanced(w, p);
    }
    hipLaunchKernelGGL(k64_twiddles, dim3((A.words + 255) / 256, K, 1), dim3(256), 0, stream, A);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int f64_build_twiddles(uint32_t n, double *tw, hipStream_t stream) {
    return build_twiddles(F64_P, F64_G, F64_PRIMES, (int)n - 1, tw, stream);
}

int f64q_build_twiddles(uint32_t n, double *tw, hipStream_t stream) {
    return build_twiddles(F64Q_P, F64Q_G, F64Q_PRIMES, (int)n - 2, tw, stream);
}

// ------------------------------------------------------------------------------------------------
// Dispatch


// One candidate, timed on MI355X (us per squaring, three primes unless said).  Up to 2^12 limbs the
// two launches with a prime's transform in one workgroup beat the three (2^11 limbs 7.6 against
// 10.1, 2^12 9.7 against 10.6; at 2^13 one workgroup's arithmetic takes longer, 16.8 against 14.0;
// in batches 100 candidates of 2^13 limbs 32.8 against 31.6, 512 of 2^14 230 against 228).
// With three passes, up to 2^19 limbs each is bound by latency: a wave issues one instruction in four
// clocks, and with 16 residues a thread the row pass of 2^14 limbs was 5.2 us in a few waves.  So the
// shapes that win there have many workgroups and short threads (8 residues per thread in the rows, and
// the primes side by side in the column passes, f64_few; 2^14 limbs 14.7 -> 11.0, 2^16 16.5 ->
// 12.9, 2^17 19.1 -> 16.4, 2^18 23.4 -> 21.1, 2^19 36.3 -> 34.0) and short columns (2^14 limbs: 11.4
// with 2^5-point columns, 11.9 with 2^6; 2^16: 13.0 and 13.6; 2^17 16.7 and 15.9).  From 2^20 limbs
// the passes are bound by memory and fp64 issue and longer columns pay, the digits then being read
// once for all primes (2^21 limbs: 81.8 with 2^8-point columns, 89.6 with 2^7).  The integer passes at
// the same sizes: 14.5, 15.6, 15.9, 16.5, 18.8, 20.0, 25.8, 36.9, 41.8, 57.8, 89.3 at n = 12, 13, .., 22
// (the last eight limbs of two digits where those are exact).
F64Shape f64_shape(uint32_t n) {
    F64Shape S;
    const int tn = (int)n - 1;
    S.whole = tn <= F64_WHOLE_MAX;
    S.a = tn <= 16 ? 5 : tn <= 18 ? 6 : tn == 19 ? 7 : 8;
    return S;
}

std::string f64_str(uint32_t n, int K, const F64Shape &S) {
    if (S.quad)
        return "squares in doubles (limbs of four digits, 5 45-bit primes, cols 2^" + std::to_string(S.a) + " x rows 2^" +
               std::to_string((int)n - 2 - S.a) + ")";
    std::string s = "squares in doubles (limbs of two digits, " + (K ? std::to_string(K) : std::string("2 or 3")) + " 49-bit primes, ";
    if (S.whole) return s + "a prime's 2^" + std::to_string(n - 1) + " limbs in one workgroup)";
    return s + "cols 2^" + std::to_string(S.a) + " x rows 2^" + std::to_string((int)n - 1 - S.a) + ")";
}

typedef void (*F64ColFn)(F64Args, int);
typedef void (*F64Fn)(F64Args);

template <int LOGG = F64_COL_MIN>
static F64ColFn fwd_fn(int a) {
    if constexpr (LOGG > F64_COL_MAX) return nullptr;
    else return a == LOGG ? k64_col_fwd<LOGG> : fwd_fn<LOGG + 1>(a);
}
template <int LOGG = F64_COL_MIN>
static F64Fn inv_fn(int a) {
    if constexpr (LOGG > F64_COL_MAX) return nullptr;
    else return a == LOGG ? k64_col_inv<LOGG> : inv_fn<LOGG + 1>(a);
}
template <int K, int LOGG = F64_COL_MIN>
static F64Fn split_k(int a) {
    if constexpr (LOGG > F64_SPLIT_MAX) return nullptr;
    else return a == LOGG ? k64_col_inv_split<K, LOGG> : split_k<K, LOGG + 1>(a);
}
static F64Fn split_fn(int K, int a) { return K == 2 ? split_k<2>(a) : K == 3 ? split_k<3>(a) : split_k<0>(a); }
template <int MODE, int LOGG = F64_ROW_MIN>
static F64Fn row_fn(int logg) {
    if constexpr (LOGG > (MODE == F64_EITHER ? F64_ROW_BATCH : F64_ROW_MAX)) return nullptr;
    else return logg == LOGG ? k64_row<LOGG, MODE> : row_fn<MODE, LOGG + 1>(logg);
}
template <int MODE, int LOGG = F64_WHOLE_MIN>
static F64Fn whole_fn(int logg) {
    if constexpr (LOGG > F64_WHOLE_MAX) return nullptr;
    else return logg == LOGG ? k64_whole<LOGG, MODE> : whole_fn<MODE, LOGG + 1>(logg);
}
static F64Fn all_fn(int logg) { return logg == 11 ? k64_all<11> : k64_all<12>; }
static F64Fn mid_fn(bool whole, int mode, int logg) {
    switch (mode) {
        case F64_SQUARE: return whole ? whole_fn<F64_SQUARE>(logg) : row_fn<F64_SQUARE>(logg);
        case F64_MUL: return whole ? whole_fn<F64_MUL>(logg) : row_fn<F64_MUL>(logg);
        case F64_FWD: return whole ? whole_fn<F64_FWD>(logg) : row_fn<F64_FWD>(logg);
        default: return whole ? whole_fn<F64_EITHER>(logg) : row_fn<F64_EITHER>(logg);
    }
}

// Slots are pinned to XCDs (slot s on XCD s mod 8) where that leaves at most an eighth of the XCDs'
// time idle: what one pass leaves in the XCD's L2 the next one finds there.  us per round of a
// batch, pinned and not: 301 slots of n = 12 18.5 and 26.4, 32 slots 7.8 and 9.2, 64 of n = 13 11.6 and
// 15.9, of n = 14 21.4 and 29.9, of n = 15 32.8 and 36.3, 7 of n = 18 37.1 and 40.3; equal where 4 MiB of L2
// hold little of an XCD's share (512 of n = 15 204 and 206, 24 of n = 18 88); 3 slots of n = 20 would use
// 3 of the 8 XCDs: 112 and 55.6.
static bool f64_pin(uint32_t slots) { return slots >= 7 && 7 * ((slots + 7) / 8) <= slots; }

// Whether the column passes run the primes side by side: where one after the other they would be less than
// a wave of 8 limbs a thread on every SIMD.  The forward pass then takes one prime per workgroup (else all
// from one read of the digits), the inverse one a prime per group of threads.  us per round, one after the
// other and side by side: 16 slots of n = 14 14.6 and 11.8, 16 of n = 15 17.7 and 15.6, 3 of n = 18 32.6 and
// 29.1, 2 of n = 20 (2^20 limbs) 41.7 and 40.5; past it 64 of n = 15 34.3 and 36.3, 7 of n = 18 37.8 and
// 39.0, 24 of n = 18 87.7 and 93.7, 512 of n = 15 205 and 218, 8 of n = 20 120 and 128.
static bool f64_few(const F64Args &A) { return ((uint64_t)A.nslots << A.tn) <= (1u << 19); }

// Workgroups of a launch of `per` a slot (f64_job).
static dim3 f64_grid(F64Args &A, uint32_t per) {
    A.pin = !A.K && f64_pin(A.nslots);
    return dim3(A.pin ? 8 * per * ((A.nslots + 7) / 8) : per * A.nslots);
}

void f64_launch_fwd(F64Args A, const F64Shape &S, hipStream_t stream) {
    if (S.quad) return f64q_launch_fwd(A, S, stream);
    const unsigned nb = 1u << (A.tn - S.a - 4), T = 16u << (S.a - F64_COL_E);
    const int split = f64_few(A);
    const dim3 grid = f64_grid(A, split ? 3 * nb : nb);
    hipLaunchKernelGGL(fwd_fn(S.a), grid, dim3(T), (size_t)128 << S.a, stream, A, split);
}

void f64_launch_mid(F64Args A, const F64Shape &S, int mode, hipStream_t stream) {
    if (S.quad) return f64q_launch_mid(A, S, mode, stream);
    const int L = S.whole ? A.tn : A.tn - S.a;
    if (A.mixed) {
        const F64Fn f = mode == F64_SQUARE ? k64_whole_mixed<F64_SQUARE> : mode == F64_MUL ? k64_whole_mixed<F64_MUL>
                                                                                         : k64_whole_mixed<F64_FWD>;
        const dim3 grid = f64_grid(A, 3);
        hipLaunchKernelGGL(f, grid, dim3(512), (size_t)8 * f64_row_words(12), stream, A);
        return;
    }
    const int loge = f64_row_loge(L);
    if (S.whole) {
        const dim3 grid = f64_grid(A, 3);
        hipLaunchKernelGGL(mid_fn(true, mode, L), grid, dim3(1u << (L - loge)), (size_t)8 * f64_row_words(L), stream, A);
        return;
    }
    A.ng = L - loge >= 6 ? 1 : 64 >> (L - loge);  // rows per workgroup: one wave at least
    const dim3 grid = f64_grid(A, 3 * ((1u << S.a) / A.ng));
    hipLaunchKernelGGL(mid_fn(false, mode, L), grid, dim3((unsigned)A.ng << (L - loge)),
                       (size_t)8 * A.ng * f64_row_words(L), stream, A);
}

void f64_launch_inv(F64Args A, const F64Shape &S, hipStream_t stream) {
    if (S.quad) return f64q_launch_inv(A, S, stream);
    if (S.whole) {
        const dim3 grid = f64_grid(A, (1u << A.tn) / F64_NORM_T);
        hipLaunchKernelGGL(k64_norm, grid, dim3(F64_NORM_T), 0, stream, A);
        return;
    }
    const unsigned T = 16u << (S.a - F64_COL_E), nb = 1u << (A.tn - S.a - 4);
    const dim3 grid = f64_grid(A, nb);
    if (f64_few(A)) {
        const unsigned K = A.K ? A.K : 3;
        hipLaunchKernelGGL(split_fn(A.K, S.a), grid, dim3(K * T), (size_t)K * 128 << S.a, stream, A);
        return;
    }
    hipLaunchKernelGGL(inv_fn(S.a), grid, dim3(T), (size_t)128 << S.a, stream, A);
}

// Whether a round of one-workgroup slots (n = 12, 13) runs each slot's three primes and CRT in one workgroup
// (k64_all): one launch, no residues to memory, but a CU's time for one slot or two or .. for
// all: where the last layer of 256 slots is nearly full.  us per round, k64_whole with k64_norm and k64_all:
// n = 12 128 slots 11.8 and 13.5, 200 15.1 and 13.9, 256 16.4 and 14.3, 301 19.0 and 20.2, 512 26.9 and
// 21.7, 1024 46.1 and 38.6; n = 13 128 slots 18.5 and 20.6, 256 27.5 and 22.2, 301 32.7 and 40.1, 512 46.8 and 41.3.
static bool f64_all(uint32_t slots) { return 8 * slots >= 7 * 256 * ((slots + 255) / 256); }

void f64_launch_square(F64Args A, const F64Shape &S, int mode, hipStream_t stream) {
    if (S.whole && !A.mixed && mode == F64_SQUARE && f64_all(A.nslots)) {
        const dim3 grid = f64_grid(A, 1);
        hipLaunchKernelGGL(all_fn(A.tn), grid, dim3(1u << (A.tn - f64_row_loge(A.tn))), (size_t)8 * f64_row_words(A.tn), stream, A);
        return;
    }
    if (!S.whole) f64_launch_fwd(A, S, stream);
    f64_launch_mid(A, S, mode, stream);
    f64_launch_inv(A, S, stream);
}

void f64_launch_flush(const F64Args &A, hipStream_t stream) {
    const dim3 grid(((1u << (A.tn - 4)) + 255) / 256, A.nslots);
    hipLaunchKernelGGL(k64_flush, grid, dim3(256), 0, stream, A);
    hipLaunchKernelGGL(k64_carry, grid, dim3(256), 0, stream, A);
}

void f64_launch_flush_to(const F64Args &A, const F64Shape &S, uint32_t b, int32_t *dst, hipStream_t stream) {
    if (S.quad) return f64q_launch_flush_to(A, b, dst, stream);
    hipLaunchKernelGGL(k64_flush_to, dim3((1u << (A.tn - 4)) / F64_FLUSH_R), dim3(2 * F64_FLUSH_R), 0, stream, A, b, dst);
}

void f64_set_lds_attributes() {
    static std::once_flag once;
    std::call_once(once, []() {
        auto set = [](const void *f) {
            if (f) (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        };
        for (int a = F64_COL_MIN; a <= F64_COL_MAX; ++a) {
            set((const void *)fwd_fn(a));
            set((const void *)inv_fn(a));
        }
        f64q_set_lds_attributes();
        for (int a = F64_COL_MIN; a <= F64_SPLIT_MAX; ++a) {
            for (int k : {0, 2, 3}) set((const void *)split_fn(k, a));
        }
        for (int l = F64_WHOLE_MIN; l <= F64_WHOLE_MAX; ++l) set((const void *)all_fn(l));
        for (int m = 0; m < 4; ++m) {
            for (int l = F64_ROW_MIN; l <= F64_ROW_MAX; ++l) set((const void *)mid_fn(false, m, l));
            for (int l = F64_WHOLE_MIN; l <= F64_WHOLE_MAX; ++l) set((const void *)mid_fn(true, m, l));
        }
        (void)hipGetLastError();
    });
}

}  // namespace gfe
