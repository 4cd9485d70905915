// gfe_f64q.hip -- kernels and host constants of the double-precision transform with limbs of four
// digits (gfe_f64q.h), for one candidate: three launches a squaring, as in gfe_f64.hip.
#include <cstring>

#include "gfe_f64_host.h"

namespace gfe {

// 16 columns for the five primes from one read of the digits, C / 16 workgroups, or (split) for one
// prime each, the five of a group of columns near each other on one XCD.
template <int LOGG>
__global__ void __launch_bounds__(16 << (LOGG - F64_COL_E)) k64q_col_fwd(F64Args A, int split) {
    extern __shared__ double lds64[];
    constexpr int LOGE = F64_COL_E, E = 1 << LOGE;
    const uint32_t M = 1u << A.tn, C = M >> LOGG, t = threadIdx.x;
    const F64QCrtP c = (F64QCrtP)A.crt;
    const uint32_t h = blockIdx.x >> 3;
    const int k0 = split ? h % F64Q_PRIMES : 0, k1 = split ? k0 + 1 : F64Q_PRIMES;
    const unsigned blk = xcd_block(split ? (blockIdx.x & 7u) | (h / F64Q_PRIMES) << 3 : blockIdx.x, C / 16);
    int4 d[E];
    f64q_load_digits<LOGE, LOGG>(d, A.regs + (size_t)A.src_reg * (4u << A.tn), A.absorb ? A.slots : nullptr, C, blk, t);
    const double bd = c->bd;
    double y0[E], y1[E];
#pragma unroll
    for (int rr = 0; rr < E; ++rr) {
        y0[rr] = fma((double)d[rr].y, bd, (double)d[rr].x);
        y1[rr] = fma((double)d[rr].w, bd, (double)d[rr].z);
    }
#pragma unroll 1
    for (int k = k0; k < k1; ++k) {
        const F64Mod md{c->p[k], c->pinv[k]};
        const double sq = c->sq[k];
        const auto limb = [&](int rr) { return f64q_limb(md, y0[rr], y1[rr], sq); };
        f64_col_fwd<LOGE, LOGG>(md, limb, A.ws + (size_t)k * M, A.tw + (size_t)k * A.tws, C, blk, t, lds64);
    }
}

// 5 2^a workgroups, one row each.
template <int LOGG, int MODE>
__global__ void __launch_bounds__(1 << (LOGG - f64_row_loge(LOGG))) k64q_row(F64Args A) {
    extern __shared__ double lds64[];
    constexpr int LOGE = f64_row_loge(LOGG);
    const F64QCrtP c = (F64QCrtP)A.crt;
    const uint32_t k = blockIdx.x >> A.a, row = blockIdx.x & ((1u << A.a) - 1u);
    const size_t at = ((size_t)k << A.tn) + ((size_t)row << LOGG);
    const F64Mod md{c->p[k], c->pinv[k]};
    double *data = A.ws + at;
    const auto load = [&](double (&x)[1 << LOGE], uint32_t base, auto yl) {
#pragma unroll
        for (int rr = 0; rr < 1 << LOGE; ++rr) x[rr] = data[base + ((uint32_t)rr << decltype(yl)::value)];
    };
    f64_row_pass<F64Slim, LOGG, LOGE, MODE>(md, load, F64Store<1 << LOGE>{data}, data, A.zp + at, A.tw + (size_t)k * A.tws, A.a, row, threadIdx.x, lds64, false);
}

// C / 16 workgroups.
template <int LOGG>
__global__ void __launch_bounds__(16 << (LOGG - F64_COL_E)) k64q_col_inv(F64Args A) {
    extern __shared__ double lds64[];
    constexpr int LOGE = F64_COL_E, E = 1 << LOGE, YL = LOGG - LOGE;
    const uint32_t M = 1u << A.tn, C = M >> LOGG, t = threadIdx.x;
    F64QCrtP c = (F64QCrtP)A.crt;
    const unsigned blk = xcd_block(blockIdx.x, C / 16);
    double x[F64Q_PRIMES][E];
    f64_cols_inv<F64Slim, F64Q_PRIMES, LOGE, LOGG>([&](int k) { return F64Mod{c->p[k], c->pinv[k]}; }, x, A.ws, M, A.tw, A.tws,
                                                   C, blk, t, lds64);
    const uint32_t q = t & 15u, s = t >> 4;
#pragma unroll
    for (int rr = 0; rr < E; ++rr) {
        double r[F64Q_PRIMES];
#pragma unroll
        for (int k = 0; k < F64Q_PRIMES; ++k) r[k] = x[k][rr];
        if (rr % 2 == 0) asm volatile("" : "+s"(c));  // constants read again: held through the pass they spill (27.4 us, not 24.4)
        f64q_norm_limb(c, r, A.dup, (s + ((uint32_t)rr << YL)) * C + blk * 16 + q, M, A.regs, A.slots);
    }
}

constexpr int f64q_split_loge(int logg) { return logg <= 6 ? 3 : 4; }  // at most 1024 threads
constexpr uint32_t f64q_split_threads(int logg) { return 16u << (logg - f64q_split_loge(logg)); }

// The five primes side by side: groups of 16 2^(LOGG - LOGE) threads, one prime each, then all threads
// over the limbs.  C / 16 workgroups.
template <int LOGG>
__global__ void __launch_bounds__(F64Q_PRIMES * f64q_split_threads(LOGG)) k64q_col_inv_split(F64Args A) {
    extern __shared__ double lds64[];
    constexpr int LOGE = f64q_split_loge(LOGG), E = 1 << LOGE, K = F64Q_PRIMES;
    constexpr uint32_t T = f64q_split_threads(LOGG), LIMBS = 16u << LOGG;
    const F64QCrtP c = (F64QCrtP)A.crt;
    const uint32_t M = 1u << A.tn, C = M >> LOGG;
    const int k = __builtin_amdgcn_readfirstlane(threadIdx.x / T);
    const uint32_t t = threadIdx.x % T;
    const unsigned blk = xcd_block(blockIdx.x, C / 16);
    double x[E], *L = lds64 + k * LIMBS;
    f64_col_load<LOGE, LOGG>(x, A.ws + (size_t)k * M, C, blk, t);
    f64_col_inv<F64Slim, LOGE, LOGG>(F64Mod{c->p[k], c->pinv[k]}, x, A.tw + (size_t)k * A.tws, t, L);
#pragma unroll
    for (int rr = 0; rr < E; ++rr) L[((t >> 4) + ((uint32_t)rr << (LOGG - LOGE))) * 16 + (t & 15u)] = x[rr];
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < (LIMBS + K * T - 1) / (K * T); ++j) {
        const uint32_t i = threadIdx.x + j * K * T;
        if (i >= LIMBS) break;  // whole waves
        double r[K];
#pragma unroll
        for (int m = 0; m < K; ++m) r[m] = lds64[m * LIMBS + i];
        f64q_norm_limb(c, r, A.dup, (i >> 4) * C + blk * 16 + (i & 15u), M, A.regs, A.slots);
    }
}

__global__ void __launch_bounds__(256) k64q_flush(F64Args A, uint32_t b) {
    const uint32_t w = blockIdx.x * 256u + threadIdx.x;
    if (w < (1u << A.tn) / 16) f64q_flush_body(A.regs, A.slots, b, w);
}

__global__ void __launch_bounds__(256) k64q_carry(F64Args A, uint32_t b) {
    const uint32_t nrange = (1u << A.tn) / 16, w = blockIdx.x * 256u + threadIdx.x;
    if (w < nrange) f64_carry_digits<64>(A.regs + (size_t)w * 64, w == 0 ? -A.slots[2 * nrange - 1].w : A.slots[2 * w - 1].w, b);
}

// As k64_flush_to.
__global__ void __launch_bounds__(2 * F64_FLUSH_R) k64q_flush_to(F64Args A, uint32_t b, int32_t *dst) {
    const auto range = [&](auto st, uint32_t w) { return f64q_flush_range<decltype(st)::value>(A.regs, dst, A.slots, b, w); };
    f64_flush_to_body<64>(range, dst, (1u << A.tn) / 16, b);
}

// ------------------------------------------------------------------------------------------------
// Host

// As f64_bound with limbs L of four digits; a range's first limb takes four pieces of the limbs below
// (digits up to 1.06 b), its second one piece g more.  b >= 2^20 for the products' pieces and g < b / 2 (above 1.5 M),
// b^2 < 1.5 2^52 for the digit pairs (1.07 b^2 with the range carries).
bool f64q_ok(uint32_t b, uint32_t n) {
    if (n < F64Q_MIN_N || n > 23 || b < (1u << 20) || (double)b * b > 0x1p52 * 1.5) return false;
    const long double bb = b, M = (long double)((uint64_t)1 << (n - 2)), b4 = bb * bb * bb * bb;
    long double P = 1;
    for (int k = 0; k < F64Q_PRIMES; ++k) P *= (long double)F64Q_P[k];
    const long double up = (bb + 1) * (bb * bb + 1), L = (bb / 2 + 4) * up, g = (M < bb / 2 ? M : bb / 2) - 4;
    const long double L0 = (1.06L * bb + g + 8) * up, L1 = L + g;
    const long double X = 2 * (M / 16) * (L0 * L0 + L1 * L1 + 14 * L * L);
    return X < 0.3L * P && X / b4 / b4 + 4 < g;
}

void make_f64q_crt(uint32_t n, uint32_t b, F64QCrt *out) {
    F64QCrt &c = *out;
    memset(&c, 0, sizeof(c));
    struct Inverses {
        double i[5][4];
        Inverses() {
            for (int k = 0; k < F64Q_PRIMES; ++k)
                for (int j = 0; j < k; ++j) i[k][j] = f64_balanced(f64_inv_mod(F64Q_P[j], F64Q_P[k]), F64Q_P[k]);
        }
    };
    static const Inverses inv;
    for (int k = 0; k < F64Q_PRIMES; ++k) {
        const uint64_t p = F64Q_P[k];
        c.p[k] = (double)p;
        c.pinv[k] = 1.0 / (double)p;
        // n - 4 of the transform's n - 2 levels are run and undone
        const uint64_t s = f64_inv_pow2((int)n - 4, p);
        c.s[0][k] = f64_balanced(s, p);
        c.s[1][k] = f64_balanced(2 * s % p, p);
        for (int j = 0; j < k; ++j) c.inv[k][j] = inv.i[k][j];
        c.sq[k] = f64_balanced((uint64_t)b * b % p, p);
    }
    // base-b pieces of p1, p1 p2, .. and of 2^23 times each
    auto times = [b](int64_t (&w)[9], uint64_t f) {
        __int128 carry = 0;
        for (int i = 0; i < 9; ++i) {
            const __int128 x = w[i] * (__int128)f + carry;
            __int128 r = x % b;
            if (r > b / 2) r -= b;
            else if (r < -(__int128)(b / 2)) r += b;
            w[i] = (int64_t)r;
            carry = (x - r) / b;
        }
    };
    int64_t w[9] = {1};
    for (int j = 0; j < 4; ++j) {
        times(w, F64Q_P[j]);
        int64_t u[9];
        memcpy(u, w, sizeof(u));
        times(u, (uint64_t)1 << 23);
        for (int i = 0; i < 9; ++i) {
            c.w[j][i] = (double)w[i];
            c.u[j][i] = (double)u[i];
        }
    }
    c.bd = (double)b;
    c.binv = 1.0 / (double)b;
    c.qb = 0.25 * c.binv;
}

// Passes of one squaring, us (forward, rows, inverse; after the bar limbs of two digits on the same machine):
//   n = 19   4.6  6.8  6.3 | 4.6  7.6  4.6 (equal sums: limbs of two digits stay)
//   n = 20   6.2 11.0  6.8, the primes side by side (7.7 11.0 11.0 one after the other); 2^7-point
//            columns 7.3 9.3 11.1 | 6.9 11.9 7.0
//   n = 21  10.1 15.5 12.5, side by side (inverse 13.6 one after the other); 2^6-point columns 9.6 22.1
//            10.7 | 11.5 18.0 13.0
//   n = 22  17.8 27.1 26.4, 2^8-point columns one prime after the other (forward with a workgroup per
//            prime 23.1); 2^7-point columns side by side 16.3 33.8 22.1 | 17.8 38.8 23.4
//   n = 23  34.8 57.3 49.6 | 31.0 79.7 40.4
F64Shape f64q_shape(uint32_t n) {
    F64Shape S;
    S.quad = 1;
    S.a = n >= 22 ? F64Q_COL_MAX : n == 21 ? 7 : 6;
    return S;
}

typedef void (*F64QFn)(F64Args);
static void (*qfwd_fn(int a))(F64Args, int) {
    return a == 6 ? k64q_col_fwd<6> : a == 7 ? k64q_col_fwd<7> : k64q_col_fwd<8>;
}
static F64QFn qsplit_fn(int a) { return a == 6 ? k64q_col_inv_split<6> : k64q_col_inv_split<7>; }
template <int MODE>
static F64QFn qrow_mode(int logg) {
    return logg == F64Q_ROW_MIN ? k64q_row<F64Q_ROW_MIN, MODE> : k64q_row<F64Q_ROW_MAX, MODE>;
}
static F64QFn qrow_fn(int mode, int logg) {
    return mode == F64_SQUARE ? qrow_mode<F64_SQUARE>(logg) : mode == F64_MUL ? qrow_mode<F64_MUL>(logg) : qrow_mode<F64_FWD>(logg);
}

void f64q_launch_fwd(const F64Args &A, const F64Shape &S, hipStream_t stream) {
    const unsigned nb = 1u << (A.tn - S.a - 4);
    const int split = S.a <= F64Q_SPLIT_MAX;  // the primes side by side
    hipLaunchKernelGGL(qfwd_fn(S.a), dim3(split ? F64Q_PRIMES * nb : nb), dim3(16u << (S.a - F64_COL_E)), (size_t)128 << S.a, stream, A, split);
}

void f64q_launch_mid(const F64Args &A, const F64Shape &S, int mode, hipStream_t stream) {
    const int L = A.tn - S.a;
    hipLaunchKernelGGL(qrow_fn(mode, L), dim3(F64Q_PRIMES << S.a), dim3(1u << (L - f64_row_loge(L))), (size_t)8 * f64_row_words(L), stream, A);
}

void f64q_launch_inv(const F64Args &A, const F64Shape &S, hipStream_t stream) {
    const unsigned nb = 1u << (A.tn - S.a - 4);
    const size_t lds = (size_t)128 << S.a;
    if (S.a <= F64Q_SPLIT_MAX) hipLaunchKernelGGL(qsplit_fn(S.a), dim3(nb), dim3(F64Q_PRIMES * f64q_split_threads(S.a)), F64Q_PRIMES * lds, stream, A);
    else hipLaunchKernelGGL((k64q_col_inv<F64Q_COL_MAX>), dim3(nb), dim3(16u << (S.a - F64_COL_E)), (F64Geo<F64Q_COL_MAX, F64_COL_E>::NCH * lds), stream, A);
}

void f64q_launch_flush(const F64Args &A, uint32_t b, hipStream_t stream) {
    const dim3 grid(((1u << (A.tn - 4)) + 255) / 256);
    hipLaunchKernelGGL(k64q_flush, grid, dim3(256), 0, stream, A, b);
    hipLaunchKernelGGL(k64q_carry, grid, dim3(256), 0, stream, A, b);
}

void f64q_launch_flush_to(const F64Args &A, uint32_t b, int32_t *dst, hipStream_t stream) {
    hipLaunchKernelGGL(k64q_flush_to, dim3((1u << (A.tn - 4)) / F64_FLUSH_R), dim3(2 * F64_FLUSH_R), 0, stream, A, b, dst);
}

void f64q_set_lds_attributes() {
    auto set = [](auto f) {
        (void)hipFuncSetAttribute((const void *)f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    };
    for (int a = F64Q_COL_MIN; a <= F64Q_COL_MAX; ++a) set(qfwd_fn(a));
    for (int a = F64Q_COL_MIN; a <= F64Q_SPLIT_MAX; ++a) set(qsplit_fn(a));
    set(k64q_col_inv<F64Q_COL_MAX>);
    for (int m = 0; m < 3; ++m)
        for (int l = F64Q_ROW_MIN; l <= F64Q_ROW_MAX; ++l) set(qrow_fn(m, l));
    (void)hipGetLastError();
}

}  // namespace gfe
