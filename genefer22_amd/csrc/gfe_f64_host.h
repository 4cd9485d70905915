// gfe_f64_host.h -- host side of the double-precision limb transform (gfe_f64.h): where it is exact,
// its constants and shapes, and its launches, for one candidate or for a batch's slots.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>

#include "gfe_f64q.h"

namespace gfe {

// Shape of the passes at one n.  whole: a prime's transform in one workgroup and the normalisation
// after it; else three passes over 2^a rows of 2^(n-1-a) limbs, or with quad of 2^(n-2-a) limbs of four
// digits (gfe_f64q.h).
struct F64Shape {
    int whole = 0, a = 0, quad = 0;
};

// Primes the transform needs for (b, n): 2 or 3, or 0 where it is not exact (or out of range).
int f64_primes(uint32_t b, uint32_t n);
// Largest n at which it is exact for every base.
constexpr uint32_t F64_ALL_BASES_N = 20;
F64Shape f64_shape(uint32_t n);
std::string f64_str(uint32_t n, int K, const F64Shape &S);  // K = 0: by the slot
F64Crt make_f64_crt(uint32_t n, uint32_t b, int K);
// Table words of one prime: entries psi^bitrev(j), j < M / 4 (those of a smaller n are its first ones).
inline size_t f64_tw_words(uint32_t n) { return ((size_t)1 << n) / 8; }
int f64_build_twiddles(uint32_t n, double *tw, hipStream_t stream);
uint64_t f64_inv_mod(uint64_t a, uint64_t p);
uint64_t f64_inv_pow2(int k, uint64_t p);     // 2^-k mod p
double f64_balanced(uint64_t a, uint64_t p);  // in (-p/2, p/2]

// Limbs of four digits, for one candidate: where they are exact and pay, constants and tables.
bool f64q_ok(uint32_t b, uint32_t n);
void make_f64q_crt(uint32_t n, uint32_t b, F64QCrt *out);
inline size_t f64q_crt_bytes() { return sizeof(F64QCrt); }
inline size_t f64q_tw_words(uint32_t n) { return ((size_t)1 << n) / 16; }
int f64q_build_twiddles(uint32_t n, double *tw, hipStream_t stream);
F64Shape f64q_shape(uint32_t n);

// Slot s of a launch: registers at regs + s reg_stride (2^n digits each), residues at
// ws / zp + s ws_stride, range carries at slots + s slot_stride, constants crt[s].  One candidate is slot
// 0 with K set: its kernels then wait for no per-slot table before their first loads (0.3-0.5 us a
// launch).
struct F64Args {
    int32_t *regs;
    double *ws;             // what the pass reads and writes: the work space, or the multiplicand
    const double *zp;       // [K][M] multiplicand
    const double *tw;       // [3][tws] twiddles
    int4 *slots;            // M / 16 range carries
    const void *crt;        // F64Crt[nslots], or F64QCrt
    const uint8_t *active, *dupf, *mulf;  // per slot, or null (all, dup, none)
    long long reg_stride, ws_stride, slot_stride;
    uint32_t src_reg, tws, nslots;
    int tn, a, dup, absorb;
    int ng;                 // rows per workgroup (set by the launches)
    int pin;                // slot s on XCD s mod 8 (set by the launches)
    int mixed;              // slots of n = 12 beside those of n = 13 (tn = 12, whole)
    int K;                  // one candidate's primes, or 0: slots, each with its own
};

// Register src_reg -> (fwd and) mid -> ws, and ws -> register 0 with the carry (inv).
void f64_launch_fwd(F64Args A, const F64Shape &S, hipStream_t stream);           // three passes only
void f64_launch_mid(F64Args A, const F64Shape &S, int mode, hipStream_t stream); // row, or whole
void f64_launch_inv(F64Args A, const F64Shape &S, hipStream_t stream);
// A batch's round, mode F64_SQUARE or F64_EITHER: the three in turn of register 0 with its range carries
// (A.absorb), or one launch for all.
void f64_launch_square(F64Args A, const F64Shape &S, int mode, hipStream_t stream);
// Adds the pending range carries of register 0 and balances it.
void f64_launch_flush(const F64Args &A, hipStream_t stream);
// The same to dst (not register 0), which leaves the register and its carries; one candidate of base b.
void f64_launch_flush_to(const F64Args &A, const F64Shape &S, uint32_t b, int32_t *dst, hipStream_t stream);
void f64_set_lds_attributes();
// The same for limbs of four digits (called by the above where S.quad).
void f64q_launch_fwd(const F64Args &A, const F64Shape &S, hipStream_t stream);
void f64q_launch_mid(const F64Args &A, const F64Shape &S, int mode, hipStream_t stream);
void f64q_launch_inv(const F64Args &A, const F64Shape &S, hipStream_t stream);
void f64q_launch_flush(const F64Args &A, uint32_t b, hipStream_t stream);
void f64q_launch_flush_to(const F64Args &A, uint32_t b, int32_t *dst, hipStream_t stream);
void f64q_set_lds_attributes();

}  // namespace gfe
