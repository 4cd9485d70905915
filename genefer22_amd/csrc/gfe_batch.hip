// gfe_batch.hip -- batched squaring engine: many candidates of one n per launch (include/gfe_batch.h).
//
// Device state of a batch of `cap` slots (per slot s, strides fixed by n):
//   regs  : cap x R x N int32 digits (r0, r1 = Gerbicz-Li d(t), r2 = scratch; R = 3, or
//           3 + 2^depth in a proof batch: r3.. = the Pietrzak-Li checkpoints)
//   ws,zp : cap x 3 x N uint32 residues (transform work space, multiplicand)
//   carry : cap x N/8 int64 workgroup carries (or segment carries of fused plans)
//   crt   : cap CrtConst, slots: cap SlotInfo (b, prime count, prime width)
//   tw    : 2 x 3 x N uint32 twiddles (31-bit set, 32-bit set), shared by all slots
//   crt64, tw64 : the same for the double-precision limb transform (gfe_f64.h), in which a batch squares
//           unless gfe_batch_set_plan selects the integer passes; ws, zp and carry hold its residues
//           and range carries then
// Every kernel runs over grid.z = slot and exits at once for a slot that is not active in the
// current round (per-round activity and dup flags are uploaded per 64-round block).  Each slot
// runs its own program: squaring runs (the PRP loop, the Gerbicz-Li check's squarings) and
// register operations (copy, set, multiplicand, product, read-back), as src/genefer.h:479-615
// sequences them for one candidate.

#include <gmp.h>

#include "exponent.h"

#include <algorithm>
#include <chrono>
#include <cstring>
#include <deque>
#include <map>
#include <memory>
#include <sstream>
#include <string>
#include <vector>

#include "../../include/gfe.h"
#include "../../include/gfe_batch.h"
#include "gfe_batch_dev.h"
#include "gfe_engine.h"
#include "gfe_spec.h"
#include "gfe_fused.h"
#include "genefer.h"
#include "gint.h"

namespace gfe {

template <int LOGE>
__global__ void __launch_bounds__(LOGE >= 5 ? 512 : 1024) kb_col_fwd(BArgs A, int to_zp) {
    extern __shared__ uint32_t lds[];
    const int s = bslot(A);
    if (s < 0) return;
    const SlotInfo si = A.slots[s];
    const int prime = blockIdx.y;
    if (prime >= si.rns) return;
    const size_t N = (size_t)1 << A.n, NS = (size_t)1 << A.sn;
    const int32_t *src = A.regs + s * A.reg_stride + A.src_reg * N;
    uint32_t *dst = (to_zp ? A.zp : A.ws) + (size_t)s * 3 * NS + prime * N;
    const uint32_t *tw = A.tw + ((size_t)si.is32 * 3 + prime) * NS;
    if (si.is32) col_fwd_body<ModU, LOGE>(ModU{A.prU.p[prime], A.prU.q[prime]}, src, dst, tw, A.n, A.a, A.ng, xcd_block(blockIdx.x, gridDim.x), lds);
    else col_fwd_body<ModS, LOGE>(ModS{A.prS.p[prime], A.prS.q[prime]}, src, dst, tw, A.n, A.a, A.ng, xcd_block(blockIdx.x, gridDim.x), lds);
}

template <int LOGE>
__global__ void __launch_bounds__(LOGE >= 5 ? 512 : 1024) kb_col_inv(BArgs A) {
    extern __shared__ uint32_t lds[];
    const int s = bslot(A);
    if (s < 0) return;
    const SlotInfo si = A.slots[s];
    const int prime = blockIdx.y;
    if (prime >= si.rns) return;
    const size_t N = (size_t)1 << A.n, NS = (size_t)1 << A.sn;
    uint32_t *dst = A.ws + (size_t)s * 3 * NS + prime * N;
    const uint32_t *tw = A.tw + ((size_t)si.is32 * 3 + prime) * NS;
    if (si.is32) col_inv_body<ModU, LOGE>(ModU{A.prU.p[prime], A.prU.q[prime]}, dst, tw, A.n, A.a, A.ng, xcd_block(blockIdx.x, gridDim.x), lds);
    else col_inv_body<ModS, LOGE>(ModS{A.prS.p[prime], A.prS.q[prime]}, dst, tw, A.n, A.a, A.ng, xcd_block(blockIdx.x, gridDim.x), lds);
}

template <int LOGE, int MODE, int TWF>
__global__ void __launch_bounds__(1024) kb_row(BArgs A) {
    extern __shared__ uint32_t lds[];
    const int s = bslot(A);
    if (s < 0) return;
    const SlotInfo si = A.slots[s];
    const int prime = blockIdx.y;
    if (prime >= si.rns) return;
    const size_t N = (size_t)1 << A.n, NS = (size_t)1 << A.sn;
    uint32_t *data = ((MODE == ROW_FWD) ? A.zp : A.ws) + (size_t)s * 3 * NS + prime * N;
    const uint32_t *zp = A.zp + (size_t)s * 3 * NS + prime * N;
    const uint32_t *tw = A.tw + ((size_t)si.is32 * 3 + prime) * NS;
    const bool mul = MODE == ROW_SQUARE && A.mulf && A.mulf[s];
    if (si.is32) row_body<ModU, LOGE, MODE, TWF>(ModU{A.prU.p[prime], A.prU.q[prime]}, data, zp, tw, A.n, A.a, A.ng, blockIdx.x, lds, mul);
    else row_body<ModS, LOGE, MODE, TWF>(ModS{A.prS.p[prime], A.prS.q[prime]}, data, zp, tw, A.n, A.a, A.ng, blockIdx.x, lds, mul);
}

// Pipelined plans: persistent column and normalisation kernels over the blocks of each
// (slot, prime), prefetching the next block (see col_fwd_loop / col_inv_loop / norm_loop).
template <int LOGE>
__global__ void __launch_bounds__(LOGE >= 5 ? 512 : 1024) kb_col_fwd_p(BArgs A, int to_zp) {
    extern __shared__ uint32_t lds[];
    const int s = bslot(A);
    if (s < 0) return;
    const SlotInfo si = A.slots[s];
    const int prime = blockIdx.y;
    if (prime >= si.rns) return;
    const size_t N = (size_t)1 << A.n, NS = (size_t)1 << A.sn;
    const int32_t *src = A.regs + s * A.reg_stride + A.src_reg * N;
    uint32_t *dst = (to_zp ? A.zp : A.ws) + (size_t)s * 3 * NS + prime * N;
    const uint32_t *tw = A.tw + ((size_t)si.is32 * 3 + prime) * NS;
    if (si.is32) col_fwd_loop<ModU, LOGE>(ModU{A.prU.p[prime], A.prU.q[prime]}, src, dst, tw, A.n, A.a, A.ng, blockIdx.x, gridDim.x, lds);
    else col_fwd_loop<ModS, LOGE>(ModS{A.prS.p[prime], A.prS.q[prime]}, src, dst, tw, A.n, A.a, A.ng, blockIdx.x, gridDim.x, lds);
}

template <int LOGE>
__global__ void __launch_bounds__(LOGE >= 5 ? 512 : 1024) kb_col_inv_p(BArgs A) {
    extern __shared__ uint32_t lds[];
    const int s = bslot(A);
    if (s < 0) return;
    const SlotInfo si = A.slots[s];
    const int prime = blockIdx.y;
    if (prime >= si.rns) return;
    const size_t N = (size_t)1 << A.n, NS = (size_t)1 << A.sn;
    uint32_t *data = A.ws + (size_t)s * 3 * NS + prime * N;
    const uint32_t *tw = A.tw + ((size_t)si.is32 * 3 + prime) * NS;
    if (si.is32) col_inv_loop<ModU, LOGE>(ModU{A.prU.p[prime], A.prU.q[prime]}, data, tw, A.n, A.a, A.ng, blockIdx.x, gridDim.x, lds);
    else col_inv_loop<ModS, LOGE>(ModS{A.prS.p[prime], A.prS.q[prime]}, data, tw, A.n, A.a, A.ng, blockIdx.x, gridDim.x, lds);
}

__global__ void __launch_bounds__(256) kb_norm_p(BArgs A) {
    const int s = bslot(A);
    if (s < 0) return;
    const SlotInfo si = A.slots[s];
    const size_t N = (size_t)1 << A.n, NS = (size_t)1 << A.sn;
    const CrtConst &c = A.crt[s];
    const bool dup = A.dup ? (A.dup[s] != 0) : false;
    const uint32_t *ws = A.ws + (size_t)s * 3 * NS;
    int32_t *dst = A.regs + s * A.reg_stride;
    int64_t *wc = A.carry + (size_t)s * (NS >> 3);
    if (si.rns == 3) {
        if (si.is32) norm_loop<3, ModU, 8>(c, ws, dst, wc, si.b, dup, A.n, blockIdx.x, gridDim.x);
        else norm_loop<3, ModS, 8>(c, ws, dst, wc, si.b, dup, A.n, blockIdx.x, gridDim.x);
    } else {
        if (si.is32) norm_loop<2, ModU, 8>(c, ws, dst, wc, si.b, dup, A.n, blockIdx.x, gridDim.x);
        else norm_loop<2, ModS, 8>(c, ws, dst, wc, si.b, dup, A.n, blockIdx.x, gridDim.x);
    }
}

// Fused plans: all primes of a slot per workgroup (see col_fwd_all_body / col_inv_norm_body).
template <int LOGE>
__global__ void __launch_bounds__(512) kb_col_fwd_all(BArgs A, int to_zp) {
    extern __shared__ uint32_t lds[];
    const int s = bslot(A);
    if (s < 0) return;
    const SlotInfo si = A.slots[s];
    const int32_t *src = A.regs + s * A.reg_stride + A.src_reg * ((size_t)1 << A.n);
    uint32_t *dst = (to_zp ? A.zp : A.ws) + (size_t)s * 3 * ((size_t)1 << A.sn);
    const uint32_t *tw = A.tw + (size_t)si.is32 * 3 * ((size_t)1 << A.n);
    if (si.rns == 3) {
        if (si.is32) col_fwd_all_body<3, ModU, LOGE>(A.prU, src, dst, tw, A.n, A.a, A.ng, xcd_block(blockIdx.x, gridDim.x), lds);
        else col_fwd_all_body<3, ModS, LOGE>(A.prS, src, dst, tw, A.n, A.a, A.ng, xcd_block(blockIdx.x, gridDim.x), lds);
    } else {
        if (si.is32) col_fwd_all_body<2, ModU, LOGE>(A.prU, src, dst, tw, A.n, A.a, A.ng, xcd_block(blockIdx.x, gridDim.x), lds);
        else col_fwd_all_body<2, ModS, LOGE>(A.prS, src, dst, tw, A.n, A.a, A.ng, xcd_block(blockIdx.x, gridDim.x), lds);
    }
}

template <int LOGE>
__global__ void __launch_bounds__(512) kb_col_inv_norm(BArgs A) {
    extern __shared__ uint32_t lds[];
    const int s = bslot(A);
    if (s < 0) return;
    const SlotInfo si = A.slots[s];
    const size_t N = (size_t)1 << A.n, NS = (size_t)1 << A.sn;
    const CrtConst &c = A.crt[s];
    const bool dup = A.dup ? (A.dup[s] != 0) : false;
    const uint32_t *ws = A.ws + (size_t)s * 3 * NS;
    const uint32_t *tw = A.tw + (size_t)si.is32 * 3 * N;
    int32_t *dst = A.regs + s * A.reg_stride;
    int64_t *seg = A.carry + (size_t)s * (NS >> 3);
    if (si.rns == 3) {
        if (si.is32) col_inv_norm_body<3, ModU, LOGE>(c, ws, tw, dst, seg, si.b, dup, si.rounds, A.n, A.a, A.ng, xcd_block(blockIdx.x, gridDim.x), lds);
        else col_inv_norm_body<3, ModS, LOGE>(c, ws, tw, dst, seg, si.b, dup, si.rounds, A.n, A.a, A.ng, xcd_block(blockIdx.x, gridDim.x), lds);
    } else {
        if (si.is32) col_inv_norm_body<2, ModU, LOGE>(c, ws, tw, dst, seg, si.b, dup, si.rounds, A.n, A.a, A.ng, xcd_block(blockIdx.x, gridDim.x), lds);
        else col_inv_norm_body<2, ModS, LOGE>(c, ws, tw, dst, seg, si.b, dup, si.rounds, A.n, A.a, A.ng, xcd_block(blockIdx.x, gridDim.x), lds);
    }
}

__global__ void __launch_bounds__(256) kb_fold(BArgs A) {
    const int s = bslot(A);
    if (s < 0) return;
    const size_t N = (size_t)1 << A.n, NS = (size_t)1 << A.sn;
    const size_t nseg = N / (size_t)A.ng;
    const size_t j = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < nseg) fold_body(A.regs + s * A.reg_stride, A.carry + (size_t)s * (NS >> 3), nseg, A.ng, A.slots[s].b, j);
}

__global__ void __launch_bounds__(256) kb_norm(BArgs A) {
    const int s = bslot(A);
    if (s < 0) return;
    const SlotInfo si = A.slots[s];
    const size_t N = (size_t)1 << A.n, NS = (size_t)1 << A.sn;
    const CrtConst &c = A.crt[s];
    const bool dup = A.dup ? (A.dup[s] != 0) : false;
    const uint32_t *ws = A.ws + (size_t)s * 3 * NS;
    int32_t *dst = A.regs + s * A.reg_stride;
    int64_t *wc = A.carry + (size_t)s * (NS >> 3);
    if (si.rns == 3) {
        if (si.is32) norm_body<3, ModU, 8>(c, ws, dst, wc, si.b, dup, A.n, blockIdx.x);
        else norm_body<3, ModS, 8>(c, ws, dst, wc, si.b, dup, A.n, blockIdx.x);
    } else {
        if (si.is32) norm_body<2, ModU, 8>(c, ws, dst, wc, si.b, dup, A.n, blockIdx.x);
        else norm_body<2, ModS, 8>(c, ws, dst, wc, si.b, dup, A.n, blockIdx.x);
    }
}

__global__ void __launch_bounds__(256) kb_carry_wg(BArgs A) {
    const int s = bslot(A);
    if (s < 0) return;
    const size_t N = (size_t)1 << A.n, NS = (size_t)1 << A.sn;
    const unsigned nwg = (unsigned)(N >> 11);
    const unsigned w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w < nwg) carry_wg_body(A.regs + s * A.reg_stride, A.carry + (size_t)s * (NS >> 3), nwg, A.slots[s].b, w);
}

// r_dst = r_src of each active slot.
__global__ void __launch_bounds__(256) kb_copy(BArgs A) {
    const int s = bslot(A);
    if (s < 0) return;
    const size_t N = (size_t)1 << A.n, n4 = N / 4;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n4) return;
    const int4 *src = reinterpret_cast<const int4 *>(A.regs + s * A.reg_stride + A.src_reg * N);
    int4 *dst = reinterpret_cast<int4 *>(A.regs + s * A.reg_stride + A.dst_reg * N);
    dst[i] = src[i];
}

// r_dst = value of each active slot.
__global__ void __launch_bounds__(256) kb_set(BArgs A) {
    const int s = bslot(A);
    if (s < 0) return;
    const size_t N = (size_t)1 << A.n, NS = (size_t)1 << A.sn;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < N) A.regs[s * A.reg_stride + A.dst_reg * N + i] = (i == 0) ? A.value : 0;
}

// A slot taken by a candidate: its constants, r0 = r1 = 1, and no pending carries (the last candidate's
// would be added to r0: timed rounds leave some in a slot that only waits for its read-back).  The
// constants come as arguments of the one launch: four uploads and two kb_set launches over every
// slot's workgroups took 30-37 us a candidate.
struct SlotInit {
    SlotInfo si;
    CrtConst c;
    F64Crt d;
    SlotInfo *slots;
    CrtConst *crt;
    F64Crt *crt64;
    int4 *r0, *r1, *carry;
    uint32_t n4, c4;  // c4 <= n4: carries of the batch's largest n
    int s;
};
__global__ void __launch_bounds__(256) kb_take_slot(SlotInit A) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= A.n4) return;
    A.r0[i] = A.r1[i] = make_int4(i == 0, 0, 0, 0);
    if (i < A.c4) A.carry[i] = make_int4(0, 0, 0, 0);
    if (i == 0) {
        A.slots[A.s] = A.si;
        A.crt[A.s] = A.c;
        A.crt64[A.s] = A.d;
    }
}

// ------------------------------------------------------------------------------------------------
// Host side

static double now_s() {
    return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

enum ItemKind { IT_RUN = 0, IT_COPY, IT_SET, IT_INITMUL, IT_MUL, IT_READ_RES, IT_READ_H1, IT_READ_H2, IT_READ_MU,
                IT_READ_PKEY };
// RUN_POW: rounds of a power r0 = r0^e by square-and-multiply (r0 = 1 and rm = the base before it):
// round kinds from Slot::powseq, 0 = square, 1 = multiply by rm.
enum RunKind { RUN_PRP = 0, RUN_ZERO = 1, RUN_RES = 2, RUN_POW = 3 };

// Non-negative big integers as little-endian 32-bit words (the Pietrzak-Li exponents w_j).
typedef std::vector<uint32_t> Words;
static void words_mul(Words &x, uint32_t q) {
    uint64_t c = 0;
    for (auto &v : x) {
        const uint64_t t = (uint64_t)v * q + c;
        v = (uint32_t)t;
        c = t >> 32;
    }
    if (c) x.push_back((uint32_t)c);
    while (!x.empty() && x.back() == 0) x.pop_back();
}

struct Item {
    int kind;
    uint32_t a = 0, b = 0;            // op arguments (dst, src) / (value)
    int run = RUN_PRP;                // squaring run source
    uint64_t start = 0, len = 0;      // PRP: index (from the top) of the first squaring; length
};

struct Slot {
    bool busy = false, done = false;
    uint32_t b = 0;
    uint32_t n = 0;                   // the candidate's n
    int rns = 0, is32 = 0;
    uint64_t tag = 0, esize = 0, iters = 0;
    double t_submit = 0, t_done = 0;
    std::vector<uint64_t> ebits;      // E = b^(2^n) >> eshift, little-endian 64-bit words
    uint64_t eshift = 0;              // truncated runs keep only E's top bits (exponent_top)
    std::vector<uint8_t> resbits;     // Gerbicz-Li exponent `res`, most significant bit first
    std::vector<uint8_t> powseq;      // round kinds of the queued power runs (RUN_POW)
    // Pietrzak-Li proof (proof batches): its items are queued phase by phase, each phase after the
    // read-back of mu_(k-1) gives the exponent q = hash32(mu_(k-1)) (src/genefer.h:620-734).
    bool pl_pending = false;          // proof phases still to queue
    int pl_k = 0;                     // next mu_k to read
    std::vector<Words> w;             // exponents w_j, j < 2^depth / 2
    std::vector<uint64_t> mu_hash;    // gethash64 of mu_0, mu_1, ...
    uint64_t pkey = 0;                // proof key: gethash64 of v1 (after the last phase)
    bool zp64 = false;                // the multiplicand is the double-precision transform's
    std::deque<Item> q;
    uint64_t pos = 0;                 // progress inside the head run
    uint64_t res64 = 0, old64 = 0, hash64 = 0, h1 = 0;
    int is_prp = 0, gl_ok = -1;
    int reads_pending = 0;            // result read-backs enqueued and not yet processed

    bool bit(uint64_t k) const {  // k-th squaring of the PRP loop (bit esize - 1 - k)
        const uint64_t i = esize - 1 - k - eshift;
        return (ebits[i >> 6] >> (i & 63)) & 1;
    }
};

struct Batch {
    uint32_t n = 0, cap = 0;
    uint32_t nregs = 3;   // registers per slot: 3, or 3 + 2^depth in a proof batch
    int depth = 0;        // Pietrzak-Li depth of every submission (0: quick tests)
    int device = 0;
    size_t N = 0;        // digits of the transform being launched (the slots' n; a mixed batch switches it
                         // per group of register operations, with_n)
    size_t NA = 0;       // digits per register in the allocation: 2^nalloc
    uint32_t nalloc = 0; // the batch's n: per-slot strides
    bool mixed = false;  // slots of n = 12 and 13 share the batch (squaring blocks: kf_square_mixed)
    Plan plan;
    Plan op_plan[2];     // mixed batches: the four-step plans of n = 12 and 13 (register operations)
    hipStream_t stream = nullptr;
    int32_t *regs = nullptr;
    uint32_t *ws = nullptr, *zp = nullptr, *tw = nullptr;
    int64_t *carry = nullptr;
    CrtConst *crt = nullptr;
    SlotInfo *slots_dev = nullptr;
    uint8_t *act_dev = nullptr, *dup_dev = nullptr;   // [64][cap] each
    uint8_t *mul_dev = nullptr;                       // [64][cap]: rounds that multiply by rm
    // Pinned ring of flag uploads: a buffer is rewritten only after its last upload has ended.
    static constexpr int NSTAGE = 8;
    uint8_t *stage[NSTAGE] = {};                      // each 3 x 64 x cap
    hipEvent_t stage_ev[NSTAGE] = {};
    int stage_i = 0;
    int32_t *readback = nullptr;                      // pinned N int32 (synchronous reads)
    // Asynchronous result read-backs: pinned N-digit buffers, each with a completion event,
    // processed in stream order.
    static constexpr int NREAD = 8;
    int32_t *rbuf[NREAD] = {};
    hipEvent_t rev[NREAD] = {};
    struct Read { int slot, kind, buf; };
    std::deque<Read> reads;
    std::vector<int> rfree;
    // One event after each enqueued squaring block: the device backlog of this batch.
    static constexpr int NBLK = 8;
    hipEvent_t blk_ev[NBLK] = {};
    std::deque<int> blk_q;
    int blk_next = 0;
    uint32_t zl = 0;                                  // 1 + highest busy slot: grid.z of launches
    int cus = 0;
    std::map<std::tuple<const void *, int, size_t>, unsigned> resident;
    unsigned resident_blocks(const void *fn, int threads, size_t lds);
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    PrimeArgs prS, prU;
    // Squaring blocks as HIP graphs: the kernels of `rounds` consecutive rounds (per-round flag rows
    // act_dev / dup_dev + r cap, which the block's flag upload fills before the launch) captured
    // once per (rounds, grid depth zl, plan) and replayed.  The cache is dropped when the plan
    // changes and keeps the MAX_GRAPHS most recently launched otherwise.  An executable graph is
    // destroyed only after the stream has drained: a launch of it may still be queued.  Captured
    // kernels record no memset (fill kernels only).
    static constexpr size_t MAX_GRAPHS = 16;
    // (key: the plan, or the double-precision transform with or without multiplying rounds)
    struct BlockGraph { int rounds; uint32_t zl; uint64_t key; hipGraphExec_t exec; uint64_t last_use; };
    std::vector<BlockGraph> graphs;
    uint64_t graph_uses = 0;
    bool use_graphs = true;
    uint64_t plan_key() const;
    hipGraphExec_t block_graph(int rounds, bool has_mul = false);
    void drop_graphs();
    int run_block(int rounds, uint32_t nact, bool has_mul = false, uint32_t nbig = 0);
    // The single-workgroup squaring at n = 13 pays off once 128 or more slots are active: with
    // fewer, one workgroup per candidate leaves most CUs idle and the four-step passes finish a
    // round sooner (one candidate: 76 ms against 166 ms for 4096 squarings on MI355X).  At n = 12
    // it is the faster path at any occupancy.
    // Blocks with multiplying rounds (powers) run the four-step passes.
    bool fused_block(uint32_t nact, bool has_mul = false) const {
        return plan.fuse_sq && !has_mul && (n <= 12 || nact >= 128u);
    }
    // Squaring rounds leave the normalisation's workgroup carries in `carry` and the next round's
    // column forward pass adds them (compile-time plans); carry_wg_body clears what it applies, so
    // `carry` always holds carries not yet in register 0, or zeros, and a squaring round may absorb
    // it unconditionally.  Register operations, the single-workgroup squaring and plan changes
    // apply the pending carries first (flush_carries).  Only for rows of 2^11 or more digits: with
    // shorter rows every (2^11 / row)-th row starts a carry range, an eighth or more of the column
    // workgroups take the extra step and the column pass loses what the carry kernel cost (n = 15,
    // 512 slots, measured on MI355X: 0.367 ms per round either way; n = 20, one slot: 52.9 us against
    // 54.8 us with the carry kernel).
    bool carries_pending = false;
    // The double-precision limb transform: selected until gfe_batch_set_plan, or by the tuner
    // (n <= F64_ALL_BASES_N), but a power run ends in the transform that holds its multiplicand
    // (mode64).  Its range carries stay pending from round to round in every shape.  carry64: the form
    // `carry` holds.  timed64: what the tuner times, 0 or 1, whatever is under way (no products then).
    bool f64 = false, carry64 = false;
    int timed64 = -1;
    F64Shape shape;
    double *tw64 = nullptr;
    F64Crt *crt64 = nullptr;
    int int_tables();
    bool mode64() const;
    int use_mode(bool m);
    F64Args args64(const uint8_t *active, const uint8_t *dup, const uint8_t *mulf) const;
    bool defer_carry() const { return plan.spec && !plan.pipe && !plan.fused && (int)n - plan.a >= 11; }
    void flush_carries();
    int zero_carries();
    std::vector<Slot> slots;
    std::deque<gfe_batch_result> finished;
    double t0 = 0;
    bool ok = false;

    ~Batch();
    int init(uint32_t n, uint32_t cap, int device, int depth = 0, bool mixed = false);
    BArgs args(const uint8_t *active, const uint8_t *dup) const;
    size_t slot_N(int s) const { return (size_t)1 << slots[s].n; }
    int32_t *reg(int s, uint32_t r) const { return regs + (size_t)s * nregs * NA + (size_t)r * slot_N(s); }
    // Runs f with the transform of n = m (a mixed batch's register operations on its slots of n = m).
    template <class F> void with_n(uint32_t m, const F &f) {
        if (!mixed || m == n) { f(); return; }
        const uint32_t n0 = n;
        const size_t N0 = N;
        const Plan p0 = plan;
        n = m; N = (size_t)1 << m; plan = op_plan[m - 12];
        f();
        n = n0; N = N0; plan = p0;
    }
    void queue_power(Slot &S, uint32_t src, const Words &e);
    void queue_pl_phase(Slot &S, int k);
    void pl_read_done(Slot &S, gint &g);
    size_t lds_col() const { return (size_t)plan.col_ng * ((1u << plan.a) + ((1u << plan.a) >> plan.col_loge)) * 4; }
    size_t lds_row() const {
        const uint32_t G = 1u << (n - plan.a);
        return (size_t)plan.row_ng * (G + (G >> plan.row_loge)) * 4;
    }
    void launch_col_fwd(const BArgs &A, int to_zp);
    void launch_row(const BArgs &A, int mode);
    void launch_col_inv(const BArgs &A);
    void launch_norm_carry(const BArgs &A);
    void square(const uint8_t *active, const uint8_t *dup, const uint8_t *mulf, bool has_mul);
    void op_copy(const uint8_t *active, uint32_t dst, uint32_t src);
    void op_set(const uint8_t *active, uint32_t dst, int32_t value);
    void op_initmul(const uint8_t *active, uint32_t src);
    void op_mul(const uint8_t *active);
    uint8_t *stage_acquire();
    void stage_release();
    int submit(uint32_t b, uint64_t iters, uint64_t tag, int32_t *slot, uint32_t n_slot = 0);
    int step(int32_t *active);
    int read_residue(int s, uint32_t reg, gint &g);
    int read_issue(int s, int kind);
    int read_complete(bool wait);
    int harvest();
    int backlog();
    void update_zl();
    unsigned zdim() const { return zl ? zl : 1u; }
    int check(const char *what);
};

int check_hip(hipError_t e, const char *what) {
    if (e != hipSuccess) return set_error(GFE_EHIP, std::string(what) + ": " + hipGetErrorString(e));
    return GFE_OK;
}

int Batch::check(const char *what) { return check_hip(hipGetLastError(), what); }

uint64_t Batch::plan_key() const {
    int32_t a[6];
    plan_to_array(plan, a);
    uint64_t k = 0;
    for (int i = 0; i < 6; ++i) k = k * 1000003u + (uint32_t)a[i];
    return k;
}

void Batch::drop_graphs() {
    if (graphs.empty()) return;
    (void)hipStreamSynchronize(stream);
    for (auto &g : graphs) (void)hipGraphExecDestroy(g.exec);
    graphs.clear();
}

// The instantiated graph of a block of `rounds` squaring rounds at the current grid depth and plan
// (captured on first use; null on failure).
hipGraphExec_t Batch::block_graph(int rounds, bool has_mul) {
    const uint64_t key = mode64() ? 1 + (has_mul ? 1 : 0) : plan_key();
    for (auto &g : graphs)
        if (g.rounds == rounds && g.zl == zdim() && g.key == key) {
            g.last_use = ++graph_uses;
            return g.exec;
        }
    hipGraph_t graph = nullptr;
    if (hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal) != hipSuccess) return nullptr;
    for (int r = 0; r < rounds; ++r)
        square(act_dev + (size_t)r * cap, dup_dev + (size_t)r * cap, mul_dev + (size_t)r * cap, has_mul);
    if (hipStreamEndCapture(stream, &graph) != hipSuccess || !graph) {
        (void)hipGetLastError();
        return nullptr;
    }
    hipGraphExec_t exec = nullptr;
    const hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    if (graphs.size() >= MAX_GRAPHS) {
        auto lru = std::min_element(graphs.begin(), graphs.end(),
                                    [](const BlockGraph &x, const BlockGraph &y) { return x.last_use < y.last_use; });
        (void)hipStreamSynchronize(stream);
        (void)hipGraphExecDestroy(lru->exec);
        graphs.erase(lru);
    }
    graphs.push_back({rounds, zdim(), key, exec, ++graph_uses});
    return exec;
}

// Enqueues `rounds` squaring rounds (flag rows already uploaded): one graph launch, or the
// kernels one by one when graphs are off or the plan uses persistent grids (their sizes come from
// occupancy queries, which stay out of captures).
// A mixed batch runs its slots of n = 12 in the single-workgroup kernel and its slots of n = 13 in
// the same launch when 128 or more of them are active (nbig), otherwise on the four-step passes of
// n = 13 after it (fused_block's rule for one n).
int Batch::run_block(int rounds, uint32_t nact, bool has_mul, uint32_t nbig) {
    const int rc = use_mode(mode64());
    if (rc != GFE_OK) return rc;
    if (mode64()) {
        if (use_graphs) {
            if (hipGraphExec_t g = block_graph(rounds, has_mul)) {
                carries_pending = true;
                return check_hip(hipGraphLaunch(g, stream), "graph launch");
            }
            return set_error(GFE_EHIP, "squaring block graph capture failed");
        }
        for (int r = 0; r < rounds; ++r)
            square(act_dev + (size_t)r * cap, dup_dev + (size_t)r * cap, mul_dev + (size_t)r * cap, has_mul);
        carries_pending = true;
        return check("square block");
    }
    const bool mixed_fused = mixed && (nbig == 0 || nbig >= 128u);
    if (mixed || fused_block(nact, has_mul)) {  // one launch runs the whole block, one workgroup per slot
        flush_carries();
        FusedArgs A;
        memset(&A, 0, sizeof(A));
        A.regs = regs; A.tw = tw; A.crt = crt; A.slots = slots_dev; A.act = act_dev; A.dupf = dup_dev;
        A.reg_stride = (long long)(nregs * NA); A.stride = cap; A.rounds = rounds; A.prS = prS; A.prU = prU;
        A.tws = (uint32_t)NA;
        if (mixed) {
            A.only_n = mixed_fused ? 0 : 12;
            hipLaunchKernelGGL(fused_square_mixed_fn(), dim3(zdim()), dim3(512), fused_lds_bytes(13), stream, A);
        } else {
            hipLaunchKernelGGL(fused_square_fn((int)n), dim3(zdim()), dim3(fused_threads((int)n)), fused_lds_bytes((int)n),
                               stream, A);
        }
        if (!mixed || mixed_fused) return check("fused square block");
        // the slots of n = 13 on the four-step passes (the four-step kernels skip the other slots)
    }
    if (defer_carry()) carries_pending = true;
    if (use_graphs && !plan.pipe) {
        if (hipGraphExec_t g = block_graph(rounds)) return check_hip(hipGraphLaunch(g, stream), "graph launch");
        return set_error(GFE_EHIP, "squaring block graph capture failed");
    }
    for (int r = 0; r < rounds; ++r)
        square(act_dev + (size_t)r * cap, dup_dev + (size_t)r * cap, mul_dev + (size_t)r * cap, has_mul);
    return check("square block");
}

Batch::~Batch() {
    if (!ok) return;
    (void)hipSetDevice(device);
    if (stream) (void)hipStreamSynchronize(stream);
    drop_graphs();
    (void)hipFree(regs); (void)hipFree(ws); (void)hipFree(zp); (void)hipFree(tw); (void)hipFree(carry);
    (void)hipFree(crt); (void)hipFree(slots_dev); (void)hipFree(act_dev); (void)hipFree(dup_dev);
    (void)hipFree(mul_dev);
    (void)hipFree(tw64); (void)hipFree(crt64);
    for (int i = 0; i < NSTAGE; ++i) {
        if (stage[i]) (void)hipHostFree(stage[i]);
        if (stage_ev[i]) (void)hipEventDestroy(stage_ev[i]);
    }
    for (int i = 0; i < NREAD; ++i) {
        if (rbuf[i]) (void)hipHostFree(rbuf[i]);
        if (rev[i]) (void)hipEventDestroy(rev[i]);
    }
    for (int i = 0; i < NBLK; ++i)
        if (blk_ev[i]) (void)hipEventDestroy(blk_ev[i]);
    if (readback) (void)hipHostFree(readback);
    if (ev0) (void)hipEventDestroy(ev0);
    if (ev1) (void)hipEventDestroy(ev1);
    if (stream) (void)hipStreamDestroy(stream);
}

void set_lds_attr(const void *fn);

template <int TWF> void set_row_attrs() {
    set_lds_attr((const void *)kb_row<3, ROW_SQUARE, TWF>); set_lds_attr((const void *)kb_row<4, ROW_SQUARE, TWF>);
    set_lds_attr((const void *)kb_row<5, ROW_SQUARE, TWF>);
    set_lds_attr((const void *)kb_row<3, ROW_MUL, TWF>); set_lds_attr((const void *)kb_row<4, ROW_MUL, TWF>);
    set_lds_attr((const void *)kb_row<5, ROW_MUL, TWF>);
    set_lds_attr((const void *)kb_row<3, ROW_FWD, TWF>); set_lds_attr((const void *)kb_row<4, ROW_FWD, TWF>);
    set_lds_attr((const void *)kb_row<5, ROW_FWD, TWF>);
}

int Batch::init(uint32_t n_, uint32_t cap_, int device_, int depth_, bool mixed_) {
    n = n_; cap = cap_; device = device_;
    depth = depth_;
    mixed = mixed_;
    nregs = depth > 0 ? 3u + (1u << depth) : 3u;
    N = (size_t)1 << n;
    NA = N;
    nalloc = n;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return set_error(GFE_ENODEV, "no HIP device");
    if (device < 0 || device >= ndev) return set_error(GFE_ENODEV, "device index out of range");
    if (hipSetDevice(device) != hipSuccess) return set_error(GFE_EHIP, "hipSetDevice");
    ok = true;
    if (hipStreamCreateWithFlags(&stream, hipStreamNonBlocking) != hipSuccess) return set_error(GFE_EHIP, "stream");
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) cus = 256;
    plan = default_batch_plan(n, cap);
    if (hipMalloc(&regs, (size_t)cap * nregs * NA * 4) != hipSuccess || hipMalloc(&ws, (size_t)cap * 3 * NA * 4) != hipSuccess ||
        hipMalloc(&zp, (size_t)cap * 3 * NA * 4) != hipSuccess ||
        hipMalloc(&carry, (size_t)cap * (NA >> 3) * 8) != hipSuccess || hipMalloc(&crt, (size_t)cap * sizeof(CrtConst)) != hipSuccess ||
        hipMalloc(&slots_dev, (size_t)cap * sizeof(SlotInfo)) != hipSuccess ||
        hipMalloc(&act_dev, (size_t)64 * cap) != hipSuccess || hipMalloc(&dup_dev, (size_t)64 * cap) != hipSuccess ||
        hipMalloc(&mul_dev, (size_t)64 * cap) != hipSuccess ||
        (n <= F64_ALL_BASES_N && hipMalloc(&tw64, F64_PRIMES * f64_tw_words(n) * 8) != hipSuccess) ||
        hipMalloc(&crt64, (size_t)cap * sizeof(F64Crt)) != hipSuccess)
        return set_error(GFE_ENOMEM, "device allocation failed");
    for (int i = 0; i < NSTAGE; ++i) {
        if (hipHostMalloc((void **)&stage[i], (size_t)3 * 64 * cap) != hipSuccess) return set_error(GFE_ENOMEM, "pinned");
        if (hipEventCreateWithFlags(&stage_ev[i], hipEventDisableTiming) != hipSuccess) return set_error(GFE_EHIP, "event");
    }
    for (int i = 0; i < NREAD; ++i) {
        if (hipHostMalloc((void **)&rbuf[i], NA * 4) != hipSuccess) return set_error(GFE_ENOMEM, "pinned");
        if (hipEventCreateWithFlags(&rev[i], hipEventDisableTiming) != hipSuccess) return set_error(GFE_EHIP, "event");
        rfree.push_back(i);
    }
    for (int i = 0; i < NBLK; ++i)
        if (hipEventCreateWithFlags(&blk_ev[i], hipEventDisableTiming) != hipSuccess) return set_error(GFE_EHIP, "event");
    if (hipHostMalloc((void **)&readback, NA * 4) != hipSuccess) return set_error(GFE_ENOMEM, "pinned");
    if (hipEventCreate(&ev0) != hipSuccess || hipEventCreate(&ev1) != hipSuccess) return set_error(GFE_EHIP, "event");
    for (int k = 0; k < 3; ++k) {
        prS.p[k] = prime_of(0, k); prU.p[k] = prime_of(1, k);
        CrtConst c0 = make_crt(3, 0, n), c1 = make_crt(3, 1, n);
        prS.q[k] = c0.q[k]; prU.q[k] = c1.q[k];
    }
    std::vector<SlotInfo> si(cap);
    for (auto &x : si) { x.b = 1024; x.rns = 0; x.is32 = 0; x.rounds = 1; x.n = (int32_t)n; }
    if (hipMemcpy(slots_dev, si.data(), cap * sizeof(SlotInfo), hipMemcpyHostToDevice) != hipSuccess)
        return set_error(GFE_EHIP, "slot upload");
    if (hipMemsetAsync(regs, 0, (size_t)cap * nregs * NA * 4, stream) != hipSuccess ||
        hipMemsetAsync(mul_dev, 0, (size_t)64 * cap, stream) != hipSuccess ||
        hipMemsetAsync(crt64, 0, (size_t)cap * sizeof(F64Crt), stream) != hipSuccess ||
        hipMemsetAsync(carry, 0, (size_t)cap * (NA >> 3) * 8, stream) != hipSuccess ||
        hipMemsetAsync(act_dev, 0, (size_t)64 * cap, stream) != hipSuccess ||
        hipMemsetAsync(dup_dev, 0, (size_t)64 * cap, stream) != hipSuccess)
        return set_error(GFE_EHIP, "memset");
    set_lds_attr((const void *)kb_col_fwd<3>); set_lds_attr((const void *)kb_col_fwd<4>); set_lds_attr((const void *)kb_col_fwd<5>);
    set_lds_attr((const void *)kb_col_inv<3>); set_lds_attr((const void *)kb_col_inv<4>); set_lds_attr((const void *)kb_col_inv<5>);
    set_row_attrs<0>();
    set_row_attrs<1>();
    f64_set_lds_attributes();
    f64 = carry64 = n <= F64_ALL_BASES_N;
    shape = f64_shape(n);
    if (f64 && f64_build_twiddles(n, tw64, stream) != 0) return set_error(GFE_EHIP, "twiddles");
    if (!f64) {
        const int rc = int_tables();
        if (rc != GFE_OK) return rc;
    }
    spec_batch_set_lds_attributes();
    fused_set_lds_attributes();
    set_lds_attr((const void *)kb_col_fwd_p<3>); set_lds_attr((const void *)kb_col_fwd_p<4>); set_lds_attr((const void *)kb_col_fwd_p<5>);
    set_lds_attr((const void *)kb_col_inv_p<3>); set_lds_attr((const void *)kb_col_inv_p<4>); set_lds_attr((const void *)kb_col_inv_p<5>);
    set_lds_attr((const void *)kb_col_fwd_all<3>); set_lds_attr((const void *)kb_col_fwd_all<4>);
    set_lds_attr((const void *)kb_col_inv_norm<3>); set_lds_attr((const void *)kb_col_inv_norm<4>);
    slots.resize(cap);
    for (auto &S : slots) S.n = n;
    if (mixed) {  // register operations of each n on the four-step passes
        op_plan[0] = default_plan(12);
        op_plan[1] = default_plan(13);
    }
    t0 = now_s();
    return check_hip(hipStreamSynchronize(stream), "init");
}


// The integer passes' twiddle tables, made when those passes are first selected.
int Batch::int_tables() {
    if (tw) return GFE_OK;
    std::vector<uint32_t> h(6 * NA);
    const int sets[6] = {0, 0, 0, 1, 1, 1}, primes[6] = {0, 1, 2, 0, 1, 2};
    make_twiddle_tables(sets, primes, 6, nalloc, h.data());
    uint32_t *t = nullptr;
    if (hipMalloc(&t, (size_t)6 * NA * 4) != hipSuccess) return set_error(GFE_ENOMEM, "device allocation failed");
    if (hipMemcpy(t, h.data(), 6 * NA * 4, hipMemcpyHostToDevice) != hipSuccess) {
        (void)hipFree(t);
        return set_error(GFE_EHIP, "twiddle upload");
    }
    tw = t;
    return GFE_OK;
}

F64Args Batch::args64(const uint8_t *active, const uint8_t *dup, const uint8_t *mulf) const {
    F64Args A;
    memset(&A, 0, sizeof(A));
    A.regs = regs; A.ws = reinterpret_cast<double *>(ws); A.zp = reinterpret_cast<const double *>(zp);
    A.tw = tw64; A.tws = (uint32_t)f64_tw_words(nalloc); A.slots = reinterpret_cast<int4 *>(carry); A.crt = crt64;
    A.active = active; A.dupf = dup; A.mulf = mulf;
    A.reg_stride = (long long)(nregs * NA); A.ws_stride = (long long)(3 * NA / 2); A.slot_stride = (long long)(NA / 16);
    A.nslots = zdim(); A.tn = (int)nalloc - 1; A.a = shape.a; A.mixed = mixed;
    return A;
}

// Whether squarings and products run in doubles: as the multiplicands of the power runs under way (which
// are all in one transform, since a multiplicand made beside them goes into theirs), else as selected.
bool Batch::mode64() const {
    if (timed64 >= 0) return timed64 != 0;
    for (uint32_t s = 0; depth > 0 && s < cap; ++s)  // powers are a proof's
        if (slots[s].busy && !slots[s].q.empty() && slots[s].q.front().kind == IT_RUN && slots[s].q.front().run == RUN_POW)
            return slots[s].zp64;
    return f64;
}

// `carry` in the form of the transform about to run: pending carries of the other are applied first.
int Batch::use_mode(bool m) {
    if (m == carry64) return GFE_OK;
    flush_carries();
    carry64 = m;
    return zero_carries();
}

BArgs Batch::args(const uint8_t *active, const uint8_t *dup) const {
    BArgs A;
    memset(&A, 0, sizeof(A));
    A.regs = regs; A.ws = ws; A.zp = zp; A.carry = carry; A.crt = crt; A.slots = slots_dev; A.tw = tw;
    A.active = active; A.dup = dup; A.prS = prS; A.prU = prU; A.reg_stride = (long long)(nregs * NA); A.n = (int)n;
    A.sn = (int)nalloc;
    return A;
}

void Batch::launch_col_fwd(const BArgs &A0, int to_zp) {
    BArgs A = A0;
    A.a = plan.a; A.ng = plan.col_ng;
    if (plan.spec) {
        const uint32_t C = 1u << (n - plan.a);
        const int T = plan.col_ng * (1 << plan.a) / (1 << plan.col_loge);
        hipLaunchKernelGGL(spec_batch_col_fwd(plan.col_loge, plan.a), dim3(C / plan.col_ng, 3, zdim()), dim3(T),
                           col_pass_lds_words(plan.a, plan.col_loge, plan.col_ng) * 4, stream, A, to_zp);
        return;
    }
    const uint32_t C = 1u << (n - plan.a);
    const int T = plan.col_ng * (1 << plan.a) / (1 << plan.col_loge);
    if (plan.fused) {
        const dim3 g1(C / plan.col_ng, 1, zdim());
        if (plan.col_loge == 3) hipLaunchKernelGGL(kb_col_fwd_all<3>, g1, dim3(T), lds_col(), stream, A, to_zp);
        else hipLaunchKernelGGL(kb_col_fwd_all<4>, g1, dim3(T), lds_col(), stream, A, to_zp);
        return;
    }
    if (plan.pipe) {
        const size_t lds = lds_col() + ((size_t)4 << plan.a);
        const void *fn = plan.col_loge == 3 ? (const void *)kb_col_fwd_p<3> : plan.col_loge == 4 ? (const void *)kb_col_fwd_p<4>
                                                                                                  : (const void *)kb_col_fwd_p<5>;
        const dim3 g1(persistent_grid(C / plan.col_ng, 3 * zdim(), resident_blocks(fn, T, lds)), 3, zdim());
        switch (plan.col_loge) {
            case 3: hipLaunchKernelGGL(kb_col_fwd_p<3>, g1, dim3(T), lds, stream, A, to_zp); break;
            case 4: hipLaunchKernelGGL(kb_col_fwd_p<4>, g1, dim3(T), lds, stream, A, to_zp); break;
            default: hipLaunchKernelGGL(kb_col_fwd_p<5>, g1, dim3(T), lds, stream, A, to_zp); break;
        }
        return;
    }
    const dim3 grid(C / plan.col_ng, 3, zdim());
    switch (plan.col_loge) {
        case 3: hipLaunchKernelGGL(kb_col_fwd<3>, grid, dim3(T), lds_col(), stream, A, to_zp); break;
        case 4: hipLaunchKernelGGL(kb_col_fwd<4>, grid, dim3(T), lds_col(), stream, A, to_zp); break;
        default: hipLaunchKernelGGL(kb_col_fwd<5>, grid, dim3(T), lds_col(), stream, A, to_zp); break;
    }
}

void Batch::launch_col_inv(const BArgs &A0) {
    BArgs A = A0;
    A.a = plan.a; A.ng = plan.col_ng;
    if (plan.spec) {
        const uint32_t C = 1u << (n - plan.a);
        const int T = plan.col_ng * (1 << plan.a) / (1 << plan.col_loge);
        hipLaunchKernelGGL(spec_batch_col_inv(plan.col_loge, plan.a), dim3(C / plan.col_ng, 3, zdim()), dim3(T),
                           col_pass_lds_words(plan.a, plan.col_loge, plan.col_ng) * 4, stream, A, 0);
        return;
    }
    const uint32_t C = 1u << (n - plan.a);
    const int T = plan.col_ng * (1 << plan.a) / (1 << plan.col_loge);
    if (plan.fused) {
        const dim3 g1(C / plan.col_ng, 1, zdim());
        if (plan.col_loge == 3) hipLaunchKernelGGL(kb_col_inv_norm<3>, g1, dim3(T), lds_col(), stream, A);
        else hipLaunchKernelGGL(kb_col_inv_norm<4>, g1, dim3(T), lds_col(), stream, A);
        return;
    }
    if (plan.pipe) {
        const size_t lds = lds_col() + ((size_t)4 << plan.a);
        const void *fn = plan.col_loge == 3 ? (const void *)kb_col_inv_p<3> : plan.col_loge == 4 ? (const void *)kb_col_inv_p<4>
                                                                                                  : (const void *)kb_col_inv_p<5>;
        const dim3 g1(persistent_grid(C / plan.col_ng, 3 * zdim(), resident_blocks(fn, T, lds)), 3, zdim());
        switch (plan.col_loge) {
            case 3: hipLaunchKernelGGL(kb_col_inv_p<3>, g1, dim3(T), lds, stream, A); break;
            case 4: hipLaunchKernelGGL(kb_col_inv_p<4>, g1, dim3(T), lds, stream, A); break;
            default: hipLaunchKernelGGL(kb_col_inv_p<5>, g1, dim3(T), lds, stream, A); break;
        }
        return;
    }
    const dim3 grid(C / plan.col_ng, 3, zdim());
    switch (plan.col_loge) {
        case 3: hipLaunchKernelGGL(kb_col_inv<3>, grid, dim3(T), lds_col(), stream, A); break;
        case 4: hipLaunchKernelGGL(kb_col_inv<4>, grid, dim3(T), lds_col(), stream, A); break;
        default: hipLaunchKernelGGL(kb_col_inv<5>, grid, dim3(T), lds_col(), stream, A); break;
    }
}

template <int MODE, int TWF>
static void launch_row_mode_t(const Batch &B, const BArgs &A, dim3 grid, int T) {
    switch (B.plan.row_loge) {
        case 3: hipLaunchKernelGGL((kb_row<3, MODE, TWF>), grid, dim3(T), B.lds_row(), B.stream, A); break;
        case 4: hipLaunchKernelGGL((kb_row<4, MODE, TWF>), grid, dim3(T), B.lds_row(), B.stream, A); break;
        default: hipLaunchKernelGGL((kb_row<5, MODE, TWF>), grid, dim3(T), B.lds_row(), B.stream, A); break;
    }
}
template <int MODE>
static void launch_row_mode(const Batch &B, const BArgs &A, dim3 grid, int T) {
    if (B.plan.row_tw) launch_row_mode_t<MODE, 1>(B, A, grid, T);
    else launch_row_mode_t<MODE, 0>(B, A, grid, T);
}

void Batch::launch_row(const BArgs &A0, int mode) {
    BArgs A = A0;
    A.a = plan.a; A.ng = plan.row_ng;
    const uint32_t R = 1u << plan.a, G = 1u << (n - plan.a);
    const int T = plan.row_ng * G / (1 << plan.row_loge);
    const dim3 grid(R / plan.row_ng, 3, zdim());
    if (plan.spec && mode == ROW_SQUARE) {
        hipLaunchKernelGGL(spec_batch_row_square(plan.row_loge, (int)n - plan.a), grid, dim3(T),
                           row_pass_lds_words((int)n - plan.a, plan.row_loge, plan.row_ng) * 4, stream, A);
        return;
    }
    if (mode == ROW_SQUARE) launch_row_mode<ROW_SQUARE>(*this, A, grid, T);
    else if (mode == ROW_MUL) launch_row_mode<ROW_MUL>(*this, A, grid, T);
    else launch_row_mode<ROW_FWD>(*this, A, grid, T);
}

void Batch::launch_norm_carry(const BArgs &A0) {
    if (plan.fused) {
        BArgs A = A0;
        A.ng = plan.col_ng;
        const size_t nseg = N / (size_t)plan.col_ng;
        hipLaunchKernelGGL(kb_fold, dim3((unsigned)((nseg + 255) / 256), 1, zdim()), dim3(256), 0, stream, A);
        return;
    }
    const BArgs &A = A0;
    const unsigned nwg = (unsigned)(N >> 11);
    if (plan.pipe) {
        const unsigned g = persistent_grid(nwg, zdim(), resident_blocks((const void *)kb_norm_p, 256, 0));
        hipLaunchKernelGGL(kb_norm_p, dim3(g, 1, zdim()), dim3(256), 0, stream, A);
    } else {
        hipLaunchKernelGGL(kb_norm, dim3(nwg, 1, zdim()), dim3(256), 0, stream, A);
    }
    if (!A.absorb) hipLaunchKernelGGL(kb_carry_wg, dim3((nwg + 255) / 256, 1, zdim()), dim3(256), 0, stream, A);
}

void Batch::flush_carries() {
    if (!carries_pending) return;
    carries_pending = false;
    if (carry64) {
        f64_launch_flush(args64(nullptr, nullptr, nullptr), stream);
        return;
    }
    const BArgs A = args(nullptr, nullptr);
    const unsigned nwg = (unsigned)(N >> 11);
    hipLaunchKernelGGL(kb_carry_wg, dim3((nwg + 255) / 256, 1, zdim()), dim3(256), 0, stream, A);
}

// Clears every slot's carries (after a plan whose passes leave other values in `carry`).
int Batch::zero_carries() {
    carries_pending = false;
    return check_hip(hipMemsetAsync(carry, 0, (size_t)cap * (NA >> 3) * 8, stream), "carry clear");
}

void Batch::square(const uint8_t *active, const uint8_t *dup, const uint8_t *mulf, bool has_mul) {
    if (mode64()) {
        F64Args A = args64(active, dup, mulf);
        A.absorb = 1;
        f64_launch_square(A, shape, has_mul ? F64_EITHER : F64_SQUARE, stream);
        return;
    }
    BArgs A = args(active, dup);
    A.mulf = mulf;
    A.src_reg = 0;
    A.absorb = defer_carry() ? 1 : 0;
    launch_col_fwd(A, 0);
    launch_row(A, ROW_SQUARE);
    launch_col_inv(A);
    launch_norm_carry(A);
}

void Batch::op_copy(const uint8_t *active, uint32_t dst, uint32_t src) {
    BArgs A = args(active, nullptr);
    A.src_reg = src; A.dst_reg = dst;
    hipLaunchKernelGGL(kb_copy, dim3((unsigned)((N / 4 + 255) / 256), 1, zdim()), dim3(256), 0, stream, A);
}

void Batch::op_set(const uint8_t *active, uint32_t dst, int32_t value) {
    BArgs A = args(active, nullptr);
    A.dst_reg = dst; A.value = value;
    hipLaunchKernelGGL(kb_set, dim3((unsigned)((N + 255) / 256), 1, zdim()), dim3(256), 0, stream, A);
}

void Batch::op_initmul(const uint8_t *active, uint32_t src) {
    if (mode64()) {
        F64Args A = args64(active, nullptr, nullptr);
        A.src_reg = src;
        A.ws = reinterpret_cast<double *>(zp);
        if (!shape.whole) f64_launch_fwd(A, shape, stream);
        f64_launch_mid(A, shape, F64_FWD, stream);
        return;
    }
    BArgs A = args(active, nullptr);
    A.src_reg = src;
    launch_col_fwd(A, 1);
    launch_row(A, ROW_FWD);
}

void Batch::op_mul(const uint8_t *active) {
    if (mode64()) {
        const F64Args A = args64(active, nullptr, nullptr);
        if (!shape.whole) f64_launch_fwd(A, shape, stream);
        f64_launch_mid(A, shape, F64_MUL, stream);
        f64_launch_inv(A, shape, stream);
        f64_launch_flush(A, stream);
        return;
    }
    BArgs A = args(active, nullptr);
    A.src_reg = 0;
    launch_col_fwd(A, 0);
    launch_row(A, ROW_MUL);
    launch_col_inv(A);
    launch_norm_carry(A);
}

// Pinned staging for per-block flags: two buffers, each reused only after its last upload ended.
uint8_t *Batch::stage_acquire() {
    (void)hipEventSynchronize(stage_ev[stage_i]);
    return stage[stage_i];
}
void Batch::stage_release() {
    (void)hipEventRecord(stage_ev[stage_i], stream);
    stage_i = (stage_i + 1) % NSTAGE;
}

unsigned Batch::resident_blocks(const void *fn, int threads, size_t lds) {
    const auto key = std::make_tuple(fn, threads, lds);
    const auto it = resident.find(key);
    if (it != resident.end()) return it->second;
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, threads, lds) != hipSuccess || nb < 1) nb = 1;
    (void)hipGetLastError();
    const unsigned r = (unsigned)nb * (unsigned)std::max(cus, 1);
    resident[key] = r;
    return r;
}

void Batch::update_zl() {
    zl = 0;
    for (uint32_t s = 0; s < cap; ++s)
        if (slots[s].busy) zl = s + 1;
}

// Squaring blocks enqueued and not yet finished on the device.
int Batch::backlog() {
    while (!blk_q.empty()) {
        const hipError_t e = hipEventQuery(blk_ev[blk_q.front()]);
        if (e == hipErrorNotReady) { (void)hipGetLastError(); break; }
        if (e != hipSuccess) return check_hip(e, "block event");
        blk_q.pop_front();
    }
    return (int)blk_q.size();
}


int Batch::submit(uint32_t b, uint64_t iters, uint64_t tag, int32_t *slot_out, uint32_t n_slot) {
    if (n_slot == 0) n_slot = nalloc;
    if (mixed ? (n_slot < 12 || n_slot > nalloc) : n_slot != nalloc)
        return set_error(GFE_EINVAL, "submit: n does not belong to this batch");
    int s = -1;
    for (uint32_t i = 0; i < cap; ++i)
        if (!slots[i].busy) { s = (int)i; break; }
    if (s < 0) return set_error(GFE_EFULL, "batch full");
    Slot &S = slots[s];
    S = Slot();
    S.busy = true;
    S.b = b;
    S.n = n_slot;
    S.tag = tag;
    S.t_submit = now_s() - t0;
    select_primes(b, S.n, &S.rns, &S.is32);
    S.is32 = transform_is32(S.rns, S.is32);
    // E = b^(2^n) and its bits (src/genefer.h:1476); the first `iters` squarings of a truncated run
    // read only E's top bits, which exponent_top gives without computing E
    mpz_t E;
    mpz_init(E);
    const bool want_all = iters == 0 || depth > 0;
    exponent_top(b, S.n, want_all ? ~uint64_t(0) >> 8 : iters, E, &S.eshift, &S.esize);
    if (!want_all && iters >= S.esize && S.eshift != 0) {  // the whole loop after all
        mpz_ui_pow_ui(E, b, 1ul << S.n);
        S.eshift = 0;
    }
    S.ebits.assign((mpz_sizeinbase(E, 2) + 63) / 64 + 1, 0);
    size_t cnt = 0;
    mpz_export(S.ebits.data(), &cnt, -1, 8, 0, 0, E);
    const bool full = (iters == 0 || iters >= S.esize) || depth > 0;  // a proof batch runs full tests
    S.iters = full ? S.esize : iters;
    if (!full) {
        Item r; r.kind = IT_RUN; r.run = RUN_PRP; r.start = 0; r.len = S.iters;
        S.q.push_back(r);
        Item rd; rd.kind = IT_READ_RES;
        S.q.push_back(rd);
    } else {
        // B_GerbiczLi (src/genefer.h:467-471) rounded up to a multiple of 64
        const uint64_t L = uint64_t(2) << (ilog2_32((uint32_t)S.esize) / 2);
        uint64_t B = (S.esize - 1) / L + 1;
        B = (B + 63) / 64 * 64;
        // Pietrzak-Li checkpoints (proof batches): r0 after bit i with i % B_PL == 0 goes to
        // register 3 + i / B_PL, B_PL = B_PietrzakLi(esize, depth) (src/genefer.h:473-476, 536-546)
        const uint64_t BPL = depth > 0 ? ((S.esize - 1) >> depth) + 1 : 0;
        // PRP loop: squaring k handles bit i = esize - 1 - k; after bit i with i % B == 0 and
        // i / B != 0, the d(t) update r2 = r0; r0 *= r1; r1 = r0; r0 = r2 (src/genefer.h:529-535),
        // then the checkpoint copy
        uint64_t k = 0;
        while (k < S.esize) {
            const uint64_t i = S.esize - 1 - k;  // first bit of this run
            uint64_t last = (i / B) * B;          // last bit of the run: next GL or PL point below
            if (BPL) last = std::max(last, (i / BPL) * BPL);
            const uint64_t len = i - last + 1;
            Item r; r.kind = IT_RUN; r.run = RUN_PRP; r.start = k; r.len = len;
            S.q.push_back(r);
            k += len;
            if (last != 0 && last % B == 0) {
                Item c; c.kind = IT_COPY; c.a = 2; c.b = 0; S.q.push_back(c);
                Item m; m.kind = IT_INITMUL; m.a = 1; S.q.push_back(m);
                Item u; u.kind = IT_MUL; S.q.push_back(u);
                Item c1; c1.kind = IT_COPY; c1.a = 1; c1.b = 0; S.q.push_back(c1);
                Item c2; c2.kind = IT_COPY; c2.a = 0; c2.b = 2; S.q.push_back(c2);
            }
            if (BPL && last % BPL == 0) {
                Item c; c.kind = IT_COPY; c.a = 3 + (uint32_t)(last / BPL); c.b = 0; S.q.push_back(c);
            }
        }
        Item rd; rd.kind = IT_READ_RES; S.q.push_back(rd);
        // Gerbicz-Li check (src/genefer.h:557-615)
        { Item m; m.kind = IT_INITMUL; m.a = 1; S.q.push_back(m); }
        { Item u; u.kind = IT_MUL; S.q.push_back(u); }
        { Item c; c.kind = IT_COPY; c.a = 2; c.b = 0; S.q.push_back(c); }
        { Item c; c.kind = IT_COPY; c.a = 0; c.b = 1; S.q.push_back(c); }
        { Item r; r.kind = IT_RUN; r.run = RUN_ZERO; r.len = B; S.q.push_back(r); }
        { Item c; c.kind = IT_COPY; c.a = 1; c.b = 0; S.q.push_back(c); }
        mpz_t res;
        mpz_init(res);
        gl_chunk_sum(res, E, (unsigned long)B);
        const size_t rs = mpz_sizeinbase(res, 2);
        for (long i = (long)rs - 1; i >= 0; --i) S.resbits.push_back((uint8_t)mpz_tstbit(res, (mp_bitcnt_t)i));
        mpz_clear(res);
        { Item st; st.kind = IT_SET; st.a = 0; st.b = 1; S.q.push_back(st); }
        { Item r; r.kind = IT_RUN; r.run = RUN_RES; r.len = S.resbits.size(); S.q.push_back(r); }
        { Item m; m.kind = IT_INITMUL; m.a = 1; S.q.push_back(m); }
        { Item u; u.kind = IT_MUL; S.q.push_back(u); }
        { Item h; h.kind = IT_READ_H1; S.q.push_back(h); }
        { Item c; c.kind = IT_COPY; c.a = 0; c.b = 2; S.q.push_back(c); }
        { Item h; h.kind = IT_READ_H2; S.q.push_back(h); }
        if (depth > 0) {  // the proof: mu_0 = checkpoint 0 (the PRP residue)
            S.pl_pending = true;
            S.pl_k = 0;
            S.w.assign(size_t(1) << (depth - 1), Words());
            { Item c; c.kind = IT_COPY; c.a = 0; c.b = 3; S.q.push_back(c); }
            { Item rd; rd.kind = IT_READ_MU; S.q.push_back(rd); }
        }
    }
    mpz_clear(E);
    // slot table and CRT constants; r0 = 1, r1 = 1 (prp: set(1); copy(1, 0))
    SlotInit A;
    A.si.b = b; A.si.rns = S.rns; A.si.is32 = S.is32; A.si.rounds = carry_rounds(b, S.n); A.si.n = (int32_t)S.n;
    A.c = make_crt(S.rns, S.is32, S.n, b);
    A.d = make_f64_crt(S.n, b, f64_primes(b, S.n));
    A.slots = slots_dev; A.crt = crt; A.crt64 = crt64; A.s = s;
    A.r0 = reinterpret_cast<int4 *>(reg(s, 0)); A.r1 = reinterpret_cast<int4 *>(reg(s, 1));
    A.n4 = (uint32_t)(slot_N(s) / 4);
    A.carry = reinterpret_cast<int4 *>(carry) + (size_t)s * (NA / 16);
    A.c4 = (uint32_t)(NA / 16);
    zl = std::max(zl, (uint32_t)s + 1);
    hipLaunchKernelGGL(kb_take_slot, dim3((A.n4 + 255) / 256), dim3(256), 0, stream, A);
    if (slot_out) *slot_out = s;
    return check("submit");
}

int Batch::read_residue(int s, uint32_t reg, gint &g) {
    int rc = check_hip(hipMemcpyAsync(readback, this->reg(s, reg), slot_N(s) * 4, hipMemcpyDeviceToHost, stream),
                       "readback");
    if (rc == GFE_OK) rc = check_hip(hipStreamSynchronize(stream), "readback sync");
    if (rc != GFE_OK) return rc;
    memcpy(g.data(), readback, slot_N(s) * 4);
    g.reset();
    return GFE_OK;
}

// r0 = r_src^e by square-and-multiply (power / powerz, src/genefer.h:441-465): rm = r_src, r0 = 1,
// then for each bit of e from the top a squaring round and, for a one bit, a multiplying round.
void Batch::queue_power(Slot &S, uint32_t src, const Words &e) {
    { Item m; m.kind = IT_INITMUL; m.a = src; S.q.push_back(m); }
    { Item st; st.kind = IT_SET; st.a = 0; st.b = 1; S.q.push_back(st); }
    if (e.empty()) return;
    Item r; r.kind = IT_RUN; r.run = RUN_POW; r.start = S.powseq.size();
    for (size_t wi = e.size(); wi-- > 0;)
        for (int bit = 31; bit >= 0; --bit) {
            if (wi == e.size() - 1 && r.len == 0 && !((e[wi] >> bit) & 1u)) continue;  // leading zeros
            S.powseq.push_back(0);
            if ((e[wi] >> bit) & 1u) S.powseq.push_back(1);
            r.len = S.powseq.size() - r.start;
        }
    S.q.push_back(r);
}

// Phase k >= 1 of the proof up to the read-back of mu_k (src/genefer.h:650-705): with i =
// 2^(depth - k), r1 = ckpt_i^w_0 prod_j ckpt_(i + 2j)^w_j over j = i, 2i, .. < 2^depth / 2, r0 = r1.
void Batch::queue_pl_phase(Slot &S, int k) {
    const size_t L = size_t(1) << depth, i = size_t(1) << (depth - k);
    { Item c; c.kind = IT_COPY; c.a = 0; c.b = 3 + (uint32_t)i; S.q.push_back(c); }
    queue_power(S, 0, S.w[0]);
    { Item c; c.kind = IT_COPY; c.a = 1; c.b = 0; S.q.push_back(c); }
    for (size_t j = i; j < L / 2; j += i) {
        { Item c; c.kind = IT_COPY; c.a = 0; c.b = 3 + (uint32_t)(i + 2 * j); S.q.push_back(c); }
        queue_power(S, 0, S.w[j]);
        { Item m; m.kind = IT_INITMUL; m.a = 1; S.q.push_back(m); }
        { Item u; u.kind = IT_MUL; S.q.push_back(u); }
        { Item c; c.kind = IT_COPY; c.a = 1; c.b = 0; S.q.push_back(c); }
    }
    { Item rd; rd.kind = IT_READ_MU; S.q.push_back(rd); }
}

// mu_k has been read back (r0): record its hash, then queue the rest of phase k -- v1 = v1 mu_k^q
// with q = hash32(mu_k) (for k = 0: v1 = mu_0^q) and the exponent update w_(i/2 + j) = w_j q --
// and phase k + 1, or after mu_depth the read-back of v1, the proof key.
void Batch::pl_read_done(Slot &S, gint &g) {
    const int k = S.pl_k;
    S.mu_hash.push_back(g.gethash64());
    const uint32_t q = g.gethash32();
    queue_power(S, 0, Words{q});
    if (k == 0) {
        S.w[0] = Words{q};
    } else {
        { Item m; m.kind = IT_INITMUL; m.a = 2; S.q.push_back(m); }
        { Item u; u.kind = IT_MUL; S.q.push_back(u); }
        const size_t L = size_t(1) << depth, i = size_t(1) << (depth - k);
        if (i > 1)
            for (size_t j = 0; j < L / 2; j += i) {
                S.w[i / 2 + j] = S.w[j];
                words_mul(S.w[i / 2 + j], q);
            }
    }
    { Item c; c.kind = IT_COPY; c.a = 2; c.b = 0; S.q.push_back(c); }
    S.pl_k = k + 1;
    if (k < depth) {
        queue_pl_phase(S, k + 1);
    } else {
        { Item c; c.kind = IT_COPY; c.a = 0; c.b = 2; S.q.push_back(c); }
        { Item rd; rd.kind = IT_READ_PKEY; S.q.push_back(rd); }
        S.pl_pending = false;
    }
}

// Enqueues the read-back of register 0 of slot s for result item `kind`.
int Batch::read_issue(int s, int kind) {
    if (rfree.empty()) {
        const int rc = read_complete(true);
        if (rc != GFE_OK) return rc;
    }
    const int k = rfree.back();
    rfree.pop_back();
    int rc = check_hip(hipMemcpyAsync(rbuf[k], reg(s, 0), slot_N(s) * 4, hipMemcpyDeviceToHost, stream), "readback");
    if (rc == GFE_OK) rc = check_hip(hipEventRecord(rev[k], stream), "readback event");
    if (rc != GFE_OK) return rc;
    reads.push_back(Read{s, kind, k});
    slots[s].reads_pending++;
    return GFE_OK;
}

// Processes the oldest pending read-back: RES64 / old64 / hash64 (src/gint.h:169-219), or the
// Gerbicz-Li hashes.  Returns 1 when there is none or (wait == false) it has not completed.
int Batch::read_complete(bool wait) {
    if (reads.empty()) return 1;
    const Read r = reads.front();
    if (wait) {
        const int rc = check_hip(hipEventSynchronize(rev[r.buf]), "readback sync");
        if (rc != GFE_OK) return rc;
    } else {
        const hipError_t e = hipEventQuery(rev[r.buf]);
        if (e == hipErrorNotReady) { (void)hipGetLastError(); return 1; }
        if (e != hipSuccess) return check_hip(e, "readback event");
    }
    reads.pop_front();
    Slot &S = slots[r.slot];
    gint gs(slot_N(r.slot), S.b);
    memcpy(gs.data(), rbuf[r.buf], slot_N(r.slot) * 4);
    gs.reset();
    rfree.push_back(r.buf);
    if (r.kind == IT_READ_RES) {
        uint64_t res = 0, old = 0;
        S.is_prp = gs.isOne(res, old) ? 1 : 0;
        S.res64 = res; S.old64 = old;
        S.hash64 = S.is_prp ? 0 : gs.gethash64();
    } else if (r.kind == IT_READ_H1) {
        S.h1 = gs.gethash64();
    } else if (r.kind == IT_READ_MU) {
        pl_read_done(S, gs);
    } else if (r.kind == IT_READ_PKEY) {
        S.pkey = gs.gethash64();
    } else {
        S.gl_ok = (gs.gethash64() == S.h1) ? 1 : 0;
    }
    S.reads_pending--;
    return GFE_OK;
}

// Completed read-backs are processed; slots whose program and read-backs are done move to
// `finished` and become free.
int Batch::harvest() {
    for (;;) {
        const int rc = read_complete(false);
        if (rc == 1) break;
        if (rc != GFE_OK) return rc;
    }
    bool freed = false;
    for (uint32_t s = 0; s < cap; ++s) {
        Slot &S = slots[s];
        if (S.busy && !S.done && S.q.empty() && S.reads_pending == 0 && !S.pl_pending) {
            S.done = true;
            S.t_done = now_s() - t0;
            gfe_batch_result r;
            memset(&r, 0, sizeof(r));
            r.tag = S.tag; r.b = S.b; r.n = S.n; r.res64 = S.res64; r.old64 = S.old64; r.hash64 = S.hash64;
            r.esize = S.esize; r.iters = S.iters; r.is_prp = S.is_prp; r.gl_ok = S.gl_ok;
            r.t_submit = S.t_submit; r.t_done = S.t_done;
            r.depth = S.mu_hash.empty() ? 0 : depth;
            r.pkey = S.pkey;
            for (size_t k = 0; k < S.mu_hash.size() && k < GFE_BATCH_MAX_DEPTH + 1; ++k) r.mu_hash64[k] = S.mu_hash[k];
            finished.push_back(r);
            S.busy = false;
            S.ebits.clear(); S.ebits.shrink_to_fit();
            S.resbits.clear(); S.resbits.shrink_to_fit();
            S.powseq.clear(); S.powseq.shrink_to_fit();
            S.w.clear(); S.mu_hash.clear();
            freed = true;
        }
    }
    if (freed) update_zl();
    return GFE_OK;
}

int Batch::step(int32_t *active_out) {
    std::vector<uint8_t> flags(cap);
    int rc0 = harvest();
    if (rc0 != GFE_OK) return rc0;
    bool issued = false;
    // 1. register operations, grouped by (kind, arguments) across slots
    for (;;) {
        std::map<std::tuple<int, uint32_t, uint32_t, uint32_t>, std::vector<int>> groups;
        for (uint32_t s = 0; s < cap; ++s) {
            Slot &S = slots[s];
            if (!S.busy || S.done || S.q.empty()) continue;
            const Item &it = S.q.front();
            if (it.kind == IT_RUN) continue;
            groups[std::make_tuple(it.kind, it.a, it.b, S.n)].push_back((int)s);
        }
        if (groups.empty()) break;
        flush_carries();
        const bool m64 = mode64();
        rc0 = use_mode(m64);
        if (rc0 != GFE_OK) return rc0;
        for (auto &kv : groups) {
            const int kind = std::get<0>(kv.first);
            const uint32_t a = std::get<1>(kv.first), b2 = std::get<2>(kv.first);
            issued = true;
            if (kind == IT_READ_RES || kind == IT_READ_H1 || kind == IT_READ_H2 || kind == IT_READ_MU ||
                kind == IT_READ_PKEY) {
                for (int s : kv.second) {
                    const int rc = read_issue(s, kind);
                    if (rc != GFE_OK) return rc;
                    slots[s].q.pop_front();
                }
                continue;
            }
            std::fill(flags.begin(), flags.end(), 0);
            for (int s : kv.second) flags[s] = 1;
            uint8_t *st = stage_acquire();
            memcpy(st, flags.data(), cap);
            int rc = check_hip(hipMemcpyAsync(act_dev, st, cap, hipMemcpyHostToDevice, stream), "flags");
            stage_release();
            if (rc != GFE_OK) return rc;
            with_n(std::get<3>(kv.first), [&]() {
                switch (kind) {
                    case IT_COPY: op_copy(act_dev, a, b2); break;
                    case IT_SET: op_set(act_dev, a, (int32_t)b2); break;
                    case IT_INITMUL: op_initmul(act_dev, a); break;
                    case IT_MUL: op_mul(act_dev); break;
                }
            });
            rc = check("op");
            if (rc != GFE_OK) return rc;
            for (int s : kv.second) {
                if (kind == IT_INITMUL) slots[s].zp64 = m64;
                slots[s].q.pop_front();
            }
        }
    }
    // 2. one block of up to 64 squaring rounds
    int rounds = 0;
    uint32_t nact = 0, nbig = 0;
    std::vector<uint64_t> len(cap, 0);
    for (uint32_t s = 0; s < cap; ++s) {
        Slot &S = slots[s];
        if (!S.busy || S.done || S.q.empty() || S.q.front().kind != IT_RUN) continue;
        len[s] = std::min<uint64_t>(64, S.q.front().len - S.pos);
        rounds = std::max(rounds, (int)len[s]);
        ++nact;
        if (S.n == nalloc) ++nbig;
    }
    if (rounds > 0) {
        uint8_t *st = stage_acquire();
        uint8_t *act = st, *dup = st + (size_t)64 * cap, *mul = st + (size_t)128 * cap;
        memset(st, 0, (size_t)3 * 64 * cap);
        bool has_mul = false;
        for (uint32_t s = 0; s < cap; ++s) {
            if (!len[s]) continue;
            const Slot &S = slots[s];
            const Item &it = S.q.front();
            for (uint64_t r = 0; r < len[s]; ++r) {
                act[r * cap + s] = 1;
                const uint64_t k = S.pos + r;
                uint8_t d = 0;
                if (it.run == RUN_PRP) d = S.bit(it.start + k) ? 1 : 0;
                else if (it.run == RUN_RES) d = S.resbits[k];
                else if (it.run == RUN_POW && S.powseq[it.start + k]) {
                    mul[r * cap + s] = 1;
                    has_mul = true;
                }
                dup[r * cap + s] = d;
            }
        }
        int rc = check_hip(hipMemcpyAsync(act_dev, act, (size_t)rounds * cap, hipMemcpyHostToDevice, stream), "act");
        if (rc == GFE_OK) rc = check_hip(hipMemcpyAsync(dup_dev, dup, (size_t)rounds * cap, hipMemcpyHostToDevice, stream), "dup");
        if (rc == GFE_OK) rc = check_hip(hipMemcpyAsync(mul_dev, mul, (size_t)rounds * cap, hipMemcpyHostToDevice, stream), "mul");
        stage_release();
        if (rc != GFE_OK) return rc;
        rc = run_block(rounds, nact, has_mul, nbig);
        if (rc != GFE_OK) return rc;
        if ((int)blk_q.size() == NBLK) {
            rc = check_hip(hipEventSynchronize(blk_ev[blk_q.front()]), "block sync");
            if (rc != GFE_OK) return rc;
            blk_q.pop_front();
        }
        rc = check_hip(hipEventRecord(blk_ev[blk_next], stream), "block event");
        if (rc != GFE_OK) return rc;
        blk_q.push_back(blk_next);
        blk_next = (blk_next + 1) % NBLK;
        issued = true;
        for (uint32_t s = 0; s < cap; ++s) {
            if (!len[s]) continue;
            Slot &S = slots[s];
            S.pos += len[s];
            if (S.pos == S.q.front().len) {
                S.q.pop_front();
                S.pos = 0;
            }
        }
    }
    // 3. nothing to enqueue but read-backs outstanding: wait for the oldest, so that repeated
    // steps always make progress.
    if (!issued && !reads.empty()) {
        const int rc = read_complete(true);
        if (rc != GFE_OK) return rc;
    }
    const int rc = harvest();
    if (rc != GFE_OK) return rc;
    if (active_out) {
        int a = 0;
        for (auto &S : slots) a += S.busy ? 1 : 0;
        *active_out = a;
    }
    return GFE_OK;
}

}  // namespace gfe

// ================================================================================================
// C ABI

using gfe::Batch;
using gfe::set_error;

struct gfe_batch {
    Batch bt;
};

extern "C" {

size_t gfe_batch_slot_bytes(uint32_t n) { return gfe_batch_proof_slot_bytes(n, 0); }

size_t gfe_batch_proof_slot_bytes(uint32_t n, uint32_t depth) {
    const size_t N = (size_t)1 << n;
    const size_t regs = depth > 0 ? 3 + ((size_t)1 << depth) : 3;
    return (regs + 6) * N * 4 + (N >> 3) * 8 + sizeof(gfe::CrtConst) + sizeof(gfe::F64Crt) + sizeof(gfe::SlotInfo);
}


static int batch_create(uint32_t n, uint32_t capacity, uint32_t depth, bool mixed, int device, gfe_batch **out) {
    if (!out) return set_error(GFE_EINVAL, "null output");
    *out = nullptr;
    if (n < 12 || n > 23) return set_error(GFE_EINVAL, "n must be in [12, 23]");
    if (capacity < 1 || capacity > 65535) return set_error(GFE_EINVAL, "capacity must be in [1, 65535]");
    if (depth > GFE_BATCH_MAX_DEPTH) return set_error(GFE_EINVAL, "depth must be in [0, " + std::to_string(GFE_BATCH_MAX_DEPTH) + "]");
    gfe_batch *b = new gfe_batch;
    const int rc = b->bt.init(n, capacity, device, (int)depth, mixed);
    if (rc != GFE_OK) {
        const std::string msg = gfe::g_last_error;
        delete b;
        return set_error(rc, msg);
    }
    *out = b;
    return GFE_OK;
}

int gfe_batch_create(uint32_t n, uint32_t capacity, int device, gfe_batch **out) {
    return batch_create(n, capacity, 0, false, device, out);
}

int gfe_batch_create_proof(uint32_t n, uint32_t capacity, uint32_t depth, int device, gfe_batch **out) {
    return batch_create(n, capacity, depth, false, device, out);
}

int gfe_batch_create_mixed(uint32_t capacity, int device, gfe_batch **out) {
    return batch_create(13, capacity, 0, true, device, out);
}

int gfe_batch_destroy(gfe_batch *b) {
    delete b;
    return GFE_OK;
}

int gfe_batch_info(const gfe_batch *b, char *buf, size_t len) {
    if (!b || !buf || len == 0) return set_error(GFE_EINVAL, "info");
    std::ostringstream ss;
    ss << "batch n=" << b->bt.n << " capacity=" << b->bt.cap << "; " << gfe::plan_str(b->bt.plan, b->bt.n);
    if (b->bt.f64) ss << "; " << gfe::f64_str(b->bt.n, 0, b->bt.shape);
    snprintf(buf, len, "%s", ss.str().c_str());
    return GFE_OK;
}

int gfe_batch_submit(gfe_batch *b, uint32_t base, uint64_t iters, uint64_t tag, int32_t *slot) {
    return gfe_batch_submit_n(b, b ? b->bt.nalloc : 0, base, iters, tag, slot);
}

int gfe_batch_submit_n(gfe_batch *b, uint32_t n, uint32_t base, uint64_t iters, uint64_t tag, int32_t *slot) {
    if (!b) return set_error(GFE_EINVAL, "null batch");
    if (base < 1024 || base > 2000000000u) return set_error(GFE_EINVAL, "b must be in [1024, 2000000000]");
    if (hipSetDevice(b->bt.device) != hipSuccess) return set_error(GFE_EHIP, "hipSetDevice");
    return b->bt.submit(base, iters, tag, slot, n);
}

int gfe_batch_step(gfe_batch *b, int32_t *active) {
    if (!b) return set_error(GFE_EINVAL, "null batch");
    if (hipSetDevice(b->bt.device) != hipSuccess) return set_error(GFE_EHIP, "hipSetDevice");
    return b->bt.step(active);
}

int gfe_batch_poll(gfe_batch *b, gfe_batch_result *out, uint32_t max, uint32_t *count) {
    if (!b || !count) return set_error(GFE_EINVAL, "poll");
    if (hipSetDevice(b->bt.device) != hipSuccess) return set_error(GFE_EHIP, "hipSetDevice");
    const int rc = b->bt.harvest();
    if (rc != GFE_OK) return rc;
    uint32_t k = 0;
    auto &f = b->bt.finished;
    while (k < max && !f.empty() && out) {
        out[k++] = f.front();
        f.pop_front();
    }
    *count = k;
    return GFE_OK;
}

int gfe_batch_active(const gfe_batch *b) {
    if (!b) return 0;
    int a = 0;
    for (auto &S : b->bt.slots) a += S.busy ? 1 : 0;
    return a;
}

int gfe_batch_get_plan(const gfe_batch *b, int32_t plan[6]) {
    if (!b || !plan) return set_error(GFE_EINVAL, "get_plan");
    gfe::plan_to_array(b->bt.plan, plan);
    return GFE_OK;
}

int gfe_batch_set_plan(gfe_batch *b, const int32_t plan[6]) {
    if (!b || !plan) return set_error(GFE_EINVAL, "set_plan");
    gfe::Plan P;
    if (!gfe::plan_from_array(plan, b->bt.n, &P)) return set_error(GFE_EINVAL, "plan not admissible for this n");
    if (P.limb) return set_error(GFE_EINVAL, "a batch does not run the two-digit-limb transform");
    if (b->bt.mixed && (!P.spec || !P.fuse_sq))
        return set_error(GFE_EINVAL, "a mixed batch keeps compile-time passes and the single-workgroup squaring");
    if (hipSetDevice(b->bt.device) != hipSuccess) return set_error(GFE_EHIP, "hipSetDevice");
    const int rc = b->bt.int_tables();
    if (rc != GFE_OK) return rc;
    b->bt.flush_carries();
    if (b->bt.zero_carries() != GFE_OK || hipStreamSynchronize(b->bt.stream) != hipSuccess)
        return set_error(GFE_EHIP, "set_plan sync");
    b->bt.plan = P;
    b->bt.f64 = false;
    b->bt.drop_graphs();
    return GFE_OK;
}

int gfe_batch_set_graphs(gfe_batch *b, int on) {
    if (!b) return set_error(GFE_EINVAL, "null batch");
    if (hipSetDevice(b->bt.device) != hipSuccess || hipStreamSynchronize(b->bt.stream) != hipSuccess)
        return set_error(GFE_EHIP, "set_graphs sync");
    b->bt.use_graphs = on != 0;
    if (!on) b->bt.drop_graphs();
    return GFE_OK;
}

int gfe_batch_backlog(gfe_batch *b) {
    if (!b) return set_error(GFE_EINVAL, "null batch");
    if (hipSetDevice(b->bt.device) != hipSuccess) return set_error(GFE_EHIP, "hipSetDevice");
    return b->bt.backlog();
}

size_t gfe_batch_device_bytes(uint32_t n, uint32_t capacity) { return gfe_batch_proof_device_bytes(n, capacity, 0); }

size_t gfe_batch_proof_device_bytes(uint32_t n, uint32_t capacity, uint32_t depth) {
    const size_t tables = n <= gfe::F64_ALL_BASES_N ? gfe::F64_PRIMES * gfe::f64_tw_words(n) * 8 : (size_t)24 << n;
    return (size_t)capacity * (gfe_batch_proof_slot_bytes(n, depth) + 3 * 64) + tables;
}

int gfe_batch_get_digits(gfe_batch *b, int32_t slot, uint32_t reg, int32_t *out) {
    if (!b || !out || slot < 0 || (uint32_t)slot >= b->bt.cap || reg >= b->bt.nregs) return set_error(GFE_EINVAL, "get_digits");
    if (hipSetDevice(b->bt.device) != hipSuccess) return set_error(GFE_EHIP, "hipSetDevice");
    gfe::gint g(b->bt.slot_N(slot), b->bt.slots[slot].busy ? b->bt.slots[slot].b : 2);
    b->bt.flush_carries();
    const int rc = b->bt.read_residue(slot, reg, g);
    if (rc != GFE_OK) return rc;
    memcpy(out, g.data(), b->bt.slot_N(slot) * 4);
    return GFE_OK;
}

int gfe_batch_time_rounds(gfe_batch *b, uint32_t rounds, double *ms) {
    if (!b || !ms || rounds == 0) return set_error(GFE_EINVAL, "time_rounds");
    Batch &B = b->bt;
    if (hipSetDevice(B.device) != hipSuccess) return set_error(GFE_EHIP, "hipSetDevice");
    // every round: the busy slots square without doubling (64 flag rows, as a squaring block)
    uint8_t *st = B.stage_acquire();
    memset(st, 0, (size_t)3 * 64 * B.cap);
    uint32_t nact = 0, nbig = 0;
    for (uint32_t s = 0; s < B.cap; ++s) {
        nact += B.slots[s].busy ? 1 : 0;
        nbig += (B.slots[s].busy && B.slots[s].n == B.nalloc) ? 1 : 0;
    }
    for (uint32_t r = 0; r < 64; ++r)
        for (uint32_t s = 0; s < B.cap; ++s) st[(size_t)r * B.cap + s] = B.slots[s].busy ? 1 : 0;
    int rc = gfe::check_hip(hipMemcpyAsync(B.act_dev, st, (size_t)64 * B.cap, hipMemcpyHostToDevice, B.stream), "act");
    if (rc == GFE_OK)
        rc = gfe::check_hip(hipMemcpyAsync(B.dup_dev, st + (size_t)64 * B.cap, (size_t)64 * B.cap, hipMemcpyHostToDevice, B.stream), "dup");
    if (rc == GFE_OK)
        rc = gfe::check_hip(hipMemcpyAsync(B.mul_dev, st + (size_t)128 * B.cap, (size_t)64 * B.cap, hipMemcpyHostToDevice, B.stream), "mul");
    B.stage_release();
    if (rc != GFE_OK) return rc;
    // captured blocks are built before the timed region
    const bool m64 = B.mode64();
    rc = B.use_mode(m64);
    if (rc != GFE_OK) return rc;
    const bool four_step = m64 ? true : B.mixed ? (nbig > 0 && nbig < 128) : !B.fused_block(nact);
    if (B.use_graphs && (m64 || !B.plan.pipe) && four_step) {
        if (rounds >= 64 && !B.block_graph(64)) return set_error(GFE_EHIP, "squaring block graph capture failed");
        if ((rounds % 64) && !B.block_graph((int)(rounds % 64))) return set_error(GFE_EHIP, "squaring block graph capture failed");
    }
    (void)hipEventRecord(B.ev0, B.stream);
    for (uint32_t done = 0; done < rounds;) {
        const int r = (int)std::min<uint32_t>(64, rounds - done);
        rc = B.run_block(r, nact, false, nbig);
        if (rc != GFE_OK) return rc;
        done += (uint32_t)r;
    }
    (void)hipEventRecord(B.ev1, B.stream);
    rc = gfe::check_hip(hipEventSynchronize(B.ev1), "time sync");
    if (rc != GFE_OK) return rc;
    float t = 0;
    (void)hipEventElapsedTime(&t, B.ev0, B.ev1);
    *ms = t;
    return B.check("time_rounds");
}

int gfe_batch_tune(gfe_batch *b, uint32_t reps) {
    if (!b) return set_error(GFE_EINVAL, "null batch");
    Batch &B = b->bt;
    if (hipSetDevice(B.device) != hipSuccess) return set_error(GFE_EHIP, "hipSetDevice");
    if (reps == 0) reps = 4;
    if (B.mixed) return set_error(GFE_EINVAL, "a mixed batch keeps its plan (not tuned)");
    bool any = false;
    for (auto &S : B.slots) any |= S.busy;
    if (!any) return set_error(GFE_EINVAL, "tune needs busy slots");
    const int rct = B.int_tables();
    if (rct != GFE_OK) return rct;
    const std::vector<gfe::Plan> plans = gfe::candidate_plans(B.n);
    B.flush_carries();
    // squarings on the busy slots' r0: save and restore register 0 of every slot
    const size_t row = B.NA * 4, pitch = (size_t)B.nregs * B.NA * 4;
    int32_t *save = nullptr;
    if (hipMalloc(&save, (size_t)B.cap * row) != hipSuccess) return set_error(GFE_ENOMEM, "tune save");
    (void)hipMemcpy2DAsync(save, row, B.regs, pitch, row, B.cap, hipMemcpyDeviceToDevice, B.stream);
    const gfe::Plan orig = B.plan;
    B.timed64 = 0;
    gfe::Plan best = orig;
    double best_ms = 1e30;
    const bool graphs = B.use_graphs;
    B.use_graphs = false;  // plans are compared on eager launches (no capture per candidate plan)
    // every plan on `reps` rounds, then the fastest eight again on 8 x reps rounds
    std::vector<std::pair<double, size_t>> screen;
    for (size_t k = 0; k < plans.size(); ++k) {
        B.plan = plans[k];
        if (B.zero_carries() != GFE_OK) break;
        double ms = 0;
        if (gfe_batch_time_rounds(b, 1, &ms) != GFE_OK) continue;
        if (gfe_batch_time_rounds(b, reps, &ms) != GFE_OK) continue;
        screen.emplace_back(ms, k);
    }
    std::sort(screen.begin(), screen.end());
    std::vector<std::pair<double, size_t>> fin;
    for (size_t j = 0; j < std::min<size_t>(8, screen.size()); ++j) {
        B.plan = plans[screen[j].second];
        if (B.zero_carries() != GFE_OK) break;
        double ms = 0;
        if (gfe_batch_time_rounds(b, 1, &ms) != GFE_OK) continue;
        if (gfe_batch_time_rounds(b, 8 * reps, &ms) != GFE_OK) continue;
        fin.emplace_back(ms, screen[j].second);
        if (ms < best_ms) { best_ms = ms; best = plans[screen[j].second]; }
    }
    // the three fastest again as the batch runs its blocks (captured 64-round graphs, when on),
    // in turn twice, each kept at its better time: eager timings rank the plans, but graph
    // launches save each plan a different share of its launch overhead
    if (graphs && fin.size() > 1) {
        std::sort(fin.begin(), fin.end());
        const size_t m = std::min<size_t>(3, fin.size());
        std::vector<double> t(m, 1e30);
        B.use_graphs = true;
        for (int pass = 0; pass < 2; ++pass)
            for (size_t i = 0; i < m; ++i) {
                B.plan = plans[fin[i].second];
                B.drop_graphs();
                if (B.zero_carries() != GFE_OK) break;
                double ms = 0;
                if (gfe_batch_time_rounds(b, 64, &ms) != GFE_OK) continue;
                if (gfe_batch_time_rounds(b, 128, &ms) != GFE_OK) continue;
                t[i] = std::min(t[i], ms);
            }
        size_t bi = 0;
        for (size_t i = 1; i < m; ++i)
            if (t[i] < t[bi]) bi = i;
        if (t[bi] < 1e30) best = plans[fin[bi].second];
    }
    B.plan = best;
    B.use_graphs = graphs;
    B.drop_graphs();
    (void)B.zero_carries();
    if (B.n <= gfe::F64_ALL_BASES_N) {  // the double-precision transform against the chosen plan, as blocks run
        double t[2] = {1e30, 1e30};
        for (int pass = 0; pass < 4; ++pass) {
            B.timed64 = pass & 1;
            double ms = 0;
            if (gfe_batch_time_rounds(b, 64, &ms) != GFE_OK || gfe_batch_time_rounds(b, 128, &ms) != GFE_OK) continue;
            t[pass & 1] = std::min(t[pass & 1], ms);
        }
        B.f64 = t[1] < t[0];
        B.drop_graphs();
        (void)B.zero_carries();
    }
    B.timed64 = -1;
    (void)hipMemcpy2DAsync(B.regs, pitch, save, row, row, B.cap, hipMemcpyDeviceToDevice, B.stream);
    (void)hipStreamSynchronize(B.stream);
    (void)hipFree(save);
    return B.check("tune");
}

int gfe_batch_run(uint32_t n, const uint32_t *b, uint32_t count, uint64_t iters, uint32_t capacity, int device,
                  gfe_batch_result *results) {
    if (!b || !results || count == 0) return set_error(GFE_EINVAL, "batch_run");
    gfe_batch *bt = nullptr;
    int rc = gfe_batch_create(n, std::min(count, capacity ? capacity : count), device, &bt);
    if (rc != GFE_OK) return rc;
    uint32_t next = 0, done = 0;
    std::vector<gfe_batch_result> buf(bt->bt.cap);
    while (done < count) {
        while (next < count) {
            int32_t slot;
            rc = gfe_batch_submit(bt, b[next], iters, next, &slot);
            if (rc == GFE_EFULL) break;
            if (rc != GFE_OK) { gfe_batch_destroy(bt); return rc; }
            ++next;
        }
        int32_t active = 0;
        rc = gfe_batch_step(bt, &active);
        if (rc != GFE_OK) { gfe_batch_destroy(bt); return rc; }
        uint32_t got = 0;
        gfe_batch_poll(bt, buf.data(), (uint32_t)buf.size(), &got);
        for (uint32_t k = 0; k < got; ++k) results[buf[k].tag] = buf[k];
        done += got;
    }
    gfe_batch_destroy(bt);
    return GFE_OK;
}

}  // extern "C"
