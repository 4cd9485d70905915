// gfe_noalloc.hip -- squarings that allocate nothing (gfe_square_noalloc, include/gfe.h).
//
// For callers that cannot call hipMalloc (code under HIP graph capture, tight serving loops,
// harnesses that forbid allocation): the caller owns the digits, and everything else a squaring
// needs -- the transform work space, the twiddle tables, the normalisation carries and the CRT
// constants -- lives in `scratch`, one static device array per device, held until the process ends.
// The squarings run the engine's own passes in double precision (Engine::bind), so the digits equal
// those of gfe_square_dup on an engine of the same (b, n).
//
// Every call rebuilds the twiddles and the CRT constants for its (b, n) with two small kernels (no
// host staging, no memset, no copy), so a call never depends on what an earlier call left in the
// array; calls that overlap on one device race on it.
#include <hip/hip_runtime.h>

#include <mutex>
#include <string>

#include "../../include/gfe.h"
#include "gfe_engine.h"

namespace gfe {

namespace {

constexpr size_t NA_N = (size_t)1 << GFE_NOALLOC_MAX_N;
constexpr size_t NA_WS = 3 * NA_N * 4;      // 3 x N/2 residues of 8 bytes
constexpr size_t NA_TW = 3 * NA_N * 4;      // twiddles (a quarter of it) and CRT constants
constexpr size_t NA_CARRY = NA_N;           // range carries, as the engine's carry buffer
constexpr size_t NA_PAD = 256;
static_assert(F64_PRIMES * NA_N + sizeof(F64Crt) <= NA_TW, "tables and constants fit their slot");
static_assert(NA_WS + NA_TW + NA_CARRY + NA_PAD == GFE_NOALLOC_BYTES, "the documented size is the array's");
static_assert(GFE_NOALLOC_MAX_N <= F64_ALL_BASES_N, "the double-precision transform covers every base");

// The library's scratch array.  Host code never uses this name as an address: the device address
// of each device's copy comes from hipGetSymbolAddress (scratch_on).
static __device__ __align__(256) unsigned char scratch[GFE_NOALLOC_BYTES];

constexpr int NA_MAX_DEV = 64;
std::mutex g_na_mu;
void *g_na_ptr[NA_MAX_DEV] = {};

// Device address of `scratch` on the current device `dev`, looked up once per device.
int scratch_on(int dev, unsigned char **out) {
    std::lock_guard<std::mutex> lk(g_na_mu);
    if (!g_na_ptr[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return set_error(GFE_EHIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        g_na_ptr[dev] = p;
    }
    *out = static_cast<unsigned char *>(g_na_ptr[dev]);
    return GFE_OK;
}

__global__ void k_na_crt(F64Crt c, F64Crt *dst) {
    if (threadIdx.x == 0) *dst = c;
}

}  // namespace

}  // namespace gfe

extern "C" int gfe_square_noalloc(uint32_t b, uint32_t n, int device, int32_t *digits, uint32_t count,
                                  uint64_t dup_bits, void *stream) {
    using namespace gfe;
    if (n < 12 || n > GFE_NOALLOC_MAX_N)
        return set_error(GFE_EINVAL, "square_noalloc: n must be in [12, " + std::to_string(GFE_NOALLOC_MAX_N) +
                                         "] (the scratch array's limit)");
    if (b < 1024 || b > 2000000000u) return set_error(GFE_EINVAL, "square_noalloc: b must be in [1024, 2000000000]");
    if (!digits) return set_error(GFE_EINVAL, "square_noalloc: null digits");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return set_error(GFE_ENODEV, "no HIP device");
    if (device < 0 || device >= ndev || device >= NA_MAX_DEV) return set_error(GFE_ENODEV, "device index out of range");
    hipPointerAttribute_t attr;
    if (hipPointerGetAttributes(&attr, digits) != hipSuccess || attr.type != hipMemoryTypeDevice ||
        attr.device != device) {
        (void)hipGetLastError();
        return set_error(GFE_EINVAL, "square_noalloc: digits must be device memory of the given device");
    }
    if (hipSetDevice(device) != hipSuccess) return set_error(GFE_EHIP, "hipSetDevice failed");
    unsigned char *base = nullptr;
    int rc = scratch_on(device, &base);
    if (rc != GFE_OK) return rc;
    if (count == 0) return GFE_OK;
    engine_set_lds_attributes();

    double *tw = reinterpret_cast<double *>(base + NA_WS);
    F64Crt *crt = reinterpret_cast<F64Crt *>(base + NA_WS + F64_PRIMES * NA_N);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (f64_build_twiddles(n, tw, s) != 0) return set_error(GFE_EHIP, "square_noalloc: twiddles");
    hipLaunchKernelGGL(k_na_crt, dim3(1), dim3(64), 0, s, make_f64_crt(n, b, f64_primes(b, n)), crt);

    Engine e;
    e.bind(b, n, device, s, digits, base, tw, reinterpret_cast<int64_t *>(base + NA_WS + NA_TW), crt);
    for (uint32_t i = 0; i < count; ++i) e.square((int)((dup_bits >> (i % 64)) & 1));
    e.flush_carry();
    return e.check("square_noalloc");
}
