// cd_noalloc.hip -- non-dominated sorting that allocates nothing.
//
// cd_nds may allocate device memory for its scratch (the domination bit
// matrix, dominator counts, selection state and work list).  Callers that
// cannot allocate device memory (code under graph capture, tight serving
// loops) use cd_nds_noalloc instead: the same sort in kernels of its own
// (k_sort_tiles, k_sort_fronts) over the caller's device buffers, with the
// scratch in one file-scope device array of fixed size that every GPU holds
// for the life of the process.
// Every call on a GPU shares that GPU's array, so calls that overlap on one
// GPU (different streams, other host threads) race; calls in one stream are
// ordered.  Every call writes all of the scratch that it reads.
#include <hip/hip_runtime.h>

#include <mutex>
#include <string>

#include "cd_host.h"

namespace {

constexpr int MAX_POOL = CD_NOALLOC_MAX_POOL;
constexpr int MAX_WORDS = (MAX_POOL + 63) / 64;

constexpr size_t a256(size_t x) { return (x + 255) & ~(size_t)255; }
constexpr size_t OFF_DOM = 0;
constexpr size_t OFF_ANY = OFF_DOM + a256((size_t)MAX_POOL * MAX_WORDS * 8);
constexpr size_t SCRATCH_BYTES = OFF_ANY + a256((size_t)MAX_WORDS * MAX_WORDS * 8);

// The scratch of cd_nds_noalloc on every GPU (about 8.2 MiB).  Host code uses
// the address hipGetSymbolAddress returns for the current device, never this
// name.
static __device__ __align__(256) uint8_t scratch[SCRATCH_BYTES];

std::mutex g_mu;
constexpr int MAX_DEVICES = 64;
uint8_t *g_scratch[MAX_DEVICES];  // per device: the device address of `scratch`

// The address of the current device's scratch, looked up once per device.
int scratch_of_current_device(uint8_t **out) {
    int dev = -1;
    HIPCHK(hipGetDevice(&dev));
    if (dev < 0 || dev >= MAX_DEVICES) return cdhost::fail(CD_E_DEVICE, "device ordinal out of range");
    std::lock_guard<std::mutex> lk(g_mu);
    if (!g_scratch[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return cdhost::fail(CD_E_DEVICE, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        g_scratch[dev] = (uint8_t *)p;
    }
    *out = g_scratch[dev];
    return CD_OK;
}

}  // namespace

extern "C" int cd_nds_noalloc(const float *obj, int32_t P, int32_t N, int32_t *front_of, int32_t *n_fronts,
                              void *stream) {
    if (!obj || !front_of || !n_fronts) return cdhost::fail(CD_E_INVALID, "null device buffer");
    if (P < 1 || N < 1 || N > P) return cdhost::fail(CD_E_INVALID, "need 1 <= N <= P");
    if (P > MAX_POOL)
        return cdhost::fail(CD_E_INVALID, "pool of " + std::to_string(P) + " designs exceeds cd_nds_noalloc's maximum of " +
                                              std::to_string(MAX_POOL));
    uint8_t *base = nullptr;
    const int rc = scratch_of_current_device(&base);
    if (rc != CD_OK) return rc;
    const int W = (P + 63) / 64;
    HIPCHK(cd::launch_sort(cd::SortArgs{obj, front_of, n_fronts, (uint64_t *)(base + OFF_DOM), (uint64_t *)(base + OFF_ANY), P, N, W},
                           (hipStream_t)stream));
    return CD_OK;
}
