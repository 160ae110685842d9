// sph_sort.hip - stable LSD radix sort of (key, value) uint32 pairs for gfx950.
//
// Replaces RadixSum / RadixPrefixSum / RadixAddOffsetsAndShuffle
// (source/CUDA/radixsort_kernel.cu:70-432, driver :445-472).  Contract kept:
// a stable sort of 8-byte pairs by key, 8 key bits per pass, so that pairs
// (hash, index) given in index order come out in lexicographic
// (hash, index) order.  The pass count follows the key width the caller
// asks for (ceil(log2(numCells)) bits) instead of the reference's fixed 16
// or 32 bits.
//
// Structure:
//   histogram     per tile, the digit counts of every pass in one read of the
//                 keys, added to the sort's counts with one atomic per digit;
//                 the last tile to finish scans them -> digit offsets;
//   pass (x bits/8)  per tile: stable local ranking with 64-lane ballots (peer
//                 mask per digit, rank = popcount of lower peers), tile digit
//                 counts published and prefixed across tiles by a look-back
//                 over spans of 16, of 16 spans and so on, local reorder in
//                 LDS, coalesced runs written to each digit's global range.
// A tile is 4096 pairs on 1024 threads, four to a thread: with 256 tiles at 1M
// a CU has one tile, and sixteen waves rank it in a quarter of the time of
// four.  The tiles of such a sort all publish at about the same time, so a
// tile has to add up every count before it; sums over spans of 16 tiles, over
// 16 spans and so on make that one short round of loads a level (a pass at
// 1,000,003 random keys with 256 tiles: one count at a time 28 us, 64 counts a
// round 20.6 us, spans 14.2 us; 134,217,728 pairs, three passes and the
// histogram: 5.5 ms, with spans of tiles as the only sums 27.6 ms).
//
// Two forms:
//   k_hist, k_pass  one launch each (the stand-alone sort);
//   sort_slots      (sph_sort_device.hpp) every tile of every pass by the
//                 blocks of one launch: k_resort_place runs it first on a
//                 step whose order cannot be built from the last one, so that
//                 the others pay no launch for it and a captured graph has it.
// Every wait is bounded by a spin limit that records an error instead of
// hanging.  Look-back words carry the launch's epoch, and the last block
// leaves every counter at zero, so nothing needs clearing between sorts.
#include <algorithm>
#include <mutex>

#include "sph_sort_device.hpp"

namespace sph {
using namespace sortdev;
namespace {

__global__ __launch_bounds__(kSortBlock) void k_hist(const uint32_t* __restrict__ pairs, uint32_t n, uint32_t bits,
                                                     uint32_t* __restrict__ counts, uint32_t* __restrict__ offsets,
                                                     uint32_t* __restrict__ ctl, uint2* __restrict__ copy) {
    __shared__ SortShared S;
    (void)hist_tile<2>(S, blockIdx.x, gridDim.x, pairs, n, bits, counts, offsets, ctl, copy);
}

// Tiles are numbered by a ticket, so that a tile only ever waits for tiles
// that started before it; the last ticket's holder leaves the counter at zero.
__global__ __launch_bounds__(kSortBlock) void k_pass(const uint32_t* __restrict__ in, uint32_t* __restrict__ out,
                                                     uint32_t n, uint32_t pass, uint32_t bits, uint32_t epoch,
                                                     const uint32_t* __restrict__ offsets,
                                                     uint64_t* __restrict__ status, uint32_t* __restrict__ ctl,
                                                     uint32_t* __restrict__ err) {
    __shared__ SortShared S;
    if (threadIdx.x == 0) {
        S.word = atomicAdd(&ctl[kCtlPass + pass * kLine], 1u);
        if (S.word == gridDim.x - 1) ctl[kCtlPass + pass * kLine] = 0u;
    }
    __syncthreads();
    pass_tile<true>(S, S.word, gridDim.x, epoch, in, nullptr, out, nullptr, n, 8 * pass, digit_bits(bits, pass),
                    offsets + pass * kRadix, status, err);
}

}  // namespace

uint32_t radix_num_tiles(uint32_t n) {
    const uint32_t tiles = (n + kTile - 1) / kTile;
    return tiles == 0 ? 1 : tiles;
}

namespace {

// Scratch layout: digit counts | digit offsets | control words | look-back
// words (a row of one per digit for each tile, for each span of tiles, ...).
constexpr size_t kDigits = (size_t)kMaxPasses * kRadix;
constexpr size_t kHeadBytes = 2 * kDigits * 4 + kCtlNum * 4;
static_assert(kHeadBytes % 8 == 0, "the status words are 8 bytes each");

constexpr size_t scratch_bytes_for_tiles(uint32_t tiles) {
    return kHeadBytes + (size_t)look_back_rows(tiles) * kRadix * 8;
}

void carve(RadixSortPlan& plan, uint32_t n, void* scratch) {
    plan.n = n;
    plan.num_tiles = radix_num_tiles(n);
    plan.counts = static_cast<uint32_t*>(scratch);
    plan.digit_off = plan.counts + kDigits;
    plan.ctl = plan.digit_off + kDigits;
    plan.err = plan.ctl + kCtlErr;
    plan.status = reinterpret_cast<uint64_t*>(plan.ctl + kCtlNum);
}

}  // namespace

size_t radix_scratch_bytes(uint32_t n) { return scratch_bytes_for_tiles(radix_num_tiles(n)); }

hipError_t radix_plan_init(RadixSortPlan& plan, uint32_t n, void* scratch, hipStream_t stream) {
    carve(plan, n, scratch);
    return hipMemsetAsync(scratch, 0, radix_scratch_bytes(n), stream);
}

// Stable LSD sort of plan.n (key, value) pairs in place in `pairs` (the
// KeyValuePair layout: key, value interleaved) with `temp` (plan.n pairs) as
// the ping-pong buffer (for an odd number of passes the histogram, which
// reads every pair's line anyway, copies the pairs to `temp`, from where the
// passes start: a copy back at the end took 5.4 us and a launch at 1,000,003
// pairs, the histogram 14.5 with it and 12.5 without; the call 87 -> 82 us, at
// 4,000,003 pairs 299 -> 220).
// `epoch` and the kMaxPasses - 1 numbers after it mark this sort's look-back
// words: no earlier sort in the same scratch used them, and the control words
// are zero.
hipError_t radix_sort_kv(const RadixSortPlan& plan, uint32_t bits, uint32_t epoch, uint32_t* pairs, uint32_t* temp,
                         hipStream_t stream) {
    const uint32_t n = plan.n;
    const uint32_t passes = (bits + 7) / 8;
    if (passes > (uint32_t)kMaxPasses) return hipErrorInvalidValue;
    if (passes == 0 || n == 0) return hipSuccess;
    const dim3 grid(plan.num_tiles), block(kSortBlock);
    const bool odd = (passes & 1u) != 0;
    hipLaunchKernelGGL(k_hist, grid, block, 0, stream, pairs, n, bits, plan.counts, plan.digit_off, plan.ctl,
                       odd ? reinterpret_cast<uint2*>(temp) : nullptr);
    uint32_t* src = odd ? temp : pairs;
    uint32_t* dst = odd ? pairs : temp;
    for (uint32_t p = 0; p < passes; ++p) {
        hipLaunchKernelGGL(k_pass, grid, block, 0, stream, src, dst, n, p, bits, epoch + p, plan.digit_off, plan.status,
                           plan.ctl, plan.err);
        std::swap(src, dst);
    }
    return hipGetLastError();
}

}  // namespace sph

// --------------------------------------------------------------------------
// The reference's RadixSort seam (source/CUDA/radixsort.cuh:30-32) as C ABI
// entry points: sph_radix_sort allocates its scratch for the call,
// sph_radix_sort_noalloc uses a fixed device array instead.
namespace {

using sph::RadixSortPlan;

// Largest sort the fixed array serves: the reference's 1M-particle scenes.
constexpr uint32_t kNoAllocMaxPairs = SPH_SORT_NOALLOC_MAX;
constexpr size_t kNoAllocBytes = sph::scratch_bytes_for_tiles((kNoAllocMaxPairs + sph::kTile - 1) / sph::kTile);
constexpr int kMaxDevices = 64;

// The allocation-free sort's scratch: one copy per GPU, held until the
// process ends (about 0.6 MB).  Host code uses the per-device address from
// hipGetSymbolAddress (noalloc_ptr), never this name.
__device__ __align__(256) unsigned char scratch[kNoAllocBytes];
static_assert(kNoAllocBytes % 4 == 0, "cleared by words");

std::mutex noalloc_mu;
void* noalloc_ptr[kMaxDevices] = {};
uint32_t noalloc_epoch[kMaxDevices] = {};  // the next sort's; 0: the array has to be cleared first

int status_of(hipError_t e) {
    if (e == hipSuccess) return SPH_OK;
    if (e == hipErrorOutOfMemory) return SPH_ERR_OUT_OF_MEMORY;
    if (e == hipErrorNoDevice || e == hipErrorInvalidDevice) return SPH_ERR_NO_DEVICE;
    return SPH_ERR_DEVICE;
}

int check_sort_args(const uint32_t* pairs, const uint32_t* temp, uint32_t bits) {
    if (!pairs || !temp || bits > 32 || pairs == temp) return SPH_ERR_INVALID_ARGUMENT;
    return SPH_OK;
}

// Sort, wait for it, and report a look-back wait that hit its bound.
int sort_and_wait(RadixSortPlan& plan, uint32_t bits, uint32_t epoch, uint32_t* pairs, uint32_t* temp, hipStream_t s) {
    hipError_t e = sph::radix_sort_kv(plan, bits, epoch, pairs, temp, s);
    uint32_t err = 0;
    if (e == hipSuccess) e = hipMemcpyAsync(&err, plan.err, sizeof(err), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return status_of(e);
    return err ? SPH_ERR_ORDER : SPH_OK;
}

// The same in the device's fixed array (noalloc_mu held).  The array is zero
// when the library is loaded and every sort leaves its control words zero;
// after a failed one it is cleared.
int sort_in_fixed_array(uint32_t bits, uint32_t* pairs, uint32_t* temp, uint32_t n, hipStream_t s) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return SPH_ERR_NO_DEVICE;
    if (!noalloc_ptr[dev]) {
        void* ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) return e != hipSuccess ? status_of(e) : SPH_ERR_DEVICE;
        noalloc_ptr[dev] = ptr;
    }
    RadixSortPlan plan;
    sph::carve(plan, n, noalloc_ptr[dev]);
    // epochs run up to 2^32 - 1 and start again from a cleared array
    if (noalloc_epoch[dev] == 0 || noalloc_epoch[dev] > 0xFFFFFFFFu - 2 * sph::kMaxPasses) {
        const hipError_t e = sph::launch_fill_u32(static_cast<uint32_t*>(noalloc_ptr[dev]), 0u, kNoAllocBytes / 4, s);
        if (e != hipSuccess) return status_of(e);
        noalloc_epoch[dev] = 1;
    }
    const uint32_t epoch = noalloc_epoch[dev];
    noalloc_epoch[dev] += sph::kMaxPasses;
    const int st = sort_and_wait(plan, bits, epoch, pairs, temp, s);
    if (st != SPH_OK) noalloc_epoch[dev] = 0;
    return st;
}

}  // namespace

extern "C" {

int sph_radix_sort(uint32_t* pairs, uint32_t* temp, uint32_t n, uint32_t bits, void* stream) {
    int st = check_sort_args(pairs, temp, bits);
    if (st != SPH_OK) return st;
    if (n > SPH_SORT_MAX) return SPH_ERR_CAPACITY;
    if (n == 0 || bits == 0) return SPH_OK;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    // the fixed array while no other call holds it: an allocation and its
    // release cost more than the sort of some 100k pairs (about 40 us a call)
    if (n <= kNoAllocMaxPairs) {
        std::unique_lock<std::mutex> lock(noalloc_mu, std::try_to_lock);
        if (lock.owns_lock()) return sort_in_fixed_array(bits, pairs, temp, n, s);
    }
    void* buf = nullptr;
    const size_t bytes = sph::radix_scratch_bytes(n);
    hipError_t e = sph::device_malloc(&buf, bytes);
    if (e != hipSuccess) return status_of(e);
    RadixSortPlan plan;
    sph::carve(plan, n, buf);
    e = sph::launch_fill_u32(static_cast<uint32_t*>(buf), 0u, bytes / 4, s);
    st = e == hipSuccess ? sort_and_wait(plan, bits, 1u, pairs, temp, s) : status_of(e);
    (void)hipFree(buf);
    return st;
}

int sph_radix_sort_noalloc(uint32_t* pairs, uint32_t* temp, uint32_t n, uint32_t bits, void* stream) {
    int st = check_sort_args(pairs, temp, bits);
    if (st != SPH_OK) return st;
    if (n > kNoAllocMaxPairs) return SPH_ERR_CAPACITY;
    if (n == 0 || bits == 0) return SPH_OK;
    // one call per device at a time: the array is shared by every call on it
    std::lock_guard<std::mutex> lock(noalloc_mu);
    return sort_in_fixed_array(bits, pairs, temp, n, static_cast<hipStream_t>(stream));
}

}  // extern "C"
