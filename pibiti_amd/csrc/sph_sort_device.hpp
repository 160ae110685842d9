// sph_sort_device.hpp - the device side of the stable LSD radix sort
// (sph_sort.hip describes it): the tiles of its histogram and of its passes,
// and the whole sort by the blocks of one launch, which the step's place
// kernel runs when a step's order cannot be built from the last one.
#pragma once

#include "sph_internal.hpp"

namespace sph {
namespace sortdev {

constexpr int kSortBlock = 1024;
constexpr int kWave = 64;
constexpr int kWaves = kSortBlock / kWave;
constexpr int kItems = 4;
constexpr int kTile = kSortBlock * kItems;  // pairs per tile
constexpr int kRadix = 256;
constexpr int kMaxPasses = 4;
constexpr int kLook = kSortBlock / kRadix;  // threads per digit in the look-back
constexpr int kSpan = 16;                   // words a sum of the look-back covers
constexpr uint32_t kSpinLimit = 1u << 22;    // of a look-back, some tenths of a second
constexpr uint32_t kWaitLimit = 1u << 19;    // of wait_for, about half a second


// Inclusive scan of one value per thread over the block: a shuffle scan in
// each wave, then the totals of the waves before it.
template <int kThreads>
__device__ __forceinline__ uint32_t block_incl_scan(uint32_t v, uint32_t* s_wave) {
    const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const uint32_t u = __shfl_up(v, off);
        v += lane >= off ? u : 0u;
    }
    if (lane == kWave - 1) s_wave[w] = v;
    __syncthreads();
    uint32_t add = 0;
    for (int k = 0; k < w; ++k) add += s_wave[k];
    __syncthreads();
    return v + add;
}

// Hand-over between the blocks of one launch.  Before a block lets other blocks
// know that its part is done, every wave waits for its own stores and atomics,
// then the block meets (finish_block): a barrier alone does not wait for them,
// and a thread's fence covers its own wave only.  Atomics are then in memory;
// stores are in the XCC's L2, which one thread writes back (release_agent).
// The receiving block's one thread that waits acquires before its block meets.
__device__ __forceinline__ void finish_block() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
}
__device__ __forceinline__ void release_agent() { __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent"); }
__device__ __forceinline__ void acquire_agent() { __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent"); }

// Look-back words: (epoch << 32) | value, written once per sort and pass: a
// tile's digit counts, the sums over each kSpan tiles, over each kSpan of those
// and so on, one level behind the other.
constexpr uint32_t groups_of(uint32_t count) { return (count + kSpan - 1) / kSpan; }
constexpr uint64_t look_back_rows(uint32_t tiles) {
    uint64_t rows = tiles;
    for (uint32_t c = tiles; c > (uint32_t)kSpan; c = groups_of(c)) rows += groups_of(c);
    return rows;
}

__device__ __forceinline__ uint64_t ld_status(const uint64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_status(uint64_t* p, uint32_t epoch, uint32_t v) {
    __hip_atomic_store(p, ((uint64_t)epoch << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Sum of digit d's words of the rows row - k (k = 1 .. count, fewer than kSpan)
// that thread q of the digit's kLook takes (k = q + 1, q + 1 + kLook, ...),
// waiting for each to carry the epoch.
__device__ __forceinline__ uint32_t look_back(const uint64_t* __restrict__ words, uint32_t row, uint32_t count, int d,
                                              int q, uint32_t epoch, uint32_t* __restrict__ err) {
    constexpr int kBatch = kSpan / kLook;  // loads in flight
    static_assert(kSpan % kLook == 0, "one round of loads");
    uint64_t w[kBatch];
    for (uint32_t spins = 0;;) {
        bool waiting = false;
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const uint32_t k = (uint32_t)(q + 1 + u * kLook);
            w[u] = (uint64_t)epoch << 32;
            if (k <= count) w[u] = ld_status(words + (size_t)(row - k) * kRadix + d);
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) waiting = waiting || (uint32_t)(w[u] >> 32) != epoch;
        if (!waiting) break;
        if (++spins > kSpinLimit) {
            atomicOr(err, 1u);
            break;
        }
        __builtin_amdgcn_s_sleep(1);
    }
    uint32_t sum = 0;
#pragma unroll
    for (int u = 0; u < kBatch; ++u) sum += (uint32_t)w[u];
    return sum;
}

// The sort's control words (RadixSortPlan::ctl), all zero between sorts but the
// epoch.  Each word that many blocks update or wait for has a cache line of
// its own: in one line their polls and updates queue up behind each other.
constexpr int kLine = 32;  // words
constexpr int kStages = 1 + kMaxPasses;
constexpr int kXccs = 16;  // values of the XCC id register
enum Ctl : int {
    kCtlEpoch = 0,            // sorts finished by sort_slots
    kCtlErr = 1,              // a wait hit its bound (the plan may name another word)
    kCtlHistDone = 1 * kLine, // histogram tiles finished
    kCtlTicket = 2 * kLine,   // sort_slots: (stage, tile) tickets
    kCtlRetired = 3 * kLine,  // sort_slots: blocks that found no ticket
    kCtlReady = 4 * kLine,    // sort_slots: the digit offsets are written
    kCtlPass = 5 * kLine,     // [kMaxPasses] k_pass: tile tickets
    kCtlDone = kCtlPass + kMaxPasses * kLine,     // [kStages] sort_slots: tiles whose output is in memory
    kCtlXcc = kCtlDone + kStages * kLine,         // [kStages][kXccs] sort_slots: XccWord
    kCtlNum = kCtlXcc + kStages * kXccs * kLine
};
// A stage's tiles on one XCC: taken, finished, and of these written back.
enum XccWord : int { kXccTaken = 0, kXccFinished = 1, kXccWritten = 2 };

struct SortShared {
    uint32_t wcount[kWaves][kRadix];
    uint32_t dig_off[kRadix];
    uint32_t gbase[kRadix];
    uint32_t look[kLook][kRadix];
    uint32_t keys[kTile];
    uint32_t vals[kTile];
    uint32_t s_wave[kSortBlock / kWave];
    uint32_t word;
};

__device__ __forceinline__ uint32_t digit_bits(uint32_t bits, uint32_t p) {
    return bits - 8 * p < 8 ? bits - 8 * p : 8;
}

// Digit counts of one tile's keys for every pass, added to counts
// [kMaxPasses][kRadix]; the last of `tiles` tiles to finish scans the counts
// into the digit offsets and clears them.  Within a wave a run of consecutive
// lanes with the same digit is counted by one LDS atomic of its first lane:
// in a step the keys arrive nearly sorted, so runs are long.
// Returns whether this block wrote the offsets.
// kStride: 1 for a key array, 2 for (key, value) pairs.
template <int kStride>
__device__ __forceinline__ bool hist_tile(SortShared& S, uint32_t tile, uint32_t tiles,
                                          const uint32_t* __restrict__ keys, uint32_t n, uint32_t bits,
                                          uint32_t* __restrict__ counts, uint32_t* __restrict__ offsets,
                                          uint32_t* __restrict__ ctl, uint2* __restrict__ copy = nullptr) {
    static_assert(kWaves >= kMaxPasses, "the histogram shares wcount");
    auto& hist = S.wcount;
    const int t = threadIdx.x;
    const int lane = t % kWave;
    const uint32_t passes = (bits + 7) / 8;
    if (t < kMaxPasses * kRadix) hist[t / kRadix][t % kRadix] = 0;
    __syncthreads();
    const uint64_t after_me = lane == kWave - 1 ? 0ull : (~0ull << (lane + 1));
    const uint64_t base = (uint64_t)tile * kTile;
    uint32_t k[kItems];
#pragma unroll
    for (int it = 0; it < kItems; ++it) {
        const uint64_t e = base + (uint64_t)it * kSortBlock + t;
        if constexpr (kStride == 2) {
            if (copy) {
                const uint2 pair = reinterpret_cast<const uint2*>(keys)[e < n ? e : n - 1];
                k[it] = pair.x;
                if (e < n) copy[e] = pair;
                continue;
            }
        }
        k[it] = keys[(e < n ? e : n - 1) * kStride];
    }
#pragma unroll
    for (int it = 0; it < kItems; ++it) {
        // the valid lanes of a wave are a prefix of it (indices grow with the lane)
        const bool valid = base + (uint64_t)it * kSortBlock + t < n;
        const uint32_t nvalid = (uint32_t)__popcll(__ballot(valid));
        for (uint32_t p = 0; p < passes; ++p) {
            const uint32_t d = (k[it] >> (8 * p)) & ((1u << digit_bits(bits, p)) - 1u);
            const uint32_t dprev = __shfl_up(d, 1);
            const bool head = valid && (lane == 0 || dprev != d);
            const uint64_t later = __ballot(head) & after_me;
            const uint32_t end = later ? (uint32_t)(__ffsll((unsigned long long)later) - 1) : nvalid;
            if (head) atomicAdd(&hist[p][d], end - (uint32_t)lane);
        }
    }
    __syncthreads();
    static_assert(kSortBlock == kMaxPasses * kRadix, "one thread per pass and digit");
    const uint32_t mine = hist[t / kRadix][t % kRadix];
    if (mine) atomicAdd(&counts[t], mine);
    // the last tile scans: every count is in before its tile is counted done
    finish_block();
    if (t == 0) S.word = atomicAdd(&ctl[kCtlHistDone], 1u);
    __syncthreads();
    if (S.word != tiles - 1) return false;
    const uint32_t c = __hip_atomic_exchange(&counts[t], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // an inclusive scan over all passes' digits; a pass's offsets are relative
    // to the passes before it, whose counts sum to n each
    const uint32_t incl = block_incl_scan<kSortBlock>(c, S.s_wave);
    __hip_atomic_store(&offsets[t], incl - c - (uint32_t)(t / kRadix) * n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (t == 0) ctl[kCtlHistDone] = 0u;
    return true;
}

// One tile of one pass.  kPairs: input and output are arrays of (key, value)
// pairs (keys_in / keys_out; the others unused) instead of a key array and a
// value array.
template <bool kPairs>
__device__ __forceinline__ void pass_tile(SortShared& S, uint32_t tile, uint32_t tiles, uint32_t epoch,
                                          const uint32_t* __restrict__ keys_in, const uint32_t* __restrict__ vals_in,
                                          uint32_t* __restrict__ keys_out, uint32_t* __restrict__ vals_out,
                                          uint32_t n, uint32_t shift, uint32_t pass_bits,
                                          const uint32_t* __restrict__ digit_off, uint64_t* status,
                                          uint32_t* __restrict__ err) {
    const int t = threadIdx.x;
    const int wave = t / kWave;
    const int lane = t % kWave;
    const uint32_t mask = (1u << pass_bits) - 1u;
    const uint64_t tile_base = (uint64_t)tile * kTile;
    const uint64_t wbase = tile_base + (uint64_t)wave * (kWave * kItems);
    const uint64_t lt_mask = (lane == 0) ? 0ull : ((~0ull) >> (64 - lane));
    uint32_t k[kItems], v[kItems], rank[kItems];
#pragma unroll
    for (int it = 0; it < kItems; ++it) {
        const uint64_t e = wbase + (uint64_t)it * kWave + lane;
        k[it] = v[it] = 0u;
        if (e < n) {
            if constexpr (kPairs) {
                const uint2 kv = reinterpret_cast<const uint2*>(keys_in)[e];
                k[it] = kv.x;
                v[it] = kv.y;
            } else {
                k[it] = keys_in[e];
                v[it] = vals_in[e];
            }
        }
    }
#pragma unroll
    for (int w = 0; w < kWaves * kRadix / kSortBlock; ++w) (&S.wcount[0][0])[w * kSortBlock + t] = 0;
    __syncthreads();
#pragma unroll
    for (int it = 0; it < kItems; ++it) {
        const bool valid = wbase + (uint64_t)it * kWave + lane < n;
        const uint32_t d = (k[it] >> shift) & mask;
        uint64_t peers = __ballot(valid);
        for (uint32_t bit = 0; bit < pass_bits; ++bit) {
            const bool set = (d >> bit) & 1u;
            const uint64_t bal = __ballot(set);
            peers &= set ? bal : ~bal;
        }
        const uint32_t r = (uint32_t)__popcll(peers & lt_mask);
        uint32_t pre = 0;
        if (valid) pre = S.wcount[wave][d];
        __builtin_amdgcn_wave_barrier();
        if (valid && r == 0) S.wcount[wave][d] = pre + (uint32_t)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
        rank[it] = valid ? pre + r : 0xFFFFFFFFu;
    }
    __syncthreads();

    // Per digit (thread t < kRadix): exclusive prefix over waves, tile total,
    // which is published at once.
    const uint32_t cnt = [&]() {
        uint32_t c = 0;
        if (t < kRadix) {
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                const uint32_t x = S.wcount[w][t];
                S.wcount[w][t] = c;
                c += x;
            }
            st_status(status + (size_t)tile * kRadix + t, epoch, c);
        }
        return c;
    }();
    const uint32_t incl = block_incl_scan<kSortBlock>(cnt, S.s_wave);
    if (t < kRadix) S.dig_off[t] = incl - cnt;

    // Look back, kLook threads per digit: the counts of the tiles before this
    // one in its span, the sums of the spans before that one in its span, and
    // so on.  The last tile of a span makes and publishes the span's sum.
    const int d = t % kRadix, q = t / kRadix;
    uint32_t prefix = 0, total = cnt;
    bool last = true;
    for (uint32_t row = tile, rows = tiles;;) {
        const uint32_t before = row % kSpan;  // (the same for the whole block)
        if (before) {
            S.look[q][d] = look_back(status, row, before, d, q, epoch, err);
            __syncthreads();
            if (t < kRadix) {
                uint32_t sum = 0;
#pragma unroll
                for (int u = 0; u < kLook; ++u) sum += S.look[u][t];
                prefix += sum;
                total += sum;
            }
        }
        status += (size_t)rows * kRadix;
        last = last && before == kSpan - 1u;
        if (rows <= (uint32_t)kSpan) break;
        if (last && t < kRadix) st_status(status + (size_t)(row / kSpan) * kRadix + t, epoch, total);
        row /= kSpan;
        rows = groups_of(rows);
        if (row == 0) break;
        __syncthreads();
    }
    if (t < kRadix)
        S.gbase[t] = __hip_atomic_load(&digit_off[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + prefix;
    __syncthreads();

#pragma unroll
    for (int it = 0; it < kItems; ++it) {
        if (rank[it] == 0xFFFFFFFFu) continue;
        const uint32_t dd = (k[it] >> shift) & mask;
        const uint32_t lp = S.dig_off[dd] + S.wcount[wave][dd] + rank[it];
        S.keys[lp] = k[it];
        S.vals[lp] = v[it];
    }
    __syncthreads();

    const uint64_t rem = (uint64_t)n - tile_base;
    const uint32_t count = rem < (uint64_t)kTile ? (uint32_t)rem : (uint32_t)kTile;
#pragma unroll
    for (int it = 0; it < kItems; ++it) {
        const uint32_t i = (uint32_t)(it * kSortBlock + t);
        if (i >= count) continue;
        const uint32_t key = S.keys[i];
        const uint32_t dd = (key >> shift) & mask;
        const uint32_t g = S.gbase[dd] + (i - S.dig_off[dd]);
        if (g >= n) continue;  // only after a wait that hit its bound
        if constexpr (kPairs) {
            reinterpret_cast<uint2*>(keys_out)[g] = make_uint2(key, S.vals[i]);
        } else {
            keys_out[g] = key;
            vals_out[g] = S.vals[i];
        }
    }
}

// Thread 0 waits until *word == want; the block then sees what the blocks
// that raised it wrote before.
__device__ __forceinline__ void wait_for(const uint32_t* word, uint32_t want, uint32_t* err) {
    if (threadIdx.x == 0) {
        uint32_t spins = 0;
        while (__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != want) {
            if (++spins > kWaitLimit) {
                atomicOr(err, 1u);
                break;
            }
            __builtin_amdgcn_s_sleep(32);
        }
        acquire_agent();
    }
    __syncthreads();
}

// A tile of a stage is finished (finish_block is behind it): its output is
// counted done once it is in memory.  A write-back covers the whole L2, and
// each one walks it: 32 tiles of an XCC that end together, each with its own,
// take several times their own work.  So the one that leaves no taken tile
// behind on its XCC writes back for all that finished there before it.
// (1,048,576 particles, the place kernel of a step with the full sort: a
// write-back and an acquire in every wave 880 us, in one wave a tile 340, with
// the control words in lines of their own 207, one an XCC 117; a launch for
// each stage, which every step would pay for, 148.)
__device__ __forceinline__ void count_done(uint32_t* ctl, uint32_t stage, uint32_t xcc) {
    uint32_t* const x = ctl + kCtlXcc + (stage * kXccs + xcc) * kLine;
    uint32_t finished = atomicAdd(&x[kXccFinished], 1u) + 1u;
    // counted before the taken ones are read (the last to finish has to see
    // every one; its own was counted before its work)
    asm volatile("" : "+v"(finished)::"memory");
    if (finished != __hip_atomic_load(&x[kXccTaken], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
    const uint32_t written = atomicMax(&x[kXccWritten], finished);
    if (written >= finished) return;
    release_agent();
    atomicAdd(&ctl[kCtlDone + stage * kLine], finished - written);
}

// The XCC (and so the L2) this wave runs on.
__device__ __forceinline__ uint32_t xcc_id() {
    constexpr int kHwRegXccId = 20;
    return __builtin_amdgcn_s_getreg(kHwRegXccId | (0 << 6) | ((4 - 1) << 11)) & (kXccs - 1);
}

// The whole sort of the slots by (the low `bits` bits of nkey, original
// index), by the blocks of one launch, each of kSortBlock threads that all call
// this.  Its input is made here, (key, slot) in original-index order into
// (keys0, vals0), so that a step that needs no sort does not write it; the
// passes ping-pong with (keys1, vals1), where keys1 may be nkey.  Tickets: the
// tiles of the input and its digit counts, then those of pass 0, 1, ...; a
// block takes the next one until none is left and waits for the last pass.
// Tickets are held by running blocks only, so every wait ends whatever else
// runs on the GPU.  Returns with the sorted pairs visible to the block.
struct SlotSort {
    uint32_t* keys0;
    uint32_t* vals0;
    uint32_t* keys1;
    uint32_t* vals1;
    uint32_t n, bits, tiles;
    uint32_t* counts;
    uint32_t* offsets;
    uint64_t* status;
    uint32_t* ctl;
    uint32_t* err;
};

__device__ __forceinline__ void sort_slots(SortShared& S, const SlotSort& a, const uint32_t* nkey, const uint32_t* pid) {
    const int t = threadIdx.x;
    const uint32_t n = a.n, tiles = a.tiles, passes = (a.bits + 7) / 8;
    uint32_t* const ctl = a.ctl;
    // read before this block's first ticket; the last block to retire, which
    // raises it, does so after every block's last wait
    const uint32_t first_epoch = ctl[kCtlEpoch] * kMaxPasses + 1u;
    const uint32_t xcc = xcc_id();
    for (;;) {
        if (t == 0) {
            const uint32_t w = atomicAdd(&ctl[kCtlTicket], 1u);
            if (w < tiles * (passes + 1)) atomicAdd(&ctl[kCtlXcc + (w / tiles * kXccs + xcc) * kLine + kXccTaken], 1u);
            S.word = w;
        }
        __syncthreads();
        const uint32_t w = S.word;
        __syncthreads();
        if (w >= tiles * (passes + 1)) break;
        const uint32_t stage = w / tiles, tile = w % tiles;
        if (stage == 0) {
#pragma unroll
            for (int it = 0; it < kItems; ++it) {
                const uint64_t e = (uint64_t)tile * kTile + (uint64_t)it * kSortBlock + t;
                if (e >= n) continue;
                const uint32_t id = pid[e];
                if (id >= n) continue;
                a.keys0[id] = nkey[e];
                a.vals0[id] = (uint32_t)e;
            }
            if (hist_tile<1>(S, tile, tiles, nkey, n, a.bits, a.counts, a.offsets, ctl)) {
                finish_block();
                if (t == 0) atomicExch(&ctl[kCtlReady], 1u);
            }
        } else {
            const uint32_t p = stage - 1;
            wait_for(&ctl[kCtlDone + p * kLine], tiles, a.err);
            if (p == 0) wait_for(&ctl[kCtlReady], 1u, a.err);
            const bool odd = (p & 1u) != 0;
            pass_tile<false>(S, tile, tiles, first_epoch + p, odd ? a.keys1 : a.keys0, odd ? a.vals1 : a.vals0,
                             odd ? a.keys0 : a.keys1, odd ? a.vals0 : a.vals1, n, 8 * p, digit_bits(a.bits, p),
                             a.offsets + p * kRadix, a.status, a.err);
            finish_block();
        }
        if (t == 0) count_done(ctl, stage, xcc);
        __syncthreads();
    }
    wait_for(&ctl[kCtlDone + passes * kLine], tiles, a.err);
    if (t == 0) S.word = atomicAdd(&ctl[kCtlRetired], 1u);
    __syncthreads();
    if (S.word != gridDim.x - 1) return;
    // every other block is past its last use of the control words
    for (int c = kLine + t; c < kCtlNum; c += kSortBlock) ctl[c] = 0u;
    if (t == 0) ctl[kCtlEpoch] += 1u;
}

}  // namespace sortdev
}  // namespace sph
