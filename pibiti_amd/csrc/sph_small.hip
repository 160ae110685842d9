// sph_small.hip - density and force with nine lanes per particle, one for each
// row of neighbour cells.
//
// The one-lane gathers (k_density_entries, k_density_fast, k_force_entries)
// walk a particle's 27 cells in one lane: about 80 dependent candidate loads,
// and an array of up to some 100k particles has too few waves to hide them,
// so such a launch takes the latency of one walk whatever its size.  Here the
// nine rows (dz, dy) of a particle go to nine lanes, seven particles to a
// wave: a lane walks the three cells of its row, leaves the
// row's partial sums in LDS, and one thread per particle adds them in the
// walk's order (the force: below).  The sums are the one-lane kernels' bit for
// bit: the reference order adds per-cell partial sums in cell order (an empty
// or culled cell's +0 leaves the total as it is), FAST adds per-row partial
// sums in row order, and a compensated sum takes the terms themselves in walk
// order.
//
// What bounds it: at 2,197 to 15,625 particles the latency of a launch and of
// a dozen dependent loads, at 65,536 the vector L1 (the lanes of a wave read
// nine rows where the one-lane kernels' read one).  Density and force, us, one
// lane -> nine, in the first steps of a dam break and after 2,000 steps (the
// longest lists then hold over 100 pairs), in blocks of four waves:
//     15,625 particles   34 + 18 -> 10.3 + 8.5     48 + 47 -> 12.7 + 17
//     65,231             35 + 19 -> 24 + 16        49 + 35 -> 29 + 23
//    101,376             32 + 18 -> 41 + 24        45 + 33 -> 42 + 29
// so arrays of up to kRowGatherMax = 65,536 take the nine lanes.
//
// Between the two kernels a row's force pairs travel as in the one-lane
// kernels: entries of (first slot << kPairSlotShift) | kPairNewCell | 4-bit
// mask, here a list per lane (group-major: the lanes' first four entries lie
// side by side, then their next four) with its pair count in a byte of its own.
#include "sph_device.hpp"

namespace sph {
namespace {

using namespace dev;

constexpr int kRows = 9;
constexpr uint32_t kRowEntries = 3u * ((kMaskCap + 3u) / 4u);  // 12: three cells of at most kMaskCap slots
static_assert(kRows * kRowEntries <= 4u * list_groups(kMaskCap), "rows fit the entry lists");
static_assert(kRowEntries % 4u == 0u, "whole uint4 groups per row");
static_assert(kRows <= 4 * kMaskWords, "the lanes' pair counts fit the mask words");

constexpr int kWaveParticles = 64 / kRows;  // 7: one lane of 64 idle

// A block of kWaves waves.
template <int kWaves>
struct RowLane {
    int lp;      // particle within the block
    int row;     // 3 (dz + 1) + (dy + 1)
    uint32_t i;  // slot
    bool on;
    __device__ __forceinline__ explicit RowLane(uint32_t n) {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        lp = wave * kWaveParticles + lane / kRows;
        row = lane % kRows;
        i = xcd_tile(blockIdx.x, gridDim.x) * (kWaves * kWaveParticles) + (uint32_t)lp;
        on = lane < kRows * kWaveParticles && i < n;
    }
};

template <bool kBatch, int kPrec, int kWaves>
__global__ __launch_bounds__(64 * kWaves) void k_density_rows(sph_params one, const sph_params* __restrict__ tab,
                                                         const uint32_t* __restrict__ sid, uint32_t n,
                                                         const float4* __restrict__ pos,
                                                         const float* __restrict__ xyz,
                                                         const float4* __restrict__ vel,
                                                         const uint32_t* __restrict__ cell_start,
                                                         const uint32_t* __restrict__ cell_end,
                                                         float2* __restrict__ rhop, float4* __restrict__ rec,
                                                         uint32_t* __restrict__ entries,
                                                         uint8_t* __restrict__ lane_pairs,
                                                         uint32_t* __restrict__ nnb,
                                                         const uint32_t* __restrict__ counters) {
    constexpr bool kFast = kPrec == SPH_PREC_FAST;
    constexpr bool kKahan = kPrec == SPH_PREC_KAHAN;
    static_assert(!kKahan || kWaves == 1, "s_wgt is one wave's");
    constexpr int kSums = kFast || kKahan ? kRows : 3 * kRows;  // partial sums of a particle
    constexpr int kParticles = kWaves * kWaveParticles;
    // kKahan: each lane's weights in walk order (and one place past them,
    // which a miss writes), and their number in s_sum's place
    __shared__ float s_wgt[kKahan ? 4 * kRowEntries + 1 : 1][64];
    __shared__ float s_sum[kSums][kParticles];
    __shared__ uint32_t s_pairs[kRows][kParticles];
    const RowLane<kWaves> me(n);
    if (me.on) {
        const uint32_t i = me.i;
        uint32_t scene;
        const sph_params& p = scene_params<kBatch>(one, tab, sid, i, scene);
        const float4 xi = pos[i];
        CellWalk w;
        w.init(p, xi.x, xi.y, xi.z, walk_culled(counters));
        const float h2 = p.h2, r2f = p.force_r2_max, inv_h2 = 1.0f / h2;
        const CellWalk::Row row = w.row(me.row % 3 - 1, me.row / 3 - 1);
        // the row's three ranges: all loads go out together
        uint32_t s[3], e[3];
#pragma unroll
        for (int c = 0; c < 3; ++c)
            if (!w.open_in(row, c - 1, cell_start, cell_end, s[c], e[c])) s[c] = e[c] = 0u;
        // entry q of the lane: word q % 4 of the uint4 (q / 4) lanes + lane
        const size_t lanes = (size_t)n * kRows;
        uint32_t* out = entries + 4 * ((size_t)i * kRows + me.row);
        uint32_t count = 0, pairs = 0;
        float run = 0.0f;
        uint32_t weights = 0;
        uint32_t fresh = kPairNewCell;  // until the open partial sum (a cell's, in FAST a row's) has an entry
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            if (!kFast) fresh = kPairNewCell;
            float cell = 0.0f;
            for (uint32_t j0 = s[c]; j0 < e[c]; j0 += 4) {
                float cx[4], cy[4], cz[4];
                packed_group(xyz, j0 * kSlotBytes, cx, cy, cz);
                // slots past the cell's end and the particle itself take
                // r2 = +inf, which fails both predicates
                const uint32_t left = e[c] - j0, self = i - j0;
                uint32_t bits = 0;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const float rx = xi.x - cx[k], ry = xi.y - cy[k], rz = xi.z - cz[k];
                    float r2 = rx * rx + ry * ry + rz * rz;
                    r2 = left > (uint32_t)k && self != (uint32_t)k ? r2 : __builtin_huge_valf();
                    if constexpr (kFast) {
                        const float u = fminf(fmaxf(__builtin_fmaf(r2, -inv_h2, 1.0f), 0.0f), 1.0f);
                        run = __builtin_fmaf(u * u, u, run);
                    } else {
                        const float c3 = h2 - r2;
                        const float wgt = (c3 * c3) * c3;
                        if constexpr (kKahan) {
                            s_wgt[weights][threadIdx.x] = wgt;
                            weights += r2 < h2 ? 1u : 0u;
                        } else {
                            cell = cell + (r2 < h2 ? wgt : 0.0f);
                        }
                    }
                    bits |= force_pair(r2, r2f) ? (1u << k) : 0u;
                }
                if (bits) {
                    out[count & 3u] = (j0 << kPairSlotShift) | fresh | bits;
                    ++count;
                    if ((count & 3u) == 0u) out += 4 * lanes;
                    pairs += (uint32_t)__popc(bits);
                    fresh = 0u;
                }
            }
            if constexpr (!kFast && !kKahan) s_sum[3 * me.row + c][me.lp] = cell;
        }
        if constexpr (kFast) s_sum[me.row][me.lp] = run;
        if constexpr (kKahan) s_sum[me.row][me.lp] = __uint_as_float(weights);
        s_pairs[me.row][me.lp] = pairs;
        lane_pairs[(size_t)i * kRows + me.row] = (uint8_t)pairs;
    }
    __syncthreads();
    // one thread per particle adds the partial sums in walk order
    const int t = threadIdx.x;
    const uint32_t i = xcd_tile(blockIdx.x, gridDim.x) * kParticles + (uint32_t)t;
    if (t >= kParticles || i >= n) return;
    uint32_t scene;
    const sph_params& p = scene_params<kBatch>(one, tab, sid, i, scene);
    const float4 xi = pos[i], vi = vel[i];
    float sum = 0.0f;
    if constexpr (kKahan) {
        KahanF ks{0.0f, 0.0f};
        for (int q = 0; q < kRows; ++q) {
            const uint32_t m = __float_as_uint(s_sum[q][t]);
            for (uint32_t k = 0; k < m; ++k) ks.add(s_wgt[k][t * kRows + q]);
        }
        sum = ks.s;
    } else {
#pragma unroll
        for (int k = 0; k < kSums; ++k) sum = sum + s_sum[k][t];
    }
    uint32_t pairs = 0;
#pragma unroll
    for (int k = 0; k < kRows; ++k) pairs += s_pairs[k][t];
    float rho;
    if constexpr (kFast) {
        const float h2 = p.h2;
        rho = (sum * (((p.poly6_kern * h2) * h2) * h2)) * p.particle_mass;
    } else {
        rho = (sum * p.poly6_kern) * p.particle_mass;
    }
    const float pr = eos(p, rho);
    rhop[i] = make_float2(rho, pr);
    rec[2 * (size_t)i] = make_float4(xi.x, xi.y, xi.z, rho);
    rec[2 * (size_t)i + 1] = make_float4(vi.x, vi.y, vi.z, pr);
    nnb[i] = pairs << 16;
}

// What the lanes of a wave wrote to LDS before is what they read after (LDS
// operations of one wave complete in order; this keeps the compiler to it).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The force.  A row's pairs are few in a corner and many in the middle, so
// the nine lanes first spread their entries over one list per particle in
// LDS, in walk order, then take its pairs in turn, four at a time with their
// eight record loads in flight, and leave the terms in LDS; three lanes, one
// per axis, add them in walk order.  A particle's pairs go through the list
// kChunk at a time.  A block is one wave (15,625 particles 8.0 -> 7.7 us
// against blocks of four; 65,231 equal).
constexpr uint32_t kChunk = 64;
constexpr uint32_t kPad = kChunk + 1;  // the lists start in different banks
constexpr int kPairsAtOnce = 4;
constexpr uint32_t kOpens = 1u << 31;  // in a list word: the pair opens a partial sum

template <bool kBatch, int kPrec>
__global__ __launch_bounds__(64) void k_force_rows(sph_params one, const sph_params* __restrict__ tab,
                                                       const uint32_t* __restrict__ sid, uint32_t n,
                                                       const float4* __restrict__ vel,
                                                       const float4* __restrict__ rec,
                                                       const uint32_t* __restrict__ entries,
                                                       const uint8_t* __restrict__ lane_pairs,
                                                       float4* __restrict__ vel_out, float4* __restrict__ dvel,
                                                       const float* __restrict__ dt_dev) {
    constexpr bool kFast = kPrec == SPH_PREC_FAST;
    constexpr bool kKahan = kPrec == SPH_PREC_KAHAN;
    __shared__ uint32_t s_list[kWaveParticles][kPad];
    __shared__ float s_term[3][kWaveParticles][kPad];
    const RowLane<1> me(n);
    // every lane stays to the end: the loops below are the whole wave's
    const uint32_t i = me.on ? me.i : 0u;
    const int row = me.row, lp = me.on ? me.lp : 0;
    uint32_t scene;
    const sph_params& p = scene_params<kBatch>(one, tab, sid, i, scene);
    const float4 xi = rec[2 * (size_t)i];      // (x, y, z, rho)
    const float4 vi = rec[2 * (size_t)i + 1];  // (vx, vy, vz, p)
    const PairScale c{p.h, p.spiky_kern, p.min_dist, p.min_dens};
    const float vterm = p.lap_kern * p.viscosity;
    const size_t lanes = (size_t)n * kRows;
    const uint4* const list = reinterpret_cast<const uint4*>(entries) + ((size_t)i * kRows + row);
    const uint32_t count = me.on ? lane_pairs[(size_t)i * kRows + row] : 0u;
    // the pairs of the particle, and of its rows before this one
    uint32_t total = 0, off = 0;
    {
        const int first = (int)(threadIdx.x & 63u) - row;
#pragma unroll
        for (int q = 0; q < kRows; ++q) {
            const uint32_t x = (uint32_t)__shfl((int)count, first + q);
            total += x;
            off += q < row ? x : 0u;
        }
        if (!me.on) total = 0;
    }
    uint4 buf = list[0];
    uint32_t bits = 0, jb = 0, next = 0, done = 0;
    float a = 0.0f, f = 0.0f;  // lanes 0 .. 2: the axis's total and open partial sum
    KahanF ks{0.0f, 0.0f};     // kKahan: its compensated sum
    for (uint32_t c0 = 0; __any(c0 < total); c0 += kChunk) {
        while (done < count && off + done < c0 + kChunk) {
            uint32_t opens = 0;
            if (bits == 0u) {
                if ((next & 3u) == 0u && next) buf = list[(next >> 2) * lanes];
                const uint32_t e = buf.x;
                buf.x = buf.y, buf.y = buf.z, buf.z = buf.w;
                opens = (kFast ? next == 0u : (e & kPairNewCell) != 0u) ? kOpens : 0u;
                ++next;
                bits = e & 15u;
                jb = e >> kPairSlotShift;
            }
            s_list[lp][off + done - c0] = (jb + (uint32_t)__builtin_ctz(bits)) | opens;
            bits &= bits - 1u;
            ++done;
        }
        wave_sync();
        const uint32_t m = c0 < total ? min(kChunk, total - c0) : 0u;
        for (uint32_t k0 = (uint32_t)row; k0 < m; k0 += kPairsAtOnce * kRows) {
            uint32_t j[kPairsAtOnce];
            float4 xq[kPairsAtOnce], vq[kPairsAtOnce];
#pragma unroll
            for (int u = 0; u < kPairsAtOnce; ++u) {
                const uint32_t k = k0 + (uint32_t)(u * kRows);
                j[u] = s_list[lp][k < m ? k : k0] & ~kOpens;  // past the last pair: a repeat, not kept
            }
#pragma unroll
            for (int u = 0; u < kPairsAtOnce; ++u) {
                xq[u] = rec[2 * (size_t)j[u]];
                vq[u] = rec[2 * (size_t)j[u] + 1];
            }
            PairRange range(c);
            auto term = [&](int u, const float4& xj, const float4& vj, auto ieee) {
                const float rx = xi.x - xj.x, ry = xi.y - xj.y, rz = xi.z - xj.z;
                const float r2 = rx * rx + ry * ry + rz * rz;
                float pterm, cd;
                if constexpr (decltype(ieee)::value)
                    pair_scale_ieee(c, r2, vi.w + vj.w, xi.w * xj.w, pterm, cd);
                else
                    pair_scale(c, r2, vi.w + vj.w, xi.w * xj.w, range, pterm, cd);
                const uint32_t k = k0 + (uint32_t)(u * kRows);
                if (k < m) {
                    s_term[0][lp][k] = (pterm * rx + vterm * (vj.x - vi.x)) * cd;
                    s_term[1][lp][k] = (pterm * ry + vterm * (vj.y - vi.y)) * cd;
                    s_term[2][lp][k] = (pterm * rz + vterm * (vj.z - vi.z)) * cd;
                }
            };
#pragma unroll
            for (int u = 0; u < kPairsAtOnce; ++u) term(u, xq[u], vq[u], std::false_type{});
            if (__builtin_expect(!range.ok(), 0)) {
#pragma unroll 1
                for (int u = 0; u < kPairsAtOnce; ++u) {
                    const uint32_t k = k0 + (uint32_t)(u * kRows);
                    if (k >= m) break;
                    const uint32_t jk = s_list[lp][k] & ~kOpens;
                    term(u, rec[2 * (size_t)jk], rec[2 * (size_t)jk + 1], std::true_type{});
                }
            }
        }
        wave_sync();
        if (row < 3) {
#pragma unroll 4
            for (uint32_t k = 0; k < m; ++k) {
                if constexpr (kKahan) {
                    ks.add(s_term[row][lp][k]);
                    continue;
                }
                // (no branch: adding +0 changes neither sum, which are never -0)
                const bool opens = (s_list[lp][k] & kOpens) != 0u;
                a = a + (opens ? f : 0.0f);
                f = (opens ? 0.0f : f) + s_term[row][lp][k];
            }
        }
        wave_sync();
    }
    if (!me.on || row > 3) return;
    // lanes 0 .. 2 write the axes, lane 3 the fourth component
    const float v = reinterpret_cast<const float*>(vel + i)[row];
    a = row < 3 ? (kKahan ? ks.s : a + f) * (p.particle_mass * dt_dev[scene]) : 0.0f;
    // with other terms the pair increment only: k_extra_terms adds them and
    // finishes the update
    reinterpret_cast<float*>(vel_out + i)[row] = p.physics ? a : v + a;
    if (dvel && !p.physics) reinterpret_cast<float*>(dvel + i)[row] = a;
}

inline uint32_t row_blocks(uint32_t n, uint32_t waves) {
    const uint32_t per = waves * kWaveParticles;
    return n == 0 ? 1u : (n + per - 1) / per;
}

// Up to here the density's blocks are one wave, which waits for no other
// (2,197 particles 8.2 -> 7.8 us, 15,625 10.0 -> 9.3, 32,768 equal); larger
// arrays are bound by the L1, where one wave's sums for 28 particles are
// cheaper than four waves' for seven each (65,231: 24.0, one wave 24.7).
constexpr uint32_t kOneWaveMax = 32768;

template <bool kBatch, int kPrec>
void density_rows(const LaunchCfg& c, const StepBuffers& b, hipStream_t s) {
    const auto launch = [&](auto waves) {
        constexpr int kWaves = decltype(waves)::value;
        hipLaunchKernelGGL((k_density_rows<kBatch, kPrec, kWaves>), dim3(row_blocks(c.n, kWaves)), dim3(64 * kWaves), 0,
                           s, c.one, c.tab, b.sid_cur, c.n, b.pos_cur, b.xyz, b.vel_cur, b.cell_start, b.cell_end,
                           b.rhop, b.rec, reinterpret_cast<uint32_t*>(b.pairs), reinterpret_cast<uint8_t*>(b.masks),
                           b.pair_cnt, b.counters);
    };
    if constexpr (kPrec == SPH_PREC_KAHAN) {
        launch(std::integral_constant<int, 1>{});
    } else {
        if (c.n <= kOneWaveMax)
            launch(std::integral_constant<int, 1>{});
        else
            launch(std::integral_constant<int, 4>{});
    }
}

template <bool kBatch, int kPrec>
void force_rows(const LaunchCfg& c, const StepBuffers& b, float4* vel_out, float4* dvel, hipStream_t s) {
    hipLaunchKernelGGL((k_force_rows<kBatch, kPrec>), dim3(row_blocks(c.n, 1)), dim3(64), 0, s, c.one, c.tab,
                       b.sid_cur, c.n, b.vel_cur, b.rec, reinterpret_cast<const uint32_t*>(b.pairs),
                       reinterpret_cast<const uint8_t*>(b.masks), vel_out, dvel, b.dt_dev);
}

// Compensated sums take the terms one after another: the density's lanes
// leave their weights in LDS, 12.5 KB a wave, and one lane per particle adds
// them, so the line lies lower (density + force, us, one lane -> nine: 2,197
// particles 33 + 13 -> 10.6 + 6.1, 15,625 32 + 13 -> 13.1 + 7.0, 39,304
// 33 + 14 -> 23.6 + 11.8, 64,000 33 + 15 -> 43 + 15).
constexpr uint32_t kKahanMax = 49152;

}  // namespace

bool row_gathers_in_use(const LaunchCfg& c, const StepBuffers& b) {
    return c.n <= (c.precision == SPH_PREC_KAHAN ? kKahanMax : kRowGatherMax) && c.max_cap <= kMaskCap && b.masks && b.pairs &&
           b.pair_cnt && b.rec && b.xyz;
}

void launch_density_rows(const LaunchCfg& c, const StepBuffers& b, hipStream_t s) {
    const auto launch = [&](auto batch) {
        constexpr bool kBatch = decltype(batch)::value;
        if (c.precision == SPH_PREC_FAST)
            density_rows<kBatch, SPH_PREC_FAST>(c, b, s);
        else if (c.precision == SPH_PREC_KAHAN)
            density_rows<kBatch, SPH_PREC_KAHAN>(c, b, s);
        else
            density_rows<kBatch, SPH_PREC_REFERENCE>(c, b, s);
    };
    c.tab ? launch(std::true_type{}) : launch(std::false_type{});
}

void launch_force_rows(const LaunchCfg& c, const StepBuffers& b, float4* vel_out, float4* dvel, hipStream_t s) {
    const auto launch = [&](auto batch) {
        constexpr bool kBatch = decltype(batch)::value;
        if (c.precision == SPH_PREC_FAST)
            force_rows<kBatch, SPH_PREC_FAST>(c, b, vel_out, dvel, s);
        else if (c.precision == SPH_PREC_KAHAN)
            force_rows<kBatch, SPH_PREC_KAHAN>(c, b, vel_out, dvel, s);
        else
            force_rows<kBatch, SPH_PREC_REFERENCE>(c, b, vel_out, dvel, s);
    };
    c.tab ? launch(std::true_type{}) : launch(std::false_type{});
}

namespace {

// The pair scale of n pairs by both sequences (sph_pair_selftest).
__global__ __launch_bounds__(256) void k_pair_selftest(uint32_t n, PairScale c, const float* __restrict__ in,
                                                       float2* __restrict__ fast, float2* __restrict__ general,
                                                       uint32_t* __restrict__ in_range) {
    const uint32_t k = blockIdx.x * 256u + threadIdx.x;
    if (k >= n) return;
    const float r2 = in[k], psum = in[(size_t)n + k], rr = in[2 * (size_t)n + k];
    PairRange range(c);
    float2 f, g;
    pair_scale(c, r2, psum, rr, range, f.x, f.y);
    pair_scale_ieee(c, r2, psum, rr, g.x, g.y);
    fast[k] = f;
    general[k] = g;
    in_range[k] = range.ok() ? 1u : 0u;
}

}  // namespace
}  // namespace sph

extern "C" int sph_pair_selftest(uint32_t n, const float par[4], const float* r2, const float* psum, const float* rr,
                                 float* fast, float* general, uint32_t* in_range) {
    if (!par || !r2 || !psum || !rr || !fast || !general || !in_range || n > (1u << 26))
        return SPH_ERR_INVALID_ARGUMENT;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return SPH_ERR_NO_DEVICE;
    if (n == 0) return SPH_OK;
    const size_t row = (size_t)n * sizeof(float);
    void* mem = nullptr;  // r2, psum, rr, in_range | fast | general
    hipError_t e = sph::device_malloc(&mem, 8 * row);
    if (e != hipSuccess) return e == hipErrorOutOfMemory ? SPH_ERR_OUT_OF_MEMORY : SPH_ERR_DEVICE;
    char* m = static_cast<char*>(mem);
    const float* in[3] = {r2, psum, rr};
    for (int k = 0; k < 3 && e == hipSuccess; ++k) e = hipMemcpy(m + k * row, in[k], row, hipMemcpyHostToDevice);
    const size_t at = 4 * row;  // (a multiple of 16: the pairs are aligned)
    if (e == hipSuccess) {
        const sph::dev::PairScale c{par[0], par[1], par[2], par[3]};
        hipLaunchKernelGGL(sph::k_pair_selftest, dim3((n + 255u) / 256u), dim3(256), 0, 0, n, c,
                           reinterpret_cast<const float*>(m), reinterpret_cast<float2*>(m + at),
                           reinterpret_cast<float2*>(m + at + 2 * row), reinterpret_cast<uint32_t*>(m + 3 * row));
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(in_range, m + 3 * row, row, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(fast, m + at, 2 * row, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(general, m + at + 2 * row, 2 * row, hipMemcpyDeviceToHost);
    (void)hipFree(mem);
    return e == hipSuccess ? SPH_OK : SPH_ERR_DEVICE;
}
