// sph_fast.hip - the density gather of the FAST precision mode.
//
// The same step as the reference-order kernels (sph_kernels.hip), under the
// float contract of the task rather than bit-exactness: integer outputs stay
// exact (cell keys, order, cell ranges, and the neighbour sets with the
// per-cell cap and both predicates, r2 < h2 for the density and
// r2 <= force_r2_max for the force), every float is within 1e-5 of the FP32
// restatement of the reference and of the FP64 twin, condition-scaled.  That
// frees the arithmetic: the density is a sum per row of cells with fused
// multiply-adds instead of per-cell partial sums added in cell order
// (source/CUDA/Kernel_Cell.cui:142-199); the candidate walk and predicates
// are the reference's.  The force is the reference order's pair-entry
// kernel (k_force_entries, sph_kernels.hip) with a partial sum per row
// instead of per cell.
//
// Pair lists.  The density walk tests candidates four at a time (four
// consecutive slots of one row's run); a group with at least one force pair
// leaves one list entry, (first slot << kPairSlotShift) | 4-bit mask of the
// pairs (in the new-cell flag's place a bit that is the same for a row's
// entries and flips for the next row with any), so the walk spends one LDS
// write per group rather than per pair.  Entries are
// group-major (entries 4g .. 4g + 3 of slot i in the uint4 at g n + i) and
// there is room for every group the capped walk can produce (27 cells of at
// most ceil(max_par_in_cell / 4) groups, and one more where the particle
// splits its own row's run: list_entries), so the lists never overflow.  The
// count word of a slot holds the entries (low 16 bits) and the pairs (high
// 16 bits).
#include "sph_device.hpp"

namespace sph {
namespace {

using namespace dev;

constexpr int kBlock = 256;
constexpr int kGroup = 4;      // candidates per iteration of the density walk

// Density + EOS, the force pair list and the force record of one slot per
// thread.
//
// The walk goes by rows: the neighbour cells (dx = -1, 0, 1) of one (dy, dz)
// have consecutive keys, so their slots form one run, and the candidates of
// a row are that run, four consecutive slots at a time (three 16-byte loads
// from the packed positions).  A run breaks only after a cell capped at
// max_par_in_cell (its slots past the cap are not candidates); the slots
// before the break are walked as a run of their own, and the own row's run
// is split at the particle itself.  The lanes of one cell then walk the same
// runs in step (in the own row, nearly) and load the same cache lines, and a
// row costs one loop instead of three.  Culling drops a side
// cell of a row whose box is farther than h (the middle cell of a row that
// is kept is never farther than the row).
//
// The force record of slot i is two float4: (x, y, z, rho) and
// (vx, vy, vz, p), everything the force reads of a particle in one aligned
// 32-byte block.
template <bool kBatch, bool kByRow>
__global__ __launch_bounds__(kBlock) void k_density_fast(sph_params one, const sph_params* __restrict__ tab,
                                                         const uint32_t* __restrict__ sid, uint32_t n,
                                                         const float4* __restrict__ pos,
                                                         const float* __restrict__ xyz,
                                                         const float4* __restrict__ vel,
                                                         const uint32_t* __restrict__ cell_start,
                                                         const uint32_t* __restrict__ cell_end,
                                                         float2* __restrict__ rhop, float4* __restrict__ rec,
                                                         uint4* __restrict__ nbr, uint32_t* __restrict__ nnb,
                                                         const uint32_t* __restrict__ counters) {
    using Ring = PairRing<kByRow, kBlock>;
    __shared__ uint32_t ring_mem[Ring::kSlots * kBlock];
    const uint32_t i = xcd_tile(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    if (i >= n) return;
    uint32_t scene;
    const sph_params& p = scene_params<kBatch>(one, tab, sid, i, scene);
    const float4 xi = pos[i];
    CellWalk w;
    w.init(p, xi.x, xi.y, xi.z, walk_culled(counters));
    const float h2 = p.h2, r2f = p.force_r2_max;
    const uint32_t on = pair_bits_on(r2f);
    const float inv_h2 = 1.0f / h2;
    Ring ring(ring_mem);
    float total = 0.0f;  // of (1 - r2 / h2)^3 over the rows; times h2^3 below
    float sum = 0.0f;    // the row's part of it
    uint32_t par = 0;    // flips after each row with an entry (in kPairNewCell's place)
    // The candidates j0 .. j0 + 3; in the tail group of a run only the
    // first `left` of them (the others take r2 = +inf, which fails both
    // predicates).  The predicates use the reference's r2 exactly.  The
    // density weight is (1 - r2 / h2)^3 clamped to [0, 1], one fused
    // multiply-add with an output clamp: 0 for r2 >= h2 and for a NaN r2,
    // as the reference's (r2 < h2 ? (h2 - r2)^3 : 0) is.
    // The candidates' positions come from the packed array (packed_group:
    // three loads for four candidates); those loads are what bounds this
    // walk.
    auto group = [&](const float (&cx)[kGroup], const float (&cy)[kGroup], const float (&cz)[kGroup], uint32_t tag,
                     uint32_t left, auto tail) {
        constexpr bool kTail = decltype(tail)::value;
        float r2[kGroup];
#pragma unroll
        for (int k = 0; k < kGroup; ++k) {
            const float rx = xi.x - cx[k], ry = xi.y - cy[k], rz = xi.z - cz[k];
            r2[k] = rx * rx + ry * ry + rz * rz;
            if constexpr (kTail)
                if (k > 0) r2[k] = left > (uint32_t)k ? r2[k] : __builtin_huge_valf();
            const float c = fminf(fmaxf(__builtin_fmaf(r2[k], -inv_h2, 1.0f), 0.0f), 1.0f);
            sum = __builtin_fmaf(c * c, c, sum);
        }
        const uint32_t bits = pair_bits(r2, r2f, on);
        ring.put(tag, bits, nonzero_lanes(bits), nbr, n, i);
    };
    // the candidates [s, e): full groups, then one tail group
    // (tag: the group's first slot, shifted into place for its entry).  In a
    // single scene each group's loads go out before its predecessor's
    // arithmetic: an array that fills the chip with four waves per SIMD or
    // fewer waits for them (density, us: 79,507 particles 33.2 -> 30.0,
    // 157,464 37.6 -> 35.0, 551,368 78.8 -> 77.0, 1,048,576 unchanged).  A
    // batch, with the scene's parameters in registers, loses a wave per SIMD
    // to the second group and is slower with it (380 -> 384).
    auto walk_run = [&](uint32_t s, uint32_t e) {
        uint32_t q = s * kSlotBytes, tag = (s << kPairSlotShift) | par, left = e - s;
        float cx[kGroup], cy[kGroup], cz[kGroup];
        if constexpr (kBatch) {
            for (; left >= (uint32_t)kGroup; left -= kGroup, q += kGroup * kSlotBytes, tag += kGroup << kPairSlotShift) {
                packed_group(xyz, q, cx, cy, cz);
                group(cx, cy, cz, tag, kGroup, std::false_type{});
            }
            if (!left) return;
            packed_group(xyz, q, cx, cy, cz);
        } else {
            if (!left) return;
            packed_group(xyz, q, cx, cy, cz);
            while (left > (uint32_t)kGroup) {
                float nx[kGroup], ny[kGroup], nz[kGroup];
                q += kGroup * kSlotBytes;
                packed_group(xyz, q, nx, ny, nz);
                group(cx, cy, cz, tag, kGroup, std::false_type{});
#pragma unroll
                for (int k = 0; k < kGroup; ++k) cx[k] = nx[k], cy[k] = ny[k], cz[k] = nz[k];
                left -= kGroup, tag += kGroup << kPairSlotShift;
            }
        }
        group(cx, cy, cz, tag, left, std::true_type{});
    };
    // a run of the particle's own row without the particle itself (it is in
    // the run unless its cell is capped before it)
    auto walk_own = [&](uint32_t s, uint32_t e) {
        if (i >= s && i < e) {
            walk_run(s, i);
            walk_run(i + 1, e);
        } else {
            walk_run(s, e);
        }
    };
#pragma unroll 1
    for (int dz = -1; dz <= 1; ++dz) {
#pragma unroll 1
        for (int dy = -1; dy <= 1; ++dy) {
            const CellWalk::Row row = w.row(dy, dz);
            if (!row.ok) continue;
            const bool own = (dy | dz) == 0;
            const uint32_t before = ring.count;
            sum = 0.0f;
            uint32_t rs = 0, re = 0;  // the run so far (empty: rs == re)
#pragma unroll 1
            for (int dx = -1; dx <= 1; ++dx) {
                uint32_t s, e;
                if (!w.open_in(row, dx, cell_start, cell_end, s, e)) continue;
                if (s != re) {
                    // a break: a capped cell before (or the row's first open cell)
                    if (own)
                        walk_own(rs, re);
                    else
                        walk_run(rs, re);
                    rs = s;
                }
                re = e;
            }
            if (own)
                walk_own(rs, re);
            else
                walk_run(rs, re);
            total = total + sum;
            par ^= ring.count != before ? kPairNewCell : 0u;
            ring.row_end(nbr, n, i);
        }
    }
    nnb[i] = ring.finish(nbr, n, i);
    const float rho = (total * (((p.poly6_kern * h2) * h2) * h2)) * p.particle_mass;
    const float pr = eos(p, rho);
    rhop[i] = make_float2(rho, pr);
    const float4 vi = vel[i];
    rec[2 * (size_t)i] = make_float4(xi.x, xi.y, xi.z, rho);
    rec[2 * (size_t)i + 1] = make_float4(vi.x, vi.y, vi.z, pr);
}

inline uint32_t blocks_for(uint32_t n) { return n == 0 ? 1u : (n + kBlock - 1) / kBlock; }

}  // namespace

uint32_t fast_list_groups(uint32_t max_par_in_cell, uint32_t n) {
    const uint32_t least = n <= kRowGatherMax ? kMaskCap : 0u;  // a row lane's list has room for full cells
    const uint32_t cap = max_par_in_cell < least ? least : max_par_in_cell;
    return list_groups(cap);
}

hipError_t launch_density_fast(const LaunchCfg& c, const StepBuffers& b, float4* rec, uint4* nbr, uint32_t* nnb,
                               hipStream_t s) {
    if (!b.xyz) return hipErrorInvalidValue;  // the place kernel packs the positions
    if (row_gathers_in_use(c, b)) {
        launch_density_rows(c, b, s);
        return hipGetLastError();
    }
    const dim3 grid(blocks_for(c.n)), block(kBlock);
    const auto launch = [&](auto batch, auto by_row) {
        hipLaunchKernelGGL((k_density_fast<decltype(batch)::value, decltype(by_row)::value>), grid, block, 0, s, c.one,
                           c.tab, b.sid_cur, c.n, b.pos_cur, b.xyz, b.vel_cur, b.cell_start, b.cell_end, b.rhop, rec,
                           nbr, nnb, b.counters);
    };
    const std::true_type yes{};
    const std::false_type no{};
    const bool by_row = c.max_cap <= kMaskCap;  // a row's entries fit the ring
    if (c.tab)
        by_row ? launch(yes, yes) : launch(yes, no);
    else
        by_row ? launch(no, yes) : launch(no, no);
    return hipGetLastError();
}


}  // namespace sph
