// lj_candidates.h -- the 27-cell candidate count over rows of cells, a kernel of its own
// (binning.hip) or further workgroups of a force launch (force.hip), and where a batch
// counts (batch.hip).
//
// Reference: ComputeNbInteractions (Cuda-version/cudaLJ.cu:255-297).
#pragma once

#include "lj_internal.h"

namespace lj {

// The lane's part of sum over cells of n_c * (S_c - 1), S_c = the clipped 27-cell count
// including c; equals the per-particle count of ComputeNbInteractions (cudaLJ.cu:278-292).
// One wave per (y,z) row of cells at a time, rows wave, wave + nwaves, ..., lanes along x:
// the row's neighbour rows are wave-uniform, so a cell's 27-cell count is nine x-range
// differences of the offsets (coalesced across the lanes) and no per-cell index
// arithmetic.
__device__ inline unsigned long long candidate_rows(const uint32_t* __restrict__ off, const GridGeom& g, uint32_t wave,
                                                    uint32_t nwaves) {
    const int32_t gx = g.g[0], gy = g.g[1], gz = g.g[2];
    const uint32_t nrows = (uint32_t)gy * (uint32_t)gz;
    const int32_t lane = (int32_t)__lane_id();
    unsigned long long v = 0;
    for (uint32_t r = wave; r < nrows; r += nwaves) {
        const int32_t cy = (int32_t)(r % (uint32_t)gy), cz = (int32_t)(r / (uint32_t)gy);
        const int32_t z0 = cz > 0 ? cz - 1 : 0, z1 = cz < gz - 1 ? cz + 1 : gz - 1;
        const int32_t y0 = cy > 0 ? cy - 1 : 0, y1 = cy < gy - 1 ? cy + 1 : gy - 1;
        const uint32_t* home = off + (size_t)r * (size_t)gx;
        for (int32_t cx = lane; cx < gx; cx += 64) {
            const uint32_t nh = home[cx + 1] - home[cx];
            if (!nh) continue;
            // x-cells x0 .. xe - 1 of each neighbour row (the counts of at most n
            // particles fit 32 bits)
            const int32_t x0 = cx > 0 ? cx - 1 : 0, xe = cx < gx - 1 ? cx + 2 : gx;
            uint32_t sum = 0;
            for (int32_t zz = z0; zz <= z1; ++zz)
                for (int32_t yy = y0; yy <= y1; ++yy) {
                    const uint32_t* rw = off + ((size_t)zz * (size_t)gy + (size_t)yy) * (size_t)gx;
                    sum += rw[xe] - rw[x0];
                }
            v += (unsigned long long)nh * (sum - 1);
        }
    }
    return v;
}

// Whether a batch on the cell_edge grid, of `total` cells and at most `most` in one system,
// counts its candidates in the final reduction, one workgroup a system, or on the second
// stream beside the force pass.  The reduction walks a system's cells 256 at a time after
// the force pass: it saves the fork and join (20-40 us) while its longest system takes no
// longer.  us, reduction and second stream: one system of 36,864 particles in 4,096 cells 73
// and 76, 72,000 in 8,000 94 and 85, 2,400 in 8,000 62 and 75, 140,625 in 15,625 139 and 105,
// 48,039 on a sphere in 125,000 425 and 105; 8 systems of 36,864 125 and 133, 72,000 201 and
// 198, 140,625 389 and 380; 64 of 4,687 in 15,625 cells 135 and 182.  In large batches the
// force pass's tail hides the count (4,096 systems of 12.8M cells in all: 138 us).
constexpr uint64_t kReduceCells = 1u << 20;
constexpr uint32_t kReduceSystem = 8192;
inline bool count_in_reduction(uint64_t total, uint32_t most) { return total <= kReduceCells && most <= kReduceSystem; }

}  // namespace lj
