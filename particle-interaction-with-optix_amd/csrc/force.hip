// force.hip -- cell-grid Lennard-Jones forces/energies, neighbour lists and reorder.
//
// Reference: ComputeParticleInterationsParPartNoLoop (Cuda-version/cudaLJ.cu:299-341)
// computes, per particle in cell order, the potential against every particle of
// the clipped 27-cell stencil, with no cutoff and sigma = epsilon = 1, and no force.
// Here the pair set is chosen by the predicate of lj_params (the canonical one is
// the OptiX AABB test, SDK/optixMultiSphereAABB/optixLJ.cu:162), the force is the
// analytic gradient of the same potential, and per-particle outputs are written
// in the caller's order.
//
// Cell order is z-major (cudaLJ.cu:127-134), so the x-cells of one (y,z) row of the
// stencil are one contiguous slot range: the 27 cells are 9 ranges (the stencil loop
// itself is stencil_pairs in lj_stencil.h).
#include <cmath>

#include "lj_candidates.h"
#include "lj_rows.h"
#include "lj_sort.h"
#include "lj_stencil27.h"

namespace lj {

namespace {

// One thread per sorted slot k, blocks of `block` threads (<= 256), the lane queues in
// dynamic LDS (depth x block entries of 16 bytes, one block of rings per wave; none
// without QUEUE).  Outputs go to the caller's order (pi.w holds the original index),
// or, when `so` is set (lj_compute_sorted), to the sorted slot k together with the
// particle's position and original index; each workgroup's totals go to sums and are
// reduced later in a fixed order.
// OUT: how the outputs are stored -- 0 ordinary stores, 1 non-temporal stores, 2 one
// non-temporal staged record per particle at its caller index (large outputs at
// shuffled indices; never with `so`).
template <int PRED, int PREC, bool VIR, bool QUEUE, int OUT>
__global__ __launch_bounds__(kMaxBlock, 8) void k_force(const float4* __restrict__ pos, const uint32_t* __restrict__ cell_of,
                                                     const uint32_t* __restrict__ off, uint32_t n, GridGeom g, int Rx,
                                                     int R, Trim tr, PairConst c, uint32_t depth, float* __restrict__ fx,
                                                     float* __restrict__ fy, float* __restrict__ fz,
                                                     float* __restrict__ e, BlockSums* __restrict__ sums, SortedOut so,
                                                     float4* __restrict__ stage) {
    extern __shared__ QEntry queue[];
    const uint32_t blk = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t k = blk * blockDim.x + threadIdx.x;
    // the slot rebuilt after the pair loop from wave-uniform values and the lane id, so
    // that no per-lane index stays live across it (64 VGPRs are the budget)
    const uint32_t wbase = blk * blockDim.x + (__builtin_amdgcn_readfirstlane(threadIdx.x) & ~(kWaveSize - 1u));
    const bool active = k < n;
    PairSums<PREC, PRED == LJ_PRED_CUDALJ, VIR> acc;
    const float4 pi = active ? pos[k] : make_float4(0.f, 0.f, 0.f, 0.f);
    acc.set_i(pi);
    acc.allow_exact_diff(c, pi, active);
    const uint32_t np = stencil_pairs<PRED, PREC, VIR, QUEUE>(pos, off, k, active, pi, g, 0u, active ? cell_of[k] : 0u,
                                                              Rx, R, tr, c,
                                                              queue + (threadIdx.x / kWaveSize) * depth * kWaveSize +
                                                                  __lane_id(),
                                                              depth, acc);
    double esum = 0.0, vsum = 0.0;
    const uint32_t ks = wbase + __lane_id();  // = k
    if (ks < n) {
        // caller order, or the sorted slot together with the particle itself
        const float4 ps = pos[ks];
        const float ox = (float)(-c.e24 * (double)acc.ax.value());
        const float oy = (float)(-c.e24 * (double)acc.ay.value());
        const float oz = (float)(-c.e24 * (double)acc.az.value());
        const double ei = c.e4 * (double)acc.ae.value();
        if constexpr (OUT == 2) {
            store_staged(&stage[__float_as_uint(ps.w)], ox, oy, oz, (float)ei);
        } else {
            constexpr bool NT = OUT == 1;
            const bool sorted = so.x != nullptr;  // uniform
            const uint32_t i = sorted ? ks : __float_as_uint(ps.w);
            if (sorted) {
                store_out<NT>(&so.x[ks], ps.x);
                store_out<NT>(&so.y[ks], ps.y);
                store_out<NT>(&so.z[ks], ps.z);
                if (so.perm) so.perm[ks] = __float_as_uint(ps.w);
            }
            store_out<NT>(&fx[i], ox);
            store_out<NT>(&fy[i], oy);
            store_out<NT>(&fz[i], oz);
            if (e) store_out<NT>(&e[i], (float)ei);
        }
        esum = ei;
        vsum = c.e24 * (double)acc.av.value();
    }
    store_block_sums<true, false>(&sums[blk], esum, vsum, np, 0ull);
}

// The same for systems that two_lanes takes: two lanes per particle (stencil27), outputs
// (which fit in the L2s) stored ordinarily.  The workgroups past the first nforce count the
// 27-cell candidates of the same grid (none when no result is wanted): they need only the
// offsets, and a launch of their own costs 4-5 us.
// LDS: every workgroup first copies all the particles to LDS and walks them there: a system
// of up to kLdsParticles leaves a SIMD one wave at most, which waits out each load, and is
// otherwise bound by the issue of that wave's steps.  lj_compute, us, from the caches -> from
// LDS: 200 particles of 50 neighbours 32.2 -> 31.7, 500 of 64 44.4 -> 43.0, 1,000 42.5 -> 42.1,
// 1,200 level, 2,048 of 30 36.3 -> 37.3, of 5 27.0 -> 27.9.
constexpr uint32_t kLdsParticles = 1024;

template <int PRED, int PREC, bool VIR, bool LDS, bool AHEAD>
__global__ __launch_bounds__(kMaxBlock, LDS || AHEAD ? 4 : 8) void k_force27(const float4* __restrict__ pos,
                                                      const uint32_t* __restrict__ cell_of,
                                                      const uint32_t* __restrict__ off, uint32_t n, GridGeom g, Trim tr,
                                                      PairConst c, float* __restrict__ fx, float* __restrict__ fy,
                                                      float* __restrict__ fz, float* __restrict__ e, uint32_t nforce,
                                                      BlockSums* __restrict__ sums, SortedOut so) {
    if (blockIdx.x >= nforce) {
        const uint32_t waves = blockDim.x / kWaveSize;
        const uint32_t wave = (blockIdx.x - nforce) * waves + __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
        const unsigned long long nc = candidate_rows(off, g, wave, (gridDim.x - nforce) * waves);
        store_block_sums<false, true>(&sums[blockIdx.x], 0.0, 0.0, 0ull, nc);
        return;
    }
    const uint32_t blk = xcd_block(blockIdx.x, nforce);
    const uint32_t k = (blk * blockDim.x + threadIdx.x) / kPairLanes;
    const uint32_t wbase = (blk * blockDim.x + (__builtin_amdgcn_readfirstlane(threadIdx.x) & ~(kWaveSize - 1u))) / kPairLanes;
    const bool active = k < n;
    PairSums<PREC, PRED == LJ_PRED_CUDALJ, VIR> acc;
    const float4 pi = active ? pos[k] : make_float4(0.f, 0.f, 0.f, 0.f);
    acc.set_i(pi);
    acc.allow_exact_diff(c, pi, active);
    __shared__ float4 all[LDS ? kLdsParticles + kPosSpare : 1];
    if constexpr (LDS) {
        for (uint32_t t = threadIdx.x; t < n; t += blockDim.x)
            reinterpret_cast<f32x4*>(all)[t] = reinterpret_cast<const f32x4*>(pos)[t];
        __syncthreads();
    }
    const uint32_t np = stencil27<PRED, AHEAD, !LDS>(LDS ? all : pos, off, k, active, pi, g, 0u, active ? cell_of[k] : 0u, tr, c, acc);
    acc.template merge<kPairLanes>();
    double esum = 0.0, vsum = 0.0;
    const uint32_t ks = wbase + __lane_id() / kPairLanes;  // = k
    if (ks < n && (__lane_id() & 1u) == 0u) {
        const float4 ps = pos[ks];
        const double ei = c.e4 * (double)acc.ae.value();
        const bool sorted = so.x != nullptr;  // uniform
        const uint32_t i = sorted ? ks : __float_as_uint(ps.w);
        if (sorted) {
            so.x[ks] = ps.x;
            so.y[ks] = ps.y;
            so.z[ks] = ps.z;
            if (so.perm) so.perm[ks] = __float_as_uint(ps.w);
        }
        fx[i] = (float)(-c.e24 * (double)acc.ax.value());
        fy[i] = (float)(-c.e24 * (double)acc.ay.value());
        fz[i] = (float)(-c.e24 * (double)acc.az.value());
        if (e) e[i] = (float)ei;
        esum = ei;
        vsum = c.e24 * (double)acc.av.value();
    }
    store_block_sums<true, false>(&sums[blk], esum, vsum, np, 0ull);
}

__global__ __launch_bounds__(256) void k_split_outputs(const float4* __restrict__ stage, uint32_t n,
                                                       float* __restrict__ fx, float* __restrict__ fy,
                                                       float* __restrict__ fz, float* __restrict__ e) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    const f32x4 v = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(stage) + i);
    fx[i] = v.x;
    fy[i] = v.y;
    fz[i] = v.z;
    if (e) e[i] = v.w;
}

__global__ __launch_bounds__(256) void k_coarse_counts(const uint32_t* __restrict__ foff, GridGeom fg, GridGeom cg, int Kx,
                                                       int K, uint32_t* __restrict__ ccount) {
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= cg.ncells) return;
    ccount[c] = coarse_count(foff, fg, cg, Kx, K, c);
}

// The workgroups' sums in a fixed order: stage 1 (res NULL) sums chunks of kFinalChunk of
// them into out (one workgroup per chunk), stage 2 (one workgroup) sums those, or up to
// kFinalOne sums directly, and further candidate counts into *res.
__global__ __launch_bounds__(1024) void k_finalize(const BlockSums* __restrict__ sums, uint32_t nblocks,
                                                   const unsigned long long* __restrict__ cand, uint32_t ncand,
                                                   const int* __restrict__ overflow, BlockSums* __restrict__ out,
                                                   lj_result* __restrict__ res) {
    __shared__ BlockSums total;
    double a = 0.0, b = 0.0;
    unsigned long long np = 0, nc = 0;
    const uint32_t lo = res ? 0 : blockIdx.x * kFinalChunk;
    const uint32_t hi = res ? nblocks : (lo + kFinalChunk < nblocks ? lo + kFinalChunk : nblocks);
    for (uint32_t q = lo + threadIdx.x; q < hi; q += blockDim.x) {
        a += sums[q].e;
        b += sums[q].v;
        np += sums[q].np;
        nc += sums[q].nc;
    }
    if (res)
        for (uint32_t q = threadIdx.x; q < ncand; q += blockDim.x) nc += cand[q];
    store_block_sums<true, true>(&total, a, b, np, nc);
    if (threadIdx.x != 0) return;
    if (!res) {
        out[blockIdx.x] = total;
    } else if (overflow && *overflow) {
        *res = lj_result{__builtin_nan(""), __builtin_nan(""), total.nc, ~0ull};
    } else {
        *res = lj_result{0.5 * total.e, 0.5 * total.v, total.nc, total.np};
    }
}

// ------------------------------------------------------------------ pair lists
// Sixteen lanes take a row of up to 256 entries into registers (the wave's four rows by
// the longest of them), sort it with lane exchanges that need no LDS, and store it; a
// longer row is sorted by the whole workgroup in LDS, or, above 4096 entries, where it
// lies.  Bound by the list's bytes, read and written once: 500,009 rows of 72 entries (36M,
// 290 MB moved) in 108 us, 2.7 TB/s.  As one thread's insertion sort in global memory, at
// the end of the kernel that lists the partners, that kernel took 7172 us, and 479 us
// without it.  A wave takes 16 rows, 4 lanes each, while none of them has more than 16
// entries, then in four turns of 16 lanes: lists of short rows are bound by the number of
// waves and of lanes that look at a row's length (lj_lbvh_pairs as a whole, us, four rows a
// wave -> 16: 3M uniform particles of 0.5 partners 1,461 -> 1,312, of 12 2,815 -> 2,755;
// 250,007 in clusters of 46 553 -> 555).  LONG: the rows of up to kRegRow entries are sorted already, so a thread looks
// at one row's length (with 16 lanes a row that took 15 us on those 500,009 rows).
template <bool LONG>
__global__ __launch_bounds__(kSortThreads) void k_sort_rows(const unsigned long long* __restrict__ rows, uint32_t n,
                                                            uint32_t* __restrict__ cols,
                                                            const uint32_t* __restrict__ draft) {
    constexpr uint32_t kBlock = LONG ? kSortThreads : kBlockRows;  // rows of a workgroup
    __shared__ uint32_t stage[kLdsRow];
    const uint32_t first = block_index() * kBlock;
    const uint32_t i = first + (LONG ? threadIdx.x : threadIdx.x / kShortLanes);
    unsigned long long r0 = 0, len = 0;
    if (i < n) {
        r0 = rows[i];
        len = rows[i + 1] - r0;
    }
    const bool fits = len <= kRegRow;
    if constexpr (!LONG) {
        // rows to move or to sort
        const uint32_t m = fits && (draft || len > 1) ? (uint32_t)len : 0u;
        auto from = [&](uint32_t row, unsigned long long at) { return draft ? draft + (size_t)row * kDraftRow : cols + at; };
        if (!__any(m > kShortRow)) {
            sort_short_rows(from(i, r0), cols + r0, m);
        } else {
            const uint32_t wrow = first + threadIdx.x / kWaveSize * (kWaveSize / kShortLanes);  // the wave's first
            for (int q = 0; q < kWaveSize / kShortLanes; q += kWaveSize / kRowLanes) {
                const int row = q + (int)__lane_id() / kRowLanes, lane = row * kShortLanes;
                const unsigned long long at = (unsigned long long)__shfl((uint32_t)(r0 >> 32), lane, kWaveSize) << 32 |
                                              __shfl((uint32_t)r0, lane, kWaveSize);
                sort_four_rows(from(wrow + row, at), cols + at, __shfl(m, lane, kWaveSize));
            }
        }
    }
    if (!__syncthreads_or(!fits)) return;
    for (uint32_t q = first; q < first + kBlock && q < n; ++q) {
        const unsigned long long s0 = rows[q], sl = rows[q + 1] - s0;
        if (sl <= kRegRow) continue;  // the same for every thread of the workgroup
        if (sl <= kLdsRow) {
            for (uint32_t t = threadIdx.x; t < sl; t += kSortThreads) stage[t] = cols[s0 + t];
            __syncthreads();
            block_sort(stage, (uint32_t)sl);
            for (uint32_t t = threadIdx.x; t < sl; t += kSortThreads) cols[s0 + t] = stage[t];
            __syncthreads();
        } else {
            // in place: __syncthreads orders the workgroup's own global accesses
            block_sort(cols + s0, (uint32_t)sl);
        }
    }
}

// Partners from the rc grid.  A wave takes kPairSlots consecutive sorted slots; the ones
// in one cell (a run) share the 27 cells' particles, whose slots are nine ranges, taken
// as one sequence: the lanes hold up to kPairBatches x 64 of them in registers and test
// each of the run's particles, wave-uniform, against all of them, so that a partner is
// loaded once per run, a ballot is the answer for 64 candidates, and no lane waits for
// another's longer walk.  Where cells hold few particles (kSparseRuns), the run of one or
// two slots would wait alone for its ranges and then for its candidates: there each of the
// workgroup's slots gets a lane in every wave, and a wave a quarter of the nine rows.
// FILL = false counts (a partner with a multiplicity above one
// is listed once): rowcnt[original index].  FILL = true lists: four particles at a time
// collect their partners' indices in LDS, and 16 lanes each sort them in registers and
// store them; rows above kRegRow entries are stored unsorted (sort_long_rows follows).
// Bound by VALU issue: 500,009 particles, 465 candidates and 72 partners each: count 92 us,
// list 287 us (one thread per particle: 159 and 479 us, and 108 us more for the sort).  Where
// cells hold few particles, by the latency of the offsets' and the candidates' loads.
constexpr int kPairThreads = 256;
constexpr int kPairSlots = 16;
constexpr int kPairBatches = 8;
constexpr uint32_t kNoSlot = 0xffffffffu;
constexpr uint32_t kPairChunk = kPairBatches * kWaveSize;
// entries between the four lists of a wave: a row and 16 more, so that the four groups of
// 16 lanes read different banks
constexpr int kListStride = (int)kRegRow + kRowLanes;
// Runs among a workgroup's 64 slots from which on it takes them as sparse: four slots a cell.
// lj_pairs as a whole, us, runs only -> with the sparse form (one thread per particle, with
// its sort in the list): 1,000,000 uniform particles of 0.5 neighbours 793 -> 236 (230), of 3
// 714 -> 268 (304), of 6 613 -> 316 (456), of 12 549 -> 409 (864), of 20 514 -> 504 (1,635);
// on a sphere of 3 1,127 -> 700 (790).  With the line at 20 runs the times of 6, 12 and 20
// neighbours were 1, 6 and 4 % longer.  Still behind one thread per particle at 3,000,000
// uniform particles of 0.5 and 1.5 neighbours, 550 and 569 against 490 and 512, where a cell
// in eight or less than one in two holds a particle: a workgroup of 256 particles there
// shared more of the offsets' lines.
constexpr int kSparseRuns = 16;
// A workgroup's sparse rows share its lists.
constexpr uint32_t kSparseRow = 4 * kListStride / kPairSlots;

__device__ inline void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int PRED, bool FILL>
__global__ __launch_bounds__(kPairThreads) void k_pairs(const float4* __restrict__ pos,
                                                        const uint32_t* __restrict__ cell_of,
                                                        const uint32_t* __restrict__ off, uint32_t n, GridGeom g,
                                                        PairConst c, uint32_t* __restrict__ rowcnt,
                                                        const unsigned long long* __restrict__ rows,
                                                        uint32_t* __restrict__ cols) {
    constexpr int kWaves = kPairThreads / kWaveSize;
    // every predicate but the two distance ones can accept the particle itself
    constexpr bool kSelf = PRED != LJ_PRED_AABB && PRED != LJ_PRED_CUSTOM;
    __shared__ uint32_t lists[FILL ? kWaves : 1][FILL ? 4 * kListStride : 1];
    __shared__ uint32_t partners[kWaveSize], lens[FILL ? kWaveSize : 1];
    __shared__ unsigned long long starts[FILL ? kWaveSize : 1];
    static_assert(kWaves * kPairSlots == kWaveSize, "a lane for each slot of the workgroup");
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
    const unsigned lane = __lane_id();
    const uint32_t base = xcd_block(block_index(), block_count()) * kWaves * kPairSlots;
    if (base >= n) return;  // the whole workgroup
    const uint32_t mine = base + lane;  // one of the workgroup's slots for each lane of every wave
    const bool within = mine < n;
    const uint32_t cell = cell_of[within ? mine : n - 1u];
    const uint32_t first = base + wave * kPairSlots, last = lane < (unsigned)kPairSlots ? first + lane : first + kPairSlots - 1u;
    const uint32_t key = cell_of[last < n ? last : n - 1u];  // of the wave's slots (loaded beside cell)
    const uint32_t before = (uint32_t)__shfl_up((int)cell, 1, kWaveSize);
    if (__popcll(__ballot(within && (lane == 0 || cell != before))) >= kSparseRuns) {
        // few slots to a cell: a lane for each of the workgroup's slots, a quarter of the nine
        // rows of cells for each wave, and a particle's partners in LDS in any order, since
        // the row is sorted before it is stored
        if (FILL && lane < (unsigned)kPairSlots) {
            const uint32_t slot = wave * kPairSlots + lane, k = base + slot;
            const uint32_t i = k < n ? __float_as_uint(pos[k].w) : 0u;
            const unsigned long long r0 = k < n ? rows[i] : 0ull;
            starts[slot] = r0;
            lens[slot] = k < n ? (uint32_t)(rows[i + 1] - r0) : 0u;
        }
        if (wave == 0) partners[lane] = 0u;
        __syncthreads();
        const uint32_t len = FILL ? lens[lane] : 0u;
        if (!FILL || !__any(len > kSparseRow)) {  // the same for every wave
            const bool walk = FILL ? len > 0u : within;
            const float4 pi = within ? pos[mine] : make_float4(0.f, 0.f, 0.f, 0.f);
            uint32_t* const list = &lists[0][0];
            int32_t cx, cy, cz;
            cell_coords(g, cell, cx, cy, cz);
            const int32_t x0 = cx > 0 ? cx - 1 : 0, x1 = cx < g.g[0] - 1 ? cx + 1 : g.g[0] - 1;
            constexpr int kTurns = (9 + kWaves - 1) / kWaves;
            uint32_t b[kTurns], e[kTurns];
#pragma unroll
            for (int u = 0; u < kTurns; ++u) {
                const int32_t r = (int32_t)wave + u * kWaves, zz = cz + r / 3 - 1, yy = cy + r % 3 - 1;
                b[u] = e[u] = 0;
                if (walk && r < 9 && zz >= 0 && zz < g.g[2] && yy >= 0 && yy < g.g[1]) {
                    const uint32_t row = (uint32_t)((zz * g.g[1] + yy) * g.g[0]);
                    b[u] = off[row + x0];
                    e[u] = off[row + x1 + 1];
                }
            }
            uint32_t m = 0;
#pragma unroll
            for (int u = 0; u < kTurns; ++u)
                for (uint32_t t = b[u]; t < e[u]; ++t) {
                    const float4 pj = pos[t];
                    const float d2 = dist2(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z);
                    if (t == mine || pair_mult<PRED>(c, pi, pj, d2) <= 0) continue;
                    if constexpr (FILL) list[lane * kSparseRow + atomicAdd(&partners[lane], 1u)] = __float_as_uint(pj.w);
                    else ++m;
                }
            if (!FILL && m) atomicAdd(&partners[lane], m);
            __syncthreads();
            if constexpr (!FILL) {
                if (wave == 0 && within) rowcnt[__float_as_uint(pi.w)] = partners[lane];
            } else if (!__any(len > kShortRow)) {
                // each wave a quarter of the rows
                const uint32_t slot = wave * kPairSlots + lane / kShortLanes;
                sort_short_rows(list + slot * kSparseRow, cols + starts[slot], lens[slot]);
            } else {
#pragma unroll
                for (uint32_t q = 0; q < kPairSlots; q += kWaveSize / kRowLanes) {
                    const uint32_t slot = wave * kPairSlots + q + lane / kRowLanes;
                    sort_four_rows(list + slot * kSparseRow, cols + starts[slot], lens[slot]);
                }
            }
            return;
        }
    }
    if (first >= n) return;  // the whole wave (no workgroup barrier below)
    const uint32_t cnt = n - first < (uint32_t)kPairSlots ? n - first : (uint32_t)kPairSlots;
    uint32_t found = 0;  // lane q: partners of slot first + q
    for (uint32_t j0 = 0; j0 < cnt;) {
        // the run: slots j0 .. j1 - 1, one cell (the keys are sorted)
        const uint32_t ck = __builtin_amdgcn_readlane(key, j0);
        const uint32_t j1 = 64u - (uint32_t)__builtin_clzll(__ballot(lane < cnt && key == ck));
        // its nine ranges of slots, one per lane; lanes 9 .. 63 hold empty ones
        uint32_t b = 0, len = 0;
        {
            int32_t cx, cy, cz;
            cell_coords(g, ck, cx, cy, cz);
            const int32_t zz = cz + (int32_t)(lane / 3u) - 1, yy = cy + (int32_t)(lane % 3u) - 1;
            if (lane < 9u && zz >= 0 && zz < g.g[2] && yy >= 0 && yy < g.g[1]) {
                const uint32_t row = (uint32_t)((zz * g.g[1] + yy) * g.g[0]);
                const int32_t x0 = cx > 0 ? cx - 1 : 0, x1 = cx < g.g[0] - 1 ? cx + 1 : g.g[0] - 1;
                b = off[row + x0];
                len = off[row + x1 + 1] - b;
            }
        }
        // candidate t lies in range r at slot t + shift[r], r the last one with start[r] <= t
        uint32_t start[9], shift[9], total = 0;
#pragma unroll
        for (int r = 0; r < 9; ++r) {
            start[r] = total;
            shift[r] = __builtin_amdgcn_readlane(b, r) - total;
            total += __builtin_amdgcn_readlane(len, r);
        }
        float4 pj[kPairBatches];
        uint32_t slot[kPairBatches];
        // candidates base .. base + kPairChunk - 1 (fewer at the end) into the registers
        auto load = [&](uint32_t base) {
#pragma unroll
            for (int u = 0; u < kPairBatches; ++u) {
                if (base + u * kWaveSize >= total) break;
                const uint32_t t = base + u * kWaveSize + lane;
                const uint32_t tc = t < total ? t : total - 1u;
                uint32_t s = tc + shift[0];
#pragma unroll
                for (int r = 1; r < 9; ++r) s = tc >= start[r] ? tc + shift[r] : s;
                pj[u] = pos[s];
                slot[u] = s;
                // past the end: no predicate with a distance accepts a NaN
                if (t >= total) {
                    pj[u].x = __builtin_nanf("");
                    slot[u] = kNoSlot;
                }
            }
        };
        // is this lane's candidate of batch u a partner of slot k (position pi)?
        auto partner = [&](int u, uint32_t k, const float4& pi) {
            const float d2 = dist2(pj[u].x - pi.x, pj[u].y - pi.y, pj[u].z - pi.z);
            bool in = pair_mult<PRED>(c, pi, pj[u], d2) > 0;
            if constexpr (kSelf) in = in && slot[u] != k && slot[u] != kNoSlot;
            return in;
        };
        if constexpr (!FILL) {
            for (uint32_t base = 0; base < total; base += kPairChunk) {
                load(base);
                for (uint32_t j = j0; j < j1; ++j) {
                    const float4 pi = pos[first + j];
                    uint32_t m = 0;
#pragma unroll
                    for (int u = 0; u < kPairBatches; ++u) {
                        if (base + u * kWaveSize >= total) break;
                        m += (uint32_t)__popcll(__ballot(partner(u, first + j, pi)));
                    }
                    found += lane == j ? m : 0u;
                }
            }
        } else {
            uint32_t* const list = lists[wave];
            for (uint32_t jq = j0; jq < j1; jq += 4) {
                unsigned long long r0[4];
                uint32_t len4[4], at[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t j = jq + q < j1 ? jq + q : j1 - 1u;
                    const uint32_t i = __float_as_uint(pos[first + j].w);
                    r0[q] = rows[i];
                    len4[q] = (uint32_t)(rows[i + 1] - r0[q]);
                    at[q] = 0;
                }
                for (uint32_t base = 0; base < total; base += kPairChunk) {
                    if (jq == j0 || total > kPairChunk) load(base);
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        if (jq + q >= j1) break;
                        const float4 pi = pos[first + jq + q];
#pragma unroll
                        for (int u = 0; u < kPairBatches; ++u) {
                            if (base + u * kWaveSize >= total) break;
                            const bool in = partner(u, first + jq + q, pi);
                            const uint64_t m = __ballot(in);
                            if (in) {
                                const uint32_t w = at[q] + sortk::rank_below(m);
                                const uint32_t v = __float_as_uint(pj[u].w);
                                if (len4[q] <= kRegRow) list[q * kListStride + w] = v;
                                else cols[r0[q] + w] = v;
                            }
                            at[q] += (uint32_t)__popcll(m);
                        }
                    }
                }
                wave_lds_sync();
                const uint32_t q = lane / kRowLanes;
                const unsigned long long rq = q == 0 ? r0[0] : q == 1 ? r0[1] : q == 2 ? r0[2] : r0[3];
                uint32_t mq = q == 0 ? len4[0] : q == 1 ? len4[1] : q == 2 ? len4[2] : len4[3];
                if (jq + q >= j1 || mq > kRegRow) mq = 0;
                sort_four_rows(list + q * kListStride, cols + rq, mq);
                wave_lds_sync();
            }
        }
        j0 = j1;
    }
    if (!FILL && lane < cnt) rowcnt[__float_as_uint(pos[first + lane].w)] = found;
}

__global__ __launch_bounds__(256) void k_unpack(const float4* __restrict__ pos, uint32_t n, float* __restrict__ xo,
                                                float* __restrict__ yo, float* __restrict__ zo) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const float4 p = pos[k];
    xo[k] = p.x;
    yo[k] = p.y;
    zo[k] = p.z;
}

template <int PRED>
void launch_force(int prec, bool vir, const Shape& sh, unsigned nb, hipStream_t s, const float4* pos,
                  const uint32_t* cell_of, const uint32_t* off, uint32_t n, const GridGeom& g, const Trim& tr,
                  const PairConst& c, float* fx, float* fy, float* fz, float* e, unsigned nforce, BlockSums* sums,
                  const SortedOut& so, float4* stage) {
    const size_t lds = sh.lds_bytes();
    const int out = stage ? 2 : non_temporal_outputs(n) ? 1 : 0;
    if (two_lanes(sh, n)) {
        // (`depth` has no effect: there is no queue)
#define LJ_L27N(PREC, VIR, LDS, AHEAD)                                                                                     \
    hipLaunchKernelGGL((k_force27<PRED, PREC, VIR, LDS, AHEAD>), dim3(nb), dim3(sh.block), 0, s, pos, cell_of, off, n, g, tr, c, \
                       fx, fy, fz, e, nforce, sums, so)
#define LJ_L27(PREC, VIR)                                     \
    do {                                                      \
        if (n <= kLdsParticles) LJ_L27N(PREC, VIR, true, true); \
        else if (n <= kAheadMax) LJ_L27N(PREC, VIR, false, true); \
        else LJ_L27N(PREC, VIR, false, false);                \
    } while (0)
        switch (prec) {
        case LJ_PREC_MIXED: if (vir) LJ_L27(LJ_PREC_MIXED, true); else LJ_L27(LJ_PREC_MIXED, false); break;
        case LJ_PREC_FP32: if (vir) LJ_L27(LJ_PREC_FP32, true); else LJ_L27(LJ_PREC_FP32, false); break;
        default: if (vir) LJ_L27(LJ_PREC_FP32_COMP, true); else LJ_L27(LJ_PREC_FP32_COMP, false); break;
        }
#undef LJ_L27
#undef LJ_L27N
        return;
    }
#define LJ_LAUNCH_QN(PREC, VIR, Q, OUT)                                                                              \
    hipLaunchKernelGGL((k_force<PRED, PREC, VIR, Q, OUT>), dim3(nb), dim3(sh.block), lds, s, pos, cell_of, off, n, g, \
                       sh.refine_x, sh.refine, tr, c, (uint32_t)sh.depth, fx, fy, fz, e, sums, so, stage)
#define LJ_LAUNCH_Q(PREC, VIR, Q)                      \
    do {                                               \
        if (out == 2) LJ_LAUNCH_QN(PREC, VIR, Q, 2);   \
        else if (out == 1) LJ_LAUNCH_QN(PREC, VIR, Q, 1); \
        else LJ_LAUNCH_QN(PREC, VIR, Q, 0);            \
    } while (0)
#define LJ_LAUNCH(PREC, VIR)                   \
    do {                                       \
        if (sh.queued()) LJ_LAUNCH_Q(PREC, VIR, true); \
        else LJ_LAUNCH_Q(PREC, VIR, false);    \
    } while (0)
    switch (prec) {
    case LJ_PREC_MIXED: if (vir) LJ_LAUNCH(LJ_PREC_MIXED, true); else LJ_LAUNCH(LJ_PREC_MIXED, false); break;
    case LJ_PREC_FP32: if (vir) LJ_LAUNCH(LJ_PREC_FP32, true); else LJ_LAUNCH(LJ_PREC_FP32, false); break;
    default: if (vir) LJ_LAUNCH(LJ_PREC_FP32_COMP, true); else LJ_LAUNCH(LJ_PREC_FP32_COMP, false); break;
    }
#undef LJ_LAUNCH
#undef LJ_LAUNCH_Q
#undef LJ_LAUNCH_QN
}

}  // namespace

void split_outputs(const float4* stage, uint32_t n, float* fx, float* fy, float* fz, float* e, hipStream_t s) {
    if (n == 0) return;
    hipLaunchKernelGGL(k_split_outputs, dim3(div_up(n, 256)), dim3(256), 0, s, stage, n, fx, fy, fz, e);
}

int grow_block_sums(lj_context* ctx, unsigned nblocks, BlockSums** out) {
    LJ_HIP(ctx, ctx->bin.partials.grow(((size_t)nblocks + nblocks / kFinalChunk + 1) * sizeof(BlockSums)));
    *out = ctx->bin.partials.as<BlockSums>();
    return LJ_OK;
}

int finalize_totals(lj_context* ctx, unsigned nblocks, const unsigned long long* cand, unsigned ncand,
                    const int* overflow, lj_result* res, hipStream_t s) {
    BlockSums* sums = ctx->bin.partials.as<BlockSums>();
    if (nblocks > kFinalOne) {
        // stage 1 writes behind the nblocks input sums (grow_block_sums left room)
        const unsigned chunks = (nblocks + kFinalChunk - 1) / kFinalChunk;
        BlockSums* tmp = sums + nblocks;
        hipLaunchKernelGGL(k_finalize, dim3(chunks), dim3(256), 0, s, (const BlockSums*)sums, (uint32_t)nblocks,
                           (const unsigned long long*)nullptr, 0u, (const int*)nullptr, tmp, (lj_result*)nullptr);
        sums = tmp;
        nblocks = chunks;
    }
    hipLaunchKernelGGL(k_finalize, dim3(1), dim3(1024), 0, s, (const BlockSums*)sums, (uint32_t)nblocks, cand, ncand,
                       overflow, (BlockSums*)nullptr, res);
    LJ_HIP(ctx, hipGetLastError());
    return LJ_OK;
}

// Scalar results live in the caller's lj_result or, when it is NULL, in a scratch one.
static int result_slot(lj_context* ctx, lj_result* user, lj_result** out) {
    if (user) {
        *out = user;
        return LJ_OK;
    }
    LJ_HIP(ctx, ctx->bin.counters.grow(sizeof(lj_result)));
    *out = ctx->bin.counters.as<lj_result>();
    return LJ_OK;
}

// Force grid of edge cw/Kx along x and cw/K along y and z (powers of two: exact),
// G' = (int)(L / edge) per axis.
int refine_geom(lj_context* ctx, const GridGeom& g, const lj_params* p, int Kx, int K, GridGeom* f) {
    *f = g;
    f->cw[0] = g.cw[0] / (float)Kx;
    f->cw[1] = g.cw[1] / (float)K;
    f->cw[2] = g.cw[2] / (float)K;
    uint64_t nc = 1;
    for (int d = 0; d < 3; ++d) {
        const float L = p->box_hi[d] - p->box_lo[d];
        const float q = L / f->cw[d];
        if (!(q < 16777216.0f)) return fail(ctx, LJ_ERR_OVERFLOW, "refined grid: more than 2^24 cells along one axis");
        int32_t gd = (int32_t)q;
        if (gd < 1) gd = 1;
        f->g[d] = gd;
        f->gmax[d] = (float)(gd - 1);
        nc *= (uint64_t)gd;
    }
    if (nc > 0x7fffffffull) return fail(ctx, LJ_ERR_OVERFLOW, "refined grid holds more than 2^31-1 cells");
    f->ncells = (uint32_t)nc;
    set_divisors(f);
    return LJ_OK;
}

// Shape of a call: explicit fields of p win.  Default grid: cells of rc/2 along y and
// z and rc/4 along x for large dense inputs (>= 8 particles per cell_edge cell and
// >= 2^22 particles, where fewer candidates pay for the larger key and cell arrays),
// the cell_edge grid otherwise (small inputs, and sparse ones whose extra empty cells
// cost more in the scan than they save; measured on MI355X at 0.1M-16.7M particles).
// The CUDALJ mode keeps the reference's 27 cells.  Block 256 and no queue.
Shape choose_shape(const lj_params* p, int64_t n, uint64_t ncells) {
    Shape sh;
    if (p->predicate == LJ_PRED_CUDALJ) {
        sh.refine = sh.refine_x = 1;
    } else {
        const double ppc = (double)n / (double)(ncells ? ncells : 1);
        const bool dense = ppc >= 8.0 && n >= ((int64_t)1 << 22) && (double)ncells * 16.0 < (double)(1u << 30);
        sh.refine = (p->refine == 1 || p->refine == 2 || p->refine == 4) ? p->refine : (dense ? 2 : 1);
        sh.refine_x = p->refine_x ? p->refine_x : (p->refine ? sh.refine : (dense ? 4 : 1));
        if (sh.refine_x < sh.refine) sh.refine_x = sh.refine;
    }
    sh.block = p->block ? p->block : 256;
    sh.depth = p->depth ? p->depth : 1;
    return sh;
}

Trim make_trim(const lj_params* p, const GridGeom& g) {
    Trim t;
    const double r = (double)p->rc * (1.0 + 0x1p-16);
    t.r2 = std::nextafter((float)(r * r), INFINITY);
    double mag = 0.0;
    for (int d = 0; d < 3; ++d) {
        mag = std::fmax(mag, std::fabs((double)p->box_lo[d]));
        mag = std::fmax(mag, std::fabs((double)p->box_hi[d]));
        t.hi[d] = p->box_hi[d];
    }
    // 2^-19 mag bounds the rounding of v - lo and (times the cell edge) the few ulp
    // by which (v - lo) inv_cw -+ w inv_cw and the cell coordinate (v - lo) / cw differ
    // from their exact values; the rc term covers the square root of the window
    const double cwmax = std::fmax((double)g.cw[0], std::fmax((double)g.cw[1], (double)g.cw[2]));
    t.margin = (float)(0x1p-19 * mag + (double)p->rc * 0x1p-14 + 8.0 * 0x1p-24 * cwmax);
    t.inv_cw = 1.0f / g.cw[0];
    t.on = p->predicate != LJ_PRED_CUDALJ;
    return t;
}

int compute_cellgrid(lj_context* ctx, const float* x, const float* y, const float* z, int64_t n, const lj_params* p,
                     const GridGeom& g, const PairConst& c, float* fx, float* fy, float* fz, float* e,
                     lj_result* result, hipStream_t s, const SortedOut& so) {
    const Shape sh = choose_shape(p, n, g.ncells);
    const bool refined = sh.refine > 1 || sh.refine_x > 1;
    GridGeom fg = g;
    if (refined) LJ_TRY(refine_geom(ctx, g, p, sh.refine_x, sh.refine, &fg));
    const Trim tr = make_trim(p, fg);
    {
        PhaseTimer t(ctx, LJ_PHASE_BIN, s);
        LJ_TRY(bin_particles(ctx, x, y, z, n, fg, s));
    }
    lj_result* res;
    LJ_TRY(result_slot(ctx, result, &res));
    // The candidate count, on the cell_edge grid (ComputeNbInteractions semantics), is
    // only made for a caller that takes the results: by further workgroups of the force
    // launch (two lanes a particle, count_beside_forces), else before it, on a refined grid
    // from cell_edge offsets of its own.
    const unsigned nforce = div_up((n > 0 ? n : 1) * (two_lanes(sh, n) ? kPairLanes : 1), sh.block);
    unsigned ncount = 0, nparts = 0;
    if (result && two_lanes(sh, n) && count_beside_forces(n, g.ncells)) {
        ncount = candidate_blocks(g);
    } else if (result && !refined) {
        PhaseTimer t(ctx, LJ_PHASE_OTHER, s);
        LJ_TRY(candidate_parts(ctx, g, ctx->bin.offsets.as<uint32_t>(), &nparts, s));
    } else if (result) {
        PhaseTimer t(ctx, LJ_PHASE_OTHER, s);
        BinWork& w = ctx->bin;
        LJ_HIP(ctx, w.ccounts.grow((size_t)g.ncells * 4));
        LJ_HIP(ctx, w.coffsets.grow(((size_t)g.ncells + 1) * 4));
        hipLaunchKernelGGL(k_coarse_counts, dim3(div_up(g.ncells, 256)), dim3(256), 0, s,
                           (const uint32_t*)w.offsets.as<uint32_t>(), fg, g, sh.refine_x, sh.refine,
                           w.ccounts.as<uint32_t>());
        uint32_t* coff = w.coffsets.as<uint32_t>();
        LJ_TRY(scan_u32(ctx, w.ccounts.as<uint32_t>(), coff, g.ncells, coff + g.ncells, s));
        LJ_TRY(candidate_parts(ctx, g, coff, &nparts, s));
    }
    const unsigned nb = nforce + ncount;
    BlockSums* sums;
    LJ_TRY(grow_block_sums(ctx, nb, &sums));
    const int prec = p->precision;
    const bool vir = !(p->flags & LJ_FLAG_NO_VIRIAL);
    const float4* pos = ctx->bin.pos.as<float4>();
    const uint32_t* cell_of = ctx->bin.sorted_keys();
    const uint32_t* off = ctx->bin.offsets.as<uint32_t>();
    const uint32_t nn = (uint32_t)n;
    // large outputs at shuffled indices go through the staging array
    float4* stage = nullptr;
    if (non_temporal_outputs(n) && !so.x) {
        LJ_HIP(ctx, ctx->bin.stage.grow((size_t)n * sizeof(float4)));
        stage = ctx->bin.stage.as<float4>();
    }
    {
        PhaseTimer tf(ctx, LJ_PHASE_FORCE, s);
#define LJ_PRED_CASE(P)                                                                                         \
    case P:                                                                                                     \
        launch_force<P>(prec, vir, sh, nb, s, pos, cell_of, off, nn, fg, tr, c, fx, fy, fz, e, nforce, sums, so, \
                        stage);                                                                                 \
        break;
        switch (p->predicate) {
            LJ_PRED_CASE(LJ_PRED_AABB)
            LJ_PRED_CASE(LJ_PRED_CUSTOM)
            LJ_PRED_CASE(LJ_PRED_CUDALJ)
            LJ_PRED_CASE(LJ_PRED_SPHERE)
            LJ_PRED_CASE(LJ_PRED_TRIANGLE)
        }
#undef LJ_PRED_CASE
    }
    PhaseTimer to(ctx, LJ_PHASE_OTHER, s);
    if (stage) split_outputs(stage, nn, fx, fy, fz, e, s);
    return finalize_totals(ctx, nb, ctx->bin.cand.as<unsigned long long>(), nparts, nullptr, res, s);
}

static void sort_long_rows(const unsigned long long* rows, int64_t n, uint32_t* cols, hipStream_t s) {
    if (n > 0)
        hipLaunchKernelGGL(k_sort_rows<true>, grid_of_blocks(div_up(n, kSortThreads)), dim3(kSortThreads), 0, s, rows, (uint32_t)n, cols,
                           (const uint32_t*)nullptr);
}

void sort_rows(const unsigned long long* rows, int64_t n, uint32_t* cols, const uint32_t* draft, hipStream_t s) {
    if (n > 0)
        hipLaunchKernelGGL(k_sort_rows<false>, grid_of_blocks(div_up(n, kBlockRows)), dim3(kSortThreads), 0, s, rows, (uint32_t)n, cols,
                           draft);
}

static int pairs_cellgrid(lj_context* ctx, const float* x, const float* y, const float* z, int64_t n,
                          const GridGeom& g, const PairConst& c, unsigned long long* rows, uint32_t* cols,
                          unsigned long long capacity, unsigned long long* needed, int predicate, hipStream_t s) {
    LJ_TRY(bin_particles(ctx, x, y, z, n, g, s));
    const unsigned nb = div_up(n > 0 ? n : 1, (kPairThreads / kWaveSize) * kPairSlots);
    const float4* pos = ctx->bin.pos.as<float4>();
    const uint32_t* cell_of = ctx->bin.sorted_keys();
    const uint32_t* off = ctx->bin.offsets.as<uint32_t>();
    const uint32_t nn = (uint32_t)n;
    // row counts (u32, by original index) -> u64 offsets
    LJ_HIP(ctx, ctx->bin.rows.grow(((size_t)n + 1) * sizeof(uint32_t)));
    uint32_t* rowcnt = ctx->bin.rows.as<uint32_t>();
#define LJ_PAIRS(P, FILL)                                                                                          \
    case P:                                                                                                        \
        hipLaunchKernelGGL((k_pairs<P, FILL>), grid_of_blocks(nb), dim3(kPairThreads), 0, s, pos, cell_of, off, nn, g, c, rowcnt, \
                           (const unsigned long long*)rows, cols);                                                 \
        break;
#define LJ_PAIRS_ALL(FILL)                                                                             \
    switch (predicate) {                                                                               \
        LJ_PAIRS(LJ_PRED_AABB, FILL)                                                                   \
        LJ_PAIRS(LJ_PRED_CUSTOM, FILL)                                                                 \
        LJ_PAIRS(LJ_PRED_CUDALJ, FILL)                                                                 \
        LJ_PAIRS(LJ_PRED_SPHERE, FILL)                                                                 \
        LJ_PAIRS(LJ_PRED_TRIANGLE, FILL)                                                               \
    }
    LJ_PAIRS_ALL(false)
    LJ_TRY(scan_u32_to_u64(ctx, rowcnt, rows, n, s));
    unsigned long long total = 0;
    LJ_HIP(ctx, hipMemcpyAsync(&total, rows + n, sizeof total, hipMemcpyDeviceToHost, s));
    LJ_HIP(ctx, hipStreamSynchronize(s));
    if (needed) *needed = total;
    if (total > capacity)
        return fail(ctx, LJ_ERR_CAPACITY, "pair list needs %llu entries, capacity is %llu", total, capacity);
    if (total == 0) return LJ_OK;
    LJ_PAIRS_ALL(true)
#undef LJ_PAIRS_ALL
#undef LJ_PAIRS
    sort_long_rows(rows, n, cols, s);  // the rows that k_pairs left unsorted
    LJ_HIP(ctx, hipGetLastError());
    return LJ_OK;
}

int unpack_sorted(lj_context* ctx, int64_t n, float* xo, float* yo, float* zo, hipStream_t s) {
    if (n > 0)
        hipLaunchKernelGGL(k_unpack, dim3(div_up(n, 256)), dim3(256), 0, s, ctx->bin.pos.as<float4>(), (uint32_t)n, xo,
                           yo, zo);
    LJ_HIP(ctx, hipGetLastError());
    return LJ_OK;
}

}  // namespace lj

using namespace lj;

extern "C" {

int lj_compute(lj_context* ctx, const float* x, const float* y, const float* z, int64_t n, const lj_params* p,
               float* fx, float* fy, float* fz, float* e, lj_result* result, void* stream) {
    if (!ctx) return LJ_ERR_INVALID_ARG;
    GridGeom g;
    PairConst c;
    LJ_TRY(make_geom(ctx, p, n, &g, &c));
    if (n > 0 && (!x || !y || !z || !fx || !fy || !fz))
        return fail(ctx, LJ_ERR_INVALID_ARG, "positions and forces must not be NULL");
    LJ_HIP(ctx, hipSetDevice(ctx->device));
    return compute_cellgrid(ctx, x, y, z, n, p, g, c, fx, fy, fz, e, result, (hipStream_t)stream);
}

int lj_compute_sorted(lj_context* ctx, float* x, float* y, float* z, int64_t n, const lj_params* p, float* fx,
                      float* fy, float* fz, float* e, uint32_t* perm, lj_result* result, void* stream) {
    if (!ctx) return LJ_ERR_INVALID_ARG;
    GridGeom g;
    PairConst c;
    LJ_TRY(make_geom(ctx, p, n, &g, &c));
    if (n > 0 && (!x || !y || !z || !fx || !fy || !fz))
        return fail(ctx, LJ_ERR_INVALID_ARG, "positions and forces must not be NULL");
    LJ_HIP(ctx, hipSetDevice(ctx->device));
    // the sort reads x, y, z before the force launch overwrites them
    SortedOut so;
    so.x = x;
    so.y = y;
    so.z = z;
    so.perm = perm;
    return compute_cellgrid(ctx, x, y, z, n, p, g, c, fx, fy, fz, e, result, (hipStream_t)stream, so);
}

int lj_pairs(lj_context* ctx, const float* x, const float* y, const float* z, int64_t n, const lj_params* p,
             unsigned long long* row_offsets, uint32_t* cols, unsigned long long capacity,
             unsigned long long* needed, void* stream) {
    if (!ctx) return LJ_ERR_INVALID_ARG;
    GridGeom g;
    PairConst c;
    LJ_TRY(make_geom(ctx, p, n, &g, &c));
    if (!row_offsets || (n > 0 && (!x || !y || !z)) || (capacity > 0 && !cols))
        return fail(ctx, LJ_ERR_INVALID_ARG, "NULL pointer argument");
    LJ_HIP(ctx, hipSetDevice(ctx->device));
    return pairs_cellgrid(ctx, x, y, z, n, g, c, row_offsets, cols, capacity, needed, p->predicate, (hipStream_t)stream);
}

int lj_reorder(lj_context* ctx, const float* x, const float* y, const float* z, int64_t n, const lj_params* p,
               float* xo, float* yo, float* zo, uint32_t* perm, void* stream) {
    if (!ctx) return LJ_ERR_INVALID_ARG;
    GridGeom g;
    PairConst c;
    LJ_TRY(make_geom(ctx, p, n, &g, &c));
    if (n > 0 && (!x || !y || !z || !xo || !yo || !zo))
        return fail(ctx, LJ_ERR_INVALID_ARG, "NULL pointer argument");
    LJ_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = (hipStream_t)stream;
    LJ_TRY(bin_particles(ctx, x, y, z, n, g, s));
    LJ_TRY(unpack_sorted(ctx, n, xo, yo, zo, s));
    if (perm) LJ_TRY(extract_perm(ctx, n, perm, s));
    return LJ_OK;
}

}  // extern "C"
