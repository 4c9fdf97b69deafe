// batch.hip -- many independent systems in one pipeline of launches.
//
// The reference runs one system per executeSimulation / core call (each with its own
// allocations, launches and host synchronisations, Cuda-version/cudaLJ.cu:515-677).
// Here the cell grids of all systems are concatenated into one key space: system s
// owns global cells [cell_base[s], cell_base[s+1]).  One histogram, one scan, one
// radix sort and one force launch then cover every system, whatever their sizes,
// and one more kernel reduces each system's totals in a fixed order.  Nothing in a
// steady-state call allocates or synchronises with the host, so the whole call can
// be captured in a hipGraph and replayed.
#include <cstring>
#include <vector>

#include "lj_candidates.h"
#include "lj_sort.h"
#include "lj_stencil27.h"

namespace lj {

namespace {

struct SysDesc {
    GridGeom g;   // force grid (edge cell_edge / refine); cells [cell_base, +g.ncells) of the key space
    GridGeom cg;  // cell_edge grid of the candidate count; cells [ccell_base, +cg.ncells)
    PairConst c;
    Trim tr;
    uint32_t first, n, cell_base, ccell_base;
};

// Largest s in [lo, hi) with base[s] <= v (base ascending, base[lo] <= v).
__device__ inline uint32_t find_sys_in(const uint32_t* __restrict__ base, uint32_t lo, uint32_t hi, uint32_t v) {
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (base[mid] <= v) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Search hints: hint[j] = the system of value j << kHintShift.  The system of v is
// monotone in v, so it lies between hint[v >> kHintShift] and the next entry: a search
// over one or two systems instead of all of them.  Table of (total >> kHintShift) + 2
// entries for values below `total`.
constexpr int kHintShift = 10;

__host__ __device__ inline size_t hint_entries(uint64_t total) { return (size_t)(total >> kHintShift) + 2; }

__global__ __launch_bounds__(256) void k_build_hints(const uint32_t* __restrict__ base, uint32_t nsys, uint32_t m,
                                                     uint32_t* __restrict__ hint) {
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= m) return;
    const uint64_t v = (uint64_t)j << kHintShift;
    hint[j] = find_sys_in(base, 0, nsys, v > 0xffffffffull ? 0xffffffffu : (uint32_t)v);
}

// Largest s with base[s] <= v, v below the table's total.
__device__ inline uint32_t find_sys(const uint32_t* __restrict__ base, const uint32_t* __restrict__ hint, uint32_t nsys,
                                    uint32_t v) {
    const uint32_t j = v >> kHintShift;
    const uint32_t lo = hint[j], up = hint[j + 1] + 1;
    return find_sys_in(base, lo, up < nsys ? up : nsys, v);
}

// Global cell key of particle i: its system's first cell plus the cell in that
// system's grid.
struct BatchKeyOp {
    const SysDesc* sys;
    const uint32_t* first;
    const uint32_t* hint;
    uint32_t nsys;
    __device__ uint32_t operator()(float x, float y, float z, uint32_t i) const {
        const SysDesc& d = sys[find_sys(first, hint, nsys, i)];
        return d.cell_base + cell_key(d.g, x, y, z);
    }
    __device__ bool skip() const { return false; }
};

// Particle counts of the cell_edge grids from the force grids' offsets (refine > 1).
__global__ __launch_bounds__(256) void k_batch_coarse_counts(const uint32_t* __restrict__ foff, uint32_t nccells,
                                                             const SysDesc* __restrict__ sys,
                                                             const uint32_t* __restrict__ ccbase,
                                                             const uint32_t* __restrict__ cchint, uint32_t nsys, int Kx,
                                                             int K, uint32_t* __restrict__ ccount) {
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nccells) return;
    const SysDesc& d = sys[find_sys(ccbase, cchint, nsys, c)];
    ccount[c] = coarse_count(foff + d.cell_base, d.g, d.cg, Kx, K, c - d.ccell_base);
}

// 27-cell candidates of the nh particles in global cell c of system d's cell_edge grid,
// from the offsets coff over the concatenated cell_edge cells (ComputeNbInteractions
// semantics, cudaLJ.cu:255-297).
__device__ inline unsigned long long cell_candidates(const uint32_t* __restrict__ coff, const SysDesc& d, uint32_t c,
                                                     uint32_t nh) {
    const GridGeom& g = d.cg;
    const uint32_t base = d.ccell_base;
    int32_t cx, cy, cz;
    cell_coords(g, c - base, cx, cy, cz);
    const int32_t gx = g.g[0], gy = g.g[1], gz = g.g[2];
    const int32_t x0 = cx > 0 ? cx - 1 : 0, x1 = cx < gx - 1 ? cx + 1 : gx - 1;
    // The nine rows' ranges loaded at once, with no branch between the loads: a row
    // outside the grid reads the cell's own row and counts zero.  (Loaded row by row
    // under the bounds tests, the loads went out one row at a time.)
    uint32_t lo[9], hi[9];
    bool in[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) {
        const int32_t zz = cz + q / 3 - 1, yy = cy + q % 3 - 1;
        in[q] = zz >= 0 && zz < gz && yy >= 0 && yy < gy;
        const uint32_t row = base + (uint32_t)(((in[q] ? zz : cz) * gy + (in[q] ? yy : cy)) * gx);
        lo[q] = coff[row + x0];
        hi[q] = coff[row + x1 + 1];
    }
    unsigned long long sum = 0;
#pragma unroll
    for (int q = 0; q < 9; ++q)
        if (in[q]) sum += hi[q] - lo[q];
    return nh ? (unsigned long long)nh * (sum - 1) : 0ull;
}

// The candidates of every system, added into cand[system].  A wave's cells usually belong
// to one system: it then adds its sum with one atomic.
__global__ __launch_bounds__(256) void k_batch_candidates(const uint32_t* __restrict__ coff, uint32_t nccells,
                                                          const SysDesc* __restrict__ sys,
                                                          const uint32_t* __restrict__ ccbase,
                                                          const uint32_t* __restrict__ cchint, uint32_t nsys,
                                                          unsigned long long* __restrict__ cand) {
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t s = 0xffffffffu;
    unsigned long long v = 0;
    if (c < nccells) {
        const uint32_t c0 = coff[c], c1 = coff[c + 1];  // on their way during the search
        s = find_sys(ccbase, cchint, nsys, c);
        v = cell_candidates(coff, sys[s], c, c1 - c0);
    }
    const uint32_t s0 = __shfl(s, 0, kWaveSize);
    if (__all(s == s0 || s == 0xffffffffu)) {
        v = wave_sum(v);
        if (__lane_id() == 0 && v) atomicAdd(&cand[s0], v);
    } else if (v) {
        atomicAdd(&cand[s], v);
    }
}

// Energy, virial and accepted pairs of the 64 sorted slots of one wave, when they all
// belong to system `sys`; sys = kSharedWave marks a wave whose slots belong to several
// systems (their values are then kept per slot).
struct WaveTotals {
    double e, v;
    unsigned long long np;
    uint32_t sys, pad;
};
constexpr uint32_t kSharedWave = 0xffffffffu;

// One thread per sorted slot, as the single-system kernel (the same stencil loop and
// LDS queues), with the grid, trimming and pair constants of the slot's system d:
// forces and energies to the caller's order, the slot's energy, virial and accepted
// pairs to ei, vi, np (zero for an idle lane).  Every lane of the wave calls it.
template <int PRED, int PREC, bool QUEUE>
__device__ inline void batch_pairs(const float4* __restrict__ pos, const uint32_t* __restrict__ off, uint32_t k,
                                   bool active, uint32_t key, const SysDesc& d, int Rx, int R, uint32_t depth,
                                   QEntry* __restrict__ queue, float* __restrict__ fx,
                                   float* __restrict__ fy, float* __restrict__ fz, float* __restrict__ e, double& ei,
                                   double& vi, uint32_t& np) {
    const GridGeom g = d.g;
    const PairConst c = d.c;
    const Trim tr = d.tr;
    const uint32_t base = d.cell_base;
    PairSums<PREC, PRED == LJ_PRED_CUDALJ, true> acc;
    const float4 pi = active ? pos[k] : make_float4(0.f, 0.f, 0.f, 0.f);
    acc.set_i(pi);
    acc.allow_exact_diff(c, pi, active);
    np = stencil_pairs<PRED, PREC, true, QUEUE>(pos, off, k, active, pi, g, base, key - base, Rx, R, tr, c, queue,
                                                depth, acc);
    ei = vi = 0.0;
    if (active) {
        const uint32_t i = __float_as_uint(pi.w);
        fx[i] = (float)(-c.e24 * (double)acc.ax.value());
        fy[i] = (float)(-c.e24 * (double)acc.ay.value());
        fz[i] = (float)(-c.e24 * (double)acc.az.value());
        ei = c.e4 * (double)acc.ae.value();
        if (e) e[i] = (float)ei;
        vi = c.e24 * (double)acc.av.value();
    }
}

// The waves whose 64 sorted slots belong to one system (nearly all of them): that
// system's constants are read once per wave (wave-uniform, so they sit in scalar
// registers, not in every lane), and the wave adds its energies, virials and pair
// counts (fixed butterfly order) into one WaveTotals.  A wave shared by several
// systems returns at once; k_batch_force_shared serves it.  A system's sorted slots are
// the caller's index range [first, first + n) of that system (the key space orders
// the systems).  Systems of at most `skip` particles are left out (k_batch_force27 takes
// them).
template <int PRED, int PREC, bool QUEUE>
__global__ __launch_bounds__(kMaxBlock) void k_batch_force(const float4* __restrict__ pos,
                                                           const uint32_t* __restrict__ cell_of,
                                                           const uint32_t* __restrict__ off, uint32_t n,
                                                           const SysDesc* __restrict__ sys,
                                                           const uint32_t* __restrict__ cbase,
                                                           const uint32_t* __restrict__ chint, uint32_t nsys, uint32_t skip,
                                                           int Rx, int R, uint32_t depth, float* __restrict__ fx,
                                                           float* __restrict__ fy, float* __restrict__ fz,
                                                           float* __restrict__ e, WaveTotals* __restrict__ wrec) {
    extern __shared__ QEntry queue[];
    const uint32_t k = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    const bool active = k < n;
    const uint32_t key = active ? cell_of[k] : 0u;
    const uint32_t si = find_sys(cbase, chint, nsys, key);
    // lane 0 holds the wave's lowest slot: idle only when the whole wave is
    const uint32_t s0 = __builtin_amdgcn_readfirstlane(active ? si : kSharedWave);
    if (s0 == kSharedWave || !__all(!active || si == s0) || (skip && sys[s0].n <= skip)) return;
    double ei, vi;
    uint32_t np;
    batch_pairs<PRED, PREC, QUEUE>(pos, off, k, active, key, sys[s0], Rx, R, depth,
                                   queue + (threadIdx.x / kWaveSize) * depth * kWaveSize + __lane_id(), fx,
                                   fy, fz, e, ei, vi, np);
    const double es = wave_sum(ei), vs = wave_sum(vi);
    const unsigned long long ns = wave_sum((unsigned long long)np);
    if (__lane_id() == 0) wrec[k / kWaveSize] = WaveTotals{es, vs, ns, s0, 0u};
}

// The waves shared by several systems (listed in the plan; at most one per system
// boundary), one per workgroup: each lane reads its own system's constants, and the
// slots' energies, virials and pair counts are kept per slot.
template <int PRED, int PREC, bool QUEUE>
__global__ __launch_bounds__(kWaveSize) void k_batch_force_shared(
    const float4* __restrict__ pos, const uint32_t* __restrict__ cell_of, const uint32_t* __restrict__ off, uint32_t n,
    const SysDesc* __restrict__ sys, const uint32_t* __restrict__ cbase, const uint32_t* __restrict__ chint,
    uint32_t nsys, uint32_t skip, const uint32_t* __restrict__ shared_waves, int Rx, int R, uint32_t depth,
    float* __restrict__ fx,
    float* __restrict__ fy, float* __restrict__ fz, float* __restrict__ e, double2* __restrict__ ev,
    uint32_t* __restrict__ npair, WaveTotals* __restrict__ wrec) {
    extern __shared__ QEntry queue[];
    const uint32_t w = shared_waves[blockIdx.x];
    const uint32_t k = w * kWaveSize + threadIdx.x;
    const uint32_t key = k < n ? cell_of[k] : 0u;
    const SysDesc& d = sys[find_sys(cbase, chint, nsys, key)];
    const bool active = k < n && d.n > skip;
    double ei, vi;
    uint32_t np;
    batch_pairs<PRED, PREC, QUEUE>(pos, off, k, active, key, d, Rx, R, depth,
                                   queue + (threadIdx.x / kWaveSize) * depth * kWaveSize + __lane_id(), fx, fy, fz, e,
                                   ei, vi, np);
    if (active) {
        ev[k] = make_double2(ei, vi);
        npair[k] = np;
    }
    if (threadIdx.x == 0) wrec[w] = WaveTotals{0.0, 0.0, 0ull, kSharedWave, 0u};
}

// The systems that two_lanes takes (at most `most` particles): two lanes per particle, 32
// sorted slots per wave.  A wave takes one system, its constants in scalar registers: the
// first nmain workgroups' waves the system of their first slot, and further waves, listed
// in the plan as (wave, system), the systems that begin inside a wave; those waves keep
// their values per slot, as the waves of k_batch_force_shared do.  (One wave that took its
// systems one after the other kept more alive across them than its 64 registers hold.)
constexpr uint32_t kWaveSlots27 = kWaveSize / kPairLanes;
// Threads of a workgroup where the caller names none and the call fills the chip; us, 256 ->
// 128 threads (why the middle size wins was not found out): 32 systems of 65,536 particles on spheres 647 -> 565, 28 of 450,000 of 20 neighbours 2,632 ->
// 2,476, 13 of a million 2,997 -> 2,786, 25.5M in systems of 2,000-60,000 6,321 -> 6,283; with
// 64 threads 631, 2,674, 3,020 and 6,270.  Up to kAheadMax particles 256 are level or ahead.
constexpr unsigned kBlock27 = 128;

template <int PRED, int PREC, bool AHEAD>
__global__ __launch_bounds__(kMaxBlock, AHEAD ? 4 : 8) void k_batch_force27(
    const float4* __restrict__ pos, const uint32_t* __restrict__ cell_of, const uint32_t* __restrict__ off, uint32_t n,
    const SysDesc* __restrict__ sys, const uint32_t* __restrict__ cbase, const uint32_t* __restrict__ chint,
    uint32_t nsys, uint32_t most, uint32_t nmain, const uint2* __restrict__ extra, uint32_t nextra,
    float* __restrict__ fx, float* __restrict__ fy, float* __restrict__ fz, float* __restrict__ e,
    double2* __restrict__ ev, uint32_t* __restrict__ npair, WaveTotals* __restrict__ wrec) {
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize), waves = blockDim.x / kWaveSize;
    uint32_t w, s0;  // wave-uniform
    const uint32_t blk = block_index();
    if (blk < nmain) {
        w = xcd_block(blk, nmain) * waves + wave;
        if (w * kWaveSlots27 >= n) return;
        s0 = find_sys(cbase, chint, nsys, cell_of[w * kWaveSlots27]);
    } else {
        const uint32_t q = (blk - nmain) * waves + wave;
        if (q >= nextra) return;
        w = extra[q].x;
        s0 = extra[q].y;
    }
    const SysDesc& d = sys[s0];
    if (d.n > most) return;
    const uint32_t k = w * kWaveSlots27 + __lane_id() / kPairLanes;
    // a system's sorted slots are its caller range
    const bool mine = k >= d.first && k - d.first < d.n;
    const bool whole = __all(mine || k >= n);
    const float4 pi = mine ? pos[k] : make_float4(0.f, 0.f, 0.f, 0.f);
    const uint32_t key = mine ? cell_of[k] - d.cell_base : 0u;
    const PairConst c = d.c;
    PairSums<PREC, PRED == LJ_PRED_CUDALJ, true> acc;
    acc.set_i(pi);
    acc.allow_exact_diff(c, pi, mine);
    const uint32_t np = stencil27<PRED, AHEAD>(pos, off, k, mine, pi, d.g, d.cell_base, key, d.tr, c, acc);
    acc.template merge<kPairLanes>();
    const bool first = mine && (__lane_id() & 1u) == 0u;
    double ei = 0.0, vi = 0.0;
    if (first) {
        const uint32_t i = __float_as_uint(pos[k].w);
        fx[i] = (float)(-c.e24 * (double)acc.ax.value());
        fy[i] = (float)(-c.e24 * (double)acc.ay.value());
        fz[i] = (float)(-c.e24 * (double)acc.az.value());
        ei = c.e4 * (double)acc.ae.value();
        if (e) e[i] = (float)ei;
        vi = c.e24 * (double)acc.av.value();
    }
    if (whole) {
        // (a system of at most 2^20 particles: 64 lanes' pairs fit 32 bits)
        const double es = wave_sum(ei), vs = wave_sum(vi);
        const uint32_t ns = wave_sum(np);
        if (__lane_id() == 0) wrec[w] = WaveTotals{es, vs, ns, s0, 0u};
    } else {
        const uint32_t both = np + dpp_of<1>(np);
        if (first) {
            ev[k] = make_double2(ei, vi);
            npair[k] = both;
        }
        if (__lane_id() == 0) wrec[w].sys = kSharedWave;
    }
}

// One block per system: FP64 totals over its waves in slot order -- the WaveTotals of
// the waves it fills alone, the per-slot values of its slots in the (at most two)
// waves it shares with other systems -- and its candidate count, from cand or, when cand
// is NULL, counted here from the offsets coff (count_in_reduction: one
// launch less, and no second stream to fork and join, which took 20 us).
// wrec27: the records of the systems of at most `most` particles.
__global__ __launch_bounds__(256) void k_batch_reduce(const SysDesc* __restrict__ sys,
                                                      const WaveTotals* __restrict__ wrec1,
                                                      const WaveTotals* __restrict__ wrec27, uint32_t most,
                                                      const double2* __restrict__ ev,
                                                      const uint32_t* __restrict__ npair,
                                                      const unsigned long long* __restrict__ cand,
                                                      const uint32_t* __restrict__ coff, lj_result* __restrict__ res) {
    const SysDesc& d = sys[blockIdx.x];
    const bool two = d.n <= most;
    const uint32_t slots = two ? kWaveSlots27 : (uint32_t)kWaveSize;  // of a record
    const WaveTotals* const wrec = two ? wrec27 : wrec1;
    double a = 0.0, b = 0.0;
    unsigned long long np = 0, nc = 0;
    if (d.n) {
        const uint32_t w0 = d.first / slots, w1 = (d.first + d.n - 1) / slots;
        for (uint32_t w = w0 + threadIdx.x; w <= w1; w += 256) {
            const WaveTotals r = wrec[w];
            if (r.sys != kSharedWave) {
                a += r.e;
                b += r.v;
                np += r.np;
            } else {
                const uint32_t lo = d.first > w * slots ? d.first : w * slots;
                const uint32_t hi = d.first + d.n < (w + 1) * slots ? d.first + d.n : (w + 1) * slots;
                for (uint32_t q = lo; q < hi; ++q) {
                    const double2 t = ev[q];
                    a += t.x;
                    b += t.y;
                    np += npair[q];
                }
            }
        }
        if (!cand)
            for (uint32_t c = d.ccell_base + threadIdx.x; c < d.ccell_base + d.cg.ncells; c += 256)
                nc += cell_candidates(coff, d, c, coff[c + 1] - coff[c]);
    }
    __shared__ BlockSums total;
    store_block_sums<true, true>(&total, a, b, np, nc);
    if (threadIdx.x == 0)
        res[blockIdx.x] = lj_result{0.5 * total.e, 0.5 * total.v, cand ? cand[blockIdx.x] : total.nc, total.np};
}

}  // namespace

}  // namespace lj

using namespace lj;

extern "C" int lj_compute_batched(lj_context* ctx, const lj_system* sys, int32_t nsys, const float* x, const float* y,
                                  const float* z, float* fx, float* fy, float* fz, float* e, lj_result* results,
                                  void* stream) {
    if (!ctx) return LJ_ERR_INVALID_ARG;
    if (nsys < 0 || (nsys > 0 && (!sys || !results))) return fail(ctx, LJ_ERR_INVALID_ARG, "bad system array");
    if (nsys == 0) return LJ_OK;
    // Plan: per-system geometry, contiguous particle ranges, concatenated cells.
    std::vector<SysDesc> desc((size_t)nsys);
    std::vector<uint32_t> first((size_t)nsys), cbase((size_t)nsys), ccbase((size_t)nsys);
    uint64_t ntot = 0, ctot = 0, cctot = 0;
    uint32_t most_cells = 0;  // of one system, on the cell_edge grid
    const lj_params& p0 = sys[0].params;
    for (int32_t s = 0; s < nsys; ++s) {
        const lj_params& ps = sys[s].params;
        GridGeom g;
        PairConst c;
        LJ_TRY(make_geom(ctx, &ps, sys[s].n, &g, &c));
        if (ps.predicate != p0.predicate || ps.precision != p0.precision)
            return fail(ctx, LJ_ERR_INVALID_ARG, "all systems of a batch must share predicate and precision");
        if (ps.refine != p0.refine || ps.refine_x != p0.refine_x || ps.block != p0.block || ps.depth != p0.depth)
            return fail(ctx, LJ_ERR_INVALID_ARG, "all systems of a batch must share refine, refine_x, block and depth");
        if (sys[s].first != (int64_t)ntot)
            return fail(ctx, LJ_ERR_INVALID_ARG, "system %d starts at %lld; systems must be packed back to back from 0",
                        s, (long long)sys[s].first);
        SysDesc& d = desc[(size_t)s];
        std::memset(&d, 0, sizeof d);
        d.g = g;
        d.cg = g;
        d.c = c;
        d.first = (uint32_t)ntot;
        d.n = (uint32_t)sys[s].n;
        d.ccell_base = (uint32_t)cctot;
        ntot += (uint64_t)sys[s].n;
        cctot += g.ncells;
        most_cells = g.ncells > most_cells ? g.ncells : most_cells;
        if (ntot > 0x7fffffffull) return fail(ctx, LJ_ERR_OVERFLOW, "batch holds more than 2^31-1 particles");
        if (cctot > 0x7fffffffull) return fail(ctx, LJ_ERR_OVERFLOW, "batch holds more than 2^31-1 cells");
    }
    // One shape for the batch: the default refinement from the mean occupancy.
    const Shape sh = choose_shape(&p0, (int64_t)ntot, cctot);
    for (int32_t s = 0; s < nsys; ++s) {
        SysDesc& d = desc[(size_t)s];
        if (sh.refine > 1 || sh.refine_x > 1)
            LJ_TRY(refine_geom(ctx, d.cg, &sys[s].params, sh.refine_x, sh.refine, &d.g));
        d.tr = make_trim(&sys[s].params, d.g);
        d.cell_base = (uint32_t)ctot;
        ctot += d.g.ncells;
        if (ctot > 0x7fffffffull) return fail(ctx, LJ_ERR_OVERFLOW, "batch holds more than 2^31-1 force-grid cells");
        first[(size_t)s] = d.first;
        cbase[(size_t)s] = d.cell_base;
        ccbase[(size_t)s] = d.ccell_base;
    }
    if (ntot > 0 && (!x || !y || !z || !fx || !fy || !fz))
        return fail(ctx, LJ_ERR_INVALID_ARG, "positions and forces must not be NULL");
    // waves of 64 sorted slots holding slots of more than one system: the wave of each
    // boundary between non-empty systems that does not fall on a wave boundary
    std::vector<uint32_t> shared;
    {
        bool seen = false;
        for (int32_t s = 0; s < nsys; ++s) {
            if (!desc[(size_t)s].n) continue;
            const uint32_t f = desc[(size_t)s].first;
            if (seen && f % (uint32_t)kWaveSize && (shared.empty() || shared.back() != f / (uint32_t)kWaveSize))
                shared.push_back(f / (uint32_t)kWaveSize);
            seen = true;
        }
    }
    // two lanes a particle: the systems that begin inside a wave of 32 slots, as (wave, system)
    std::vector<uint32_t> extra;
    for (int32_t q = 0; q < nsys; ++q) {
        const SysDesc& d = desc[(size_t)q];
        if (d.n && d.first % kWaveSlots27 && two_lanes(sh, d.n)) {
            extra.push_back(d.first / kWaveSlots27);
            extra.push_back((uint32_t)q);
        }
    }
    LJ_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = (hipStream_t)stream;
    BatchWork& W = ctx->batch;
    BinWork& B = ctx->bin;

    // Upload the plan only when it changed (a cached plan keeps replays free of
    // host-to-device copies).
    const size_t dbytes = desc.size() * sizeof(SysDesc), ubytes = (size_t)nsys * 4;
    // (the pairs of `extra` come right after the descriptors, 8-byte aligned)
    const size_t sbytes = shared.size() * 4, xbytes = extra.size() * 4;
    static_assert(sizeof(SysDesc) % 8 == 0, "the pairs after the descriptors are 8-byte aligned");
    std::vector<uint8_t> blob(dbytes + xbytes + 3 * ubytes + sbytes);
    std::memcpy(blob.data(), desc.data(), dbytes);
    if (xbytes) std::memcpy(blob.data() + dbytes, extra.data(), xbytes);
    const size_t ubase = dbytes + xbytes;
    std::memcpy(blob.data() + ubase, first.data(), ubytes);
    std::memcpy(blob.data() + ubase + ubytes, cbase.data(), ubytes);
    std::memcpy(blob.data() + ubase + 2 * ubytes, ccbase.data(), ubytes);
    if (sbytes) std::memcpy(blob.data() + ubase + 3 * ubytes, shared.data(), sbytes);
    const SysDesc* dsys = nullptr;
    const uint2* dextra = nullptr;
    const uint32_t *dfirst = nullptr, *dcbase = nullptr, *dccbase = nullptr, *dshared = nullptr;
    // search hints of the three base arrays (particles, force-grid cells, cell_edge cells)
    const size_t h1 = hint_entries(ntot), h2 = hint_entries(ctot), h3 = hint_entries(cctot);
    auto bind = [&]() {
        dsys = W.sys.as<SysDesc>();
        const uint8_t* dplan = W.sys.as<uint8_t>();
        dextra = reinterpret_cast<const uint2*>(dplan + dbytes);
        dfirst = reinterpret_cast<const uint32_t*>(dplan + ubase);
        dcbase = reinterpret_cast<const uint32_t*>(dplan + ubase + ubytes);
        dccbase = reinterpret_cast<const uint32_t*>(dplan + ubase + 2 * ubytes);
        dshared = reinterpret_cast<const uint32_t*>(dplan + ubase + 3 * ubytes);
    };
    if (blob != W.plan) {
        LJ_HIP(ctx, W.sys.grow(blob.size()));
        LJ_HIP(ctx, W.hints.grow((h1 + h2 + h3) * sizeof(uint32_t)));
        LJ_HIP(ctx, hipMemcpyAsync(W.sys.ptr, blob.data(), blob.size(), hipMemcpyHostToDevice, s));
        bind();
        uint32_t* hw = W.hints.as<uint32_t>();
        const uint32_t* bases[3] = {dfirst, dcbase, dccbase};
        const size_t sizes[3] = {h1, h2, h3};
        for (int t = 0; t < 3; ++t) {
            hipLaunchKernelGGL(k_build_hints, dim3(div_up((int64_t)sizes[t], 256)), dim3(256), 0, s, bases[t],
                               (uint32_t)nsys, (uint32_t)sizes[t], hw);
            hw += sizes[t];
        }
        LJ_HIP(ctx, hipGetLastError());
        LJ_HIP(ctx, hipStreamSynchronize(s));
        W.plan = std::move(blob);
    }
    bind();
    const uint32_t* hfirst = W.hints.as<uint32_t>();
    const uint32_t* hcbase = hfirst + h1;
    const uint32_t* hccbase = hcbase + h2;

    const int64_t n = (int64_t)ntot;
    const uint32_t ncells = (uint32_t)ctot, nccells = (uint32_t)cctot;
    const size_t nn = (size_t)(n > 0 ? n : 1);
    LJ_HIP(ctx, W.ev.grow(nn * sizeof(double2)));
    LJ_HIP(ctx, W.npair.grow(nn * sizeof(uint32_t)));
    // which systems take two lanes a particle, and the records of each kind of wave
    bool any_one = false, any_two = false;
    for (int32_t q = 0; q < nsys; ++q) {
        if (!sys[q].n) continue;
        (two_lanes(sh, sys[q].n) ? any_two : any_one) = true;
    }
    const uint32_t most = two_lanes(sh, 0) ? (uint32_t)kTwoLaneMax : 0u;
    const size_t nrec = div_up((int64_t)nn, kWaveSize);
    LJ_HIP(ctx, W.wrec.grow((nrec + div_up((int64_t)nn, kWaveSlots27)) * sizeof(WaveTotals)));
    uint32_t* off;
    {
        PhaseTimer tb(ctx, LJ_PHASE_BIN, s);
        int bits = 0;
        while (bits < 32 && ((uint64_t)1 << bits) < (uint64_t)ncells) ++bits;
        uint32_t* ngaps = nullptr;
        LJ_TRY(gap_list(ctx, ncells, &ngaps));
        LJ_TRY(sort_particles(ctx, x, y, z, n, BatchKeyOp{dsys, dfirst, hfirst, (uint32_t)nsys}, bits, s, ngaps));
        LJ_TRY(cell_offsets_from_sorted(ctx, n, ncells, s));
        off = B.offsets.as<uint32_t>();
    }
    // The candidate counts need only the cell offsets: they run on the context's second
    // stream beside the force pass, into an array of their own that the final
    // reduction copies into the results after the join.
    // Small systems in small batches whose cell_edge cells are the force grid's count in the reduction.
    const bool fork = sh.refine > 1 || sh.refine_x > 1 || !count_in_reduction(cctot, most_cells);
    unsigned long long* cand = nullptr;
    if (fork) {
        LJ_HIP(ctx, W.cand.grow((size_t)nsys * sizeof(unsigned long long)));
        cand = W.cand.as<unsigned long long>();
        const hipStream_t sc = ctx->aux;
        LJ_HIP(ctx, hipEventRecord(ctx->ev_fork, s));
        LJ_HIP(ctx, hipStreamWaitEvent(sc, ctx->ev_fork, 0));
        fill_u64(cand, (uint32_t)nsys, 0ull, sc);
        const uint32_t* coff = off;
        if (sh.refine > 1 || sh.refine_x > 1) {
            LJ_HIP(ctx, B.ccounts.grow((size_t)nccells * 4));
            LJ_HIP(ctx, B.coffsets.grow(((size_t)nccells + 1) * 4));
            hipLaunchKernelGGL(k_batch_coarse_counts, dim3(div_up(nccells, 256)), dim3(256), 0, sc,
                               (const uint32_t*)off, nccells, dsys, dccbase, hccbase, (uint32_t)nsys, sh.refine_x,
                               sh.refine, B.ccounts.as<uint32_t>());
            uint32_t* co = B.coffsets.as<uint32_t>();
            LJ_TRY(scan_u32(ctx, B.ccounts.as<uint32_t>(), co, nccells, co + nccells, sc));
            coff = co;
        }
        hipLaunchKernelGGL(k_batch_candidates, dim3(div_up(nccells, 256)), dim3(256), 0, sc, coff, nccells, dsys,
                           dccbase, hccbase, (uint32_t)nsys, cand);
        LJ_HIP(ctx, hipEventRecord(ctx->ev_join, sc));
    }
    double2* ev = W.ev.as<double2>();
    uint32_t* npair = W.npair.as<uint32_t>();
    WaveTotals* wrec = W.wrec.as<WaveTotals>();
    WaveTotals* wrec27 = wrec + nrec;
    const float4* pos = B.pos.as<float4>();
    const uint32_t* cell_of = B.sorted_keys();
    {
        PhaseTimer tf(ctx, LJ_PHASE_FORCE, s);
        const unsigned block27 = p0.block || n <= kAheadMax ? (unsigned)sh.block : kBlock27;
        const unsigned nb = div_up(n, sh.block), nb27 = div_up(n * kPairLanes, block27);
        const unsigned nextra = (unsigned)(extra.size() / 2), nx27 = div_up((int64_t)nextra * kWaveSize, block27);
        const size_t lds = sh.lds_bytes();
        const size_t lds_shared = sh.queued() ? (size_t)sh.depth * kWaveSize * sizeof(QEntry) : 0;
        if (n > 0) {
#define LJ_BFQ(PRED, PREC, Q)                                                                                     \
    do {                                                                                                          \
        hipLaunchKernelGGL((k_batch_force<PRED, PREC, Q>), dim3(nb), dim3(sh.block), lds, s, pos, cell_of,        \
                           (const uint32_t*)off, (uint32_t)n, dsys, dcbase, hcbase, (uint32_t)nsys, most, sh.refine_x, \
                           sh.refine, (uint32_t)sh.depth, fx, fy, fz, e, wrec);                                     \
        if (!shared.empty())                                                                                      \
            hipLaunchKernelGGL((k_batch_force_shared<PRED, PREC, Q>), dim3((unsigned)shared.size()),              \
                               dim3(kWaveSize), lds_shared, s, pos, cell_of, (const uint32_t*)off, (uint32_t)n,    \
                               dsys, dcbase, hcbase, (uint32_t)nsys, most, dshared, sh.refine_x, sh.refine,        \
                               (uint32_t)sh.depth, fx, fy, fz, e, ev, npair, wrec);                                 \
    } while (0)
#define LJ_BF27(PRED, PREC, AHEAD)                                                                                  \
    hipLaunchKernelGGL((k_batch_force27<PRED, PREC, AHEAD>), grid_of_blocks(nb27 + nx27), dim3(block27), 0, s, pos, cell_of,  \
                       (const uint32_t*)off, (uint32_t)n, dsys, dcbase, hcbase, (uint32_t)nsys, most, nb27, dextra,  \
                       nextra, fx, fy, fz, e, ev, npair, wrec27)
#define LJ_BF(PRED, PREC)                                                                                          \
    do {                                                                                                           \
        if (any_two && n <= kAheadMax) LJ_BF27(PRED, PREC, true);                                                  \
        else if (any_two) LJ_BF27(PRED, PREC, false);                                                              \
        if (any_one) {                                                                                             \
            if (sh.queued()) LJ_BFQ(PRED, PREC, true);                                                             \
            else LJ_BFQ(PRED, PREC, false);                                                                        \
        }                                                                                                          \
    } while (0)
#define LJ_BF_PREC(PRED)                                   \
    switch (p0.precision) {                                \
    case LJ_PREC_MIXED: LJ_BF(PRED, LJ_PREC_MIXED); break; \
    case LJ_PREC_FP32: LJ_BF(PRED, LJ_PREC_FP32); break;   \
    default: LJ_BF(PRED, LJ_PREC_FP32_COMP); break;        \
    }
            switch (p0.predicate) {
            case LJ_PRED_AABB: LJ_BF_PREC(LJ_PRED_AABB); break;
            case LJ_PRED_CUSTOM: LJ_BF_PREC(LJ_PRED_CUSTOM); break;
            case LJ_PRED_CUDALJ: LJ_BF_PREC(LJ_PRED_CUDALJ); break;
            case LJ_PRED_SPHERE: LJ_BF_PREC(LJ_PRED_SPHERE); break;
            case LJ_PRED_TRIANGLE: LJ_BF_PREC(LJ_PRED_TRIANGLE); break;
            }
#undef LJ_BF_PREC
#undef LJ_BF
#undef LJ_BF27
#undef LJ_BFQ
        }
    }
    {
        PhaseTimer to(ctx, LJ_PHASE_OTHER, s);
        if (fork) LJ_HIP(ctx, hipStreamWaitEvent(s, ctx->ev_join, 0));
        hipLaunchKernelGGL(k_batch_reduce, dim3((unsigned)nsys), dim3(256), 0, s, dsys, (const WaveTotals*)wrec,
                           (const WaveTotals*)wrec27, most, (const double2*)ev, (const uint32_t*)npair,
                           (const unsigned long long*)cand, (const uint32_t*)off, results);
    }
    LJ_HIP(ctx, hipGetLastError());
    return LJ_OK;
}
