// lj_stencil27.h -- the pair loop of the cell_edge grid's 27 cells: two lanes a particle.
//
// Reference: ComputeParticleInterationsParPartNoLoop (Cuda-version/cudaLJ.cu:299-341)
// gives each particle one thread, and so does stencil_pairs (lj_stencil.h), which takes the
// refined grids.
#pragma once

#include "lj_stencil.h"

namespace lj {

constexpr int kPairLanes = 2;
// The two lanes' sums are added at the end, so the two forms differ in the last bits of
// the 64-bit sums: which one a system takes follows from the system alone (and the shape),
// never from what else is in the call, and lj_compute, lj_compute_sorted,
// lj_compute_noalloc and lj_compute_batched agree bit for bit.  Up to 2^20 particles
// (lj_compute, us, one lane -> two): 100,000 of 27 neighbours 98 -> 66, 1,000,000 of 70 446 ->
// 408, on a sphere 278 -> 241; at 3,000,001 uniform of 45 867 -> 851, on a sphere 670 -> 722.
// In batches that fill the chip: 25.5M particles in systems of 2,000-60,000 of 40 and 70
// neighbours 6,419 -> 6,270 and 9,401 -> 9,172, 28 systems of 450,000 of 40 3,288 -> 3,225, 13
// of a million of 40 3,479 -> 3,518.
constexpr int64_t kTwoLaneMax = (int64_t)1 << 20;
// Calls of up to this many particles in all load a step ahead (about four waves a SIMD):
// us without -> with, 30,000 particles of 70 partners 74 -> 66, 65,000 92 -> 83, clustered
// 30,000 185 -> 171; level at 140,000 (112, 113); at 300,000 172 -> 177, since the registers
// leave fewer waves a SIMD.
constexpr int64_t kAheadMax = 140000;
inline bool two_lanes(const Shape& sh, int64_t n) { return sh.refine == 1 && sh.refine_x == 1 && n <= kTwoLaneMax; }
// Whether the candidate count of a call with two lanes a particle goes into further
// workgroups of the force launch, which saves a launch (4-7 us), or into a kernel of its own.
// Where the force kernel's registers leave four waves a SIMD, those workgroups walk a large
// grid at that occupancy too: lj_compute of 1,000 and 100,000 particles, us, in the force
// launch and by itself, in 160^3 cells 68 and 67, 114 and 119, in 256^3 97 and 86, 169 and
// 168, in 640^3 878 and 646, 791 and 744; 500,000 particles, eight waves a SIMD, 1,156 and
// 1,174 there.
constexpr uint32_t kCountCells = 1u << 23;
inline bool count_beside_forces(int64_t n, uint32_t ncells) { return n > kAheadMax || ncells <= kCountCells; }
static_assert((kCandidates - 1) * kPairLanes <= kPosSpare, "unclamped candidate loads need spare slots");

// The value of the even (or odd) lane of each pair of neighbouring lanes.
__device__ inline uint32_t of_even(uint32_t v) {
    return from_lane<0xA0>(v);  // quad_perm [0,0,2,2]
}
__device__ inline uint32_t of_odd(uint32_t v) {
    return from_lane<0xF5>(v);  // quad_perm [1,1,3,3]
}

// Accepted partners of the particle in sorted slot k (position pi, cell `key` of the
// cell_edge grid g, whose cell 0 is global cell `cbase`), given to acc.add by two
// neighbouring lanes; returns the lane's number of pairs, acc holds the lane's sums.
// The nine x-rows of the 27 cells are the particle's own and four mirror pairs, (dz, dy)
// and (-dz, -dy): the even lane finds the trimmed slot range (see stencil_pairs) of its
// own row and of one row of each pair, the odd lane those of the mirror rows, all ten
// loads at once; then the two take every second candidate of each pair of rows, walked as
// one stream.  Every lane of the wave calls this (idle ones with active = false).  pos may
// be a copy in LDS.
// AHEAD: the next iteration's candidates are loaded before this one's are tested, for calls
// that leave a SIMD a few waves to hide the loads behind (kAheadMax).
// One lane a particle (stencil_pairs) leaves most of the chip's lanes empty below 500,000
// particles and walks for twice as long; two lanes there take (lj_compute, us, one -> two
// lanes): 1,000 particles 90 -> 42 (from a copy in LDS), 100,000 of 27 partners 98 -> 66, of 70 135 -> 98,
// 300,000 clustered 248 -> 190, 131,073 CUDALJ 137 -> 87.  Splitting the rows over the lanes
// instead, or four and eight lanes, gained less at 100,000 and cost 10-50 % at a million.
template <int PRED, bool AHEAD, bool LIMITS = true, class Sink>
__device__ inline uint32_t stencil27(const float4* pos, const uint32_t* __restrict__ off, uint32_t k,
                                     bool active, const float4& pi, const GridGeom& g, uint32_t cbase, uint32_t key,
                                     const Trim& tr, const PairConst& c, Sink& acc) {
    constexpr int kSets = 5;  // the own row and four mirror pairs
    const uint32_t sub = __lane_id() & 1u;
    const int32_t sg = sub ? -1 : 1;
    int32_t cx = 0, cy = 0, cz = 0;
    cell_coords(g, key, cx, cy, cz);
    const bool trim = tr.on && pi.x >= g.lo[0] && pi.y >= g.lo[1] && pi.z >= g.lo[2] && pi.x <= tr.hi[0] &&
                      pi.y <= tr.hi[1] && pi.z <= tr.hi[2];
    // squared gaps to the rows one cell away, towards and against the lane's direction
    float gz = 0.f, gyp = 0.f, gym = 0.f;
    if (trim) {
        const float ylo = pi.y - (g.lo[1] + (float)cy * g.cw[1]), yhi = (g.lo[1] + (float)(cy + 1) * g.cw[1]) - pi.y;
        const float zlo = pi.z - (g.lo[2] + (float)cz * g.cw[2]), zhi = (g.lo[2] + (float)(cz + 1) * g.cw[2]) - pi.z;
        gz = fmaxf((sub ? zlo : zhi) - tr.margin, 0.f);
        gyp = fmaxf((sub ? ylo : yhi) - tr.margin, 0.f);
        gym = fmaxf((sub ? yhi : ylo) - tr.margin, 0.f);
        gz *= gz;
        gyp *= gyp;
        gym *= gym;
    }
    const float qx = (pi.x - g.lo[0]) * tr.inv_cw;
    const int32_t x0 = cx > 0 ? cx - 1 : 0, x1 = cx < g.g[0] - 1 ? cx + 1 : g.g[0] - 1;
    const uint32_t home = cbase + (uint32_t)((cz * g.g[1] + cy) * g.g[0]);
    const int32_t z1 = cz + sg, yp = cy + sg, ym = cy - sg;
    const bool inz = z1 >= 0 && z1 < g.g[2], inp = yp >= 0 && yp < g.g[1], inm = ym >= 0 && ym < g.g[1];
    uint32_t b[kSets], en[kSets];
    auto range = [&](int u, bool in, int32_t dz, int32_t dy, float gap2) {
        int32_t xa = x0, xb = x1;
        if (trim) {
            const float w2 = tr.r2 - gap2;
            in = in && !(w2 < 0.f);
            const float w = __builtin_amdgcn_sqrtf(fmaxf(w2, 0.f)) + tr.margin;
            xa = min(max(x0, (int32_t)__builtin_fmaf(-w, tr.inv_cw, qx)), x1);
            xb = min(x1, (int32_t)__builtin_fmaf(w, tr.inv_cw, qx));
        }
        b[u] = en[u] = 0u;
        if (in && active) {
            const uint32_t row = home + (uint32_t)(sg * (dz * g.g[1] + dy) * g.g[0]);
            b[u] = off[row + xa];
            en[u] = off[row + xb + 1];
        }
    };
    range(0, sub == 0u, 0, 0, 0.f);
    range(1, inp, 0, 1, gyp);
    range(2, inz && inm, 1, -1, gz + gym);
    range(3, inz, 1, 0, gz);
    range(4, inz && inp, 1, 1, gz + gyp);
    uint32_t np = 0;
    const f32x4* const p4 = reinterpret_cast<const f32x4*>(pos);
    // candidate t + q kPairLanes exists iff t < lim[q] (or, without LIMITS, t + q kPairLanes <
    // lim[0])
    auto limits = [](uint32_t e, uint32_t (&lim)[kCandidates]) {
        lim[0] = e;
#pragma unroll
        for (int q = 1; LIMITS && q < kCandidates; ++q) lim[q] = e > (uint32_t)(q * kPairLanes) ? e - (uint32_t)(q * kPairLanes) : 0u;
    };
    auto visit = [&](uint32_t t, const uint32_t (&lim)[kCandidates], const f32x4 (&v)[kCandidates]) {
#pragma unroll
        for (int q = 0; q < kCandidates; ++q) {
            if (q > 0 && (LIMITS ? t >= lim[q] : t + q * kPairLanes >= lim[0])) continue;
            const float4 pj = make_float4(v[q].x, v[q].y, v[q].z, v[q].w);
            const float dx = pj.x - pi.x, dy = pj.y - pi.y, dz = pj.z - pi.z;
            const float d2 = dist2(dx, dy, dz);
            if (PRED == LJ_PRED_CUDALJ && t + q * kPairLanes == k) continue;
            const int mult = pair_mult<PRED>(c, pi, pj, d2);
            if (!mult) continue;
            np += (uint32_t)mult;
            acc.add(c, pj, dx, dy, dz, d2, mult);
        }
    };
    // One 64-bit base, the candidates at immediate offsets from it, and their limits kept
    // from step to step (a batch of 25.5M particles in systems of 2,000-60,000 of 70
    // neighbours: 9,675 us with both formed anew for each candidate, 9,472 with the one base,
    // 9,182 with the limits too).  Without LIMITS the latter are formed for each candidate
    // (the copy in LDS: 1,000 particles 42.4 us with them, 42.1 without).
    auto load = [&](uint32_t t, f32x4 (&v)[kCandidates]) {
        const f32x4* const pt = p4 + t;
#pragma unroll
        for (int q = 0; q < kCandidates; ++q) v[q] = pt[q * kPairLanes];
    };
#pragma unroll
    for (int u = 0; u < kSets; ++u) {
        uint32_t t = of_even(b[u]) + sub, e = of_even(en[u]), t2 = of_odd(b[u]) + (sub ^ 1u), e2 = of_odd(en[u]);
        if (t >= e) {
            t = t2;
            e = e2;
            t2 = e2;
        }
        if constexpr (AHEAD) {
            f32x4 v[kCandidates];
            uint32_t lim[kCandidates];
            load(t, v);
            while (t < e) {
                limits(e, lim);
                uint32_t tn = t + kCandidates * kPairLanes, eN = e;
                if (tn >= e) {  // on to the mirror row
                    tn = t2;
                    eN = e2;
                    t2 = e2;
                }
                f32x4 vn[kCandidates];
                load(tn < eN ? tn : t, vn);
                visit(t, lim, v);
                t = tn;
                e = eN;
#pragma unroll
                for (int q = 0; q < kCandidates; ++q) v[q] = vn[q];
            }
        } else {
            uint32_t lim[kCandidates];
            limits(e, lim);
            while (t < e) {
                f32x4 v[kCandidates];
                load(t, v);
                visit(t, lim, v);
                t += kCandidates * kPairLanes;
                if (t >= e) {  // on to the mirror row
                    t = t2;
                    e = e2;
                    t2 = e2;
                    limits(e, lim);
                }
            }
        }
    }
    return np;
}

}  // namespace lj
