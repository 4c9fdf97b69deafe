// verlet.hip -- forces over a stored neighbour list, for time stepping with list reuse.
//
// The reference rebuilds everything for every loop (it draws new particles each time,
// Cuda-version/cudaLJ.cu:602-611), so it has no counterpart.  A molecular-dynamics
// caller instead builds a list once at rc + skin (lj_pairs / lj_lbvh_pairs), reuses it
// while no particle has moved more than skin / 2 (lj_max_displacement), and evaluates
// forces over the listed pairs with the true cutoff predicate: every pair within rc
// of the current positions is then in the list, so the pair set is exactly
// lj_compute's.
#include "lj_internal.h"
#include "lj_pair.h"
#include "lj_sort.h"

namespace lj {

namespace {

// The positions as one 16-byte record each: the list's partners lie at random indices,
// and one load then brings a partner's position where three arrays took three.
__global__ __launch_bounds__(256) void k_pack_positions(const float* __restrict__ x, const float* __restrict__ y,
                                                        const float* __restrict__ z, uint32_t n,
                                                        float4* __restrict__ pos) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < n) pos[i] = make_float4(x[i], y[i], z[i], 0.f);
}

// kListLanes lanes per particle (row i of the CSR list, caller order), each taking every
// kListLanes-th entry, kListUnroll of them loaded at once; a workgroup takes `turns` times
// kListRows rows, one set after the other.  Entries j >= n are ignored.  The workgroup's
// totals, listed and accepted pairs among them, go to sums.
// Bound by the partners' gathers, a line each.  While the positions fit in an XCD's L2 the
// rows are taken as they come; beyond (order set, see kOrderBytes and OrderIf) in a spatial order, row
// order[k].w being the k-th, so that rows taken together share their partners' lines.
// 500,009 particles at shuffled indices, 36M entries: 366 us as they come (12.6 TB/s of
// 128-byte lines from the caches), 156 us in spatial order.  One lane per row, whose loads
// of the list touched 64 lines and whose three gathers per entry waited for each other,
// took 1144 us.
constexpr int kListLanes = 8;
constexpr int kListUnroll = 4;
constexpr int kListRows = 256 / kListLanes;

// Positions above this size are gathered in spatial order: the rows by the Morton code of
// their particles, 2^kOrderBits steps per axis of the box, whose two radix passes take 45 us
// at 500,000 particles.  The line lies at one and a half times an XCD's 4 MiB L2.  Measured
// (the step with the displacement test, us, as they come -> in order): shuffled uniform
// 200,000 97 -> 97, 300,000 161 -> 126, 500,000 356 -> 198, 1M 956 -> 466; clustered 300,000
// 166 -> 187, 500,000 383 -> 324, 1M 983 -> 767; particles that already lie in cell order,
// where the sort is for nothing, 300,000 65 -> 92, 1M 196 -> 255.
// Lists of fewer than kOrderEntries a row are taken as they come, which the sort and the
// forces see from the list's own length on the device (shuffled uniform, lj_compute_list, as
// they come -> in order; before either, one lane a row): 500,000 particles of 2 neighbours
// 63 -> 99 (75), of 16 118 -> 118 (223), of 20 136 -> 124 (292); 3M of 2 206 -> 561 (416), of 16
// 859 -> 858 (2,620), of 20 1,065 -> 905 (3,386).
constexpr uint64_t kOrderBytes = 6u << 20;
constexpr int kOrderBits = 5;
constexpr uint64_t kOrderEntries = 16;

// The list's entries, on the device, and how few of them are not worth the order.
struct OrderIf {
    const unsigned long long* entries;
    unsigned long long least;
    __device__ bool no() const { return *entries < least; }
};
struct ListOrderOp : MortonKeyOp<kOrderBits> {
    OrderIf order;
    ListOrderOp(const lj_params* p, OrderIf o) : MortonKeyOp<kOrderBits>(p->box_lo, p->box_hi), order(o) {}
    __device__ bool skip() const { return order.no(); }
};

template <int PRED, int PREC, bool VIR>
__global__ __launch_bounds__(256) void k_list_force(const float4* __restrict__ pos, uint32_t n,
                                                    const float4* __restrict__ order, OrderIf want,
                                                    const unsigned long long* __restrict__ rows,
                                                    const uint32_t* __restrict__ cols, PairConst c, uint32_t turns,
                                                    float* __restrict__ fx, float* __restrict__ fy,
                                                    float* __restrict__ fz, float* __restrict__ e,
                                                    BlockSums* __restrict__ sums) {
    const uint32_t sub = threadIdx.x % kListLanes;
    const uint32_t blk = xcd_block(blockIdx.x, gridDim.x);
    if (order && want.no()) order = nullptr;
    unsigned long long np = 0, listed = 0;
    double esum = 0.0, vsum = 0.0;
    for (uint32_t turn = 0; turn < turns; ++turn) {
        const uint32_t k = (blk * turns + turn) * kListRows + threadIdx.x / kListLanes;
        PairSums<PREC, PRED == LJ_PRED_CUDALJ, VIR> acc;
        const bool active = k < n;
        const uint32_t i = order && active ? __float_as_uint(order[k].w) : k;
        const float4 pi = active ? pos[i] : make_float4(0.f, 0.f, 0.f, 0.f);
        acc.set_i(pi);
        acc.allow_exact_diff(c, pi, active);
        unsigned long long q = 0, r1 = 0;
        if (active) {
            q = rows[i] + sub;
            r1 = rows[i + 1];
        }
        for (; q < r1; q += kListLanes * kListUnroll) {
            uint32_t j[kListUnroll];
            float4 pj[kListUnroll];
            // every load issued before any is used; a place past the row's end reads the
            // lane's first entry again and is not counted
#pragma unroll
            for (int u = 0; u < kListUnroll; ++u) {
                const unsigned long long at = q + u * kListLanes;
                j[u] = cols[at < r1 ? at : q];
            }
#pragma unroll
            for (int u = 0; u < kListUnroll; ++u) pj[u] = pos[j[u] < n ? j[u] : i];
#pragma unroll
            for (int u = 0; u < kListUnroll; ++u) {
                if (q + u * kListLanes >= r1 || j[u] >= n) continue;
                ++listed;
                const float dx = pj[u].x - pi.x, dy = pj[u].y - pi.y, dz = pj[u].z - pi.z;
                const float d2 = dist2(dx, dy, dz);
                if constexpr (PRED == LJ_PRED_CUDALJ) {
                    if (j[u] == i) continue;
                }
                const int mult = pair_mult<PRED>(c, pi, pj[u], d2);
                if (!mult) continue;
                np += (unsigned long long)mult;
                acc.add(c, pj[u], dx, dy, dz, d2, mult);
            }
        }
        acc.template merge<kListLanes>();
        if (active && sub == 0) {
            fx[i] = (float)(-c.e24 * (double)acc.ax.value());
            fy[i] = (float)(-c.e24 * (double)acc.ay.value());
            fz[i] = (float)(-c.e24 * (double)acc.az.value());
            const double ei = c.e4 * (double)acc.ae.value();
            if (e) e[i] = (float)ei;
            esum += ei;
            vsum += c.e24 * (double)acc.av.value();
        }
    }
    store_block_sums<true, true>(&sums[blk], esum, vsum, np, listed);
}

// Largest |p - p0|^2 (FP32, a non-negative float: its bits order like the value).  At
// most kDispBlocks workgroups, one atomic each: with one per wave, 500,009 particles sent
// 7,800 atomics to the one counter and took 91 us.
constexpr unsigned kDispBlocks = 512;

__global__ __launch_bounds__(256) void k_max_disp(const float* __restrict__ x, const float* __restrict__ y,
                                                  const float* __restrict__ z, const float* __restrict__ x0,
                                                  const float* __restrict__ y0, const float* __restrict__ z0, uint32_t n,
                                                  unsigned int* __restrict__ max2) {
    __shared__ float wmax[256 / kWaveSize];
    float m = 0.f;
    for (uint64_t i = blockIdx.x * 256u + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256u) {
        const float dx = x[i] - x0[i], dy = y[i] - y0[i], dz = z[i] - z0[i];
        const float d2 = dist2(dx, dy, dz);
        m = fmaxf(m, d2 >= 0.f ? d2 : INFINITY);  // a NaN displacement forces a rebuild
    }
#pragma unroll
    for (int d = kWaveSize / 2; d > 0; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, kWaveSize));
    if (__lane_id() == 0) wmax[threadIdx.x / kWaveSize] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 256 / kWaveSize; ++w) m = fmaxf(m, wmax[w]);
        if (m > 0.f) atomicMax(max2, __float_as_uint(m));
    }
}

__global__ void k_zero_u32(unsigned int* p) { *p = 0u; }

}  // namespace

}  // namespace lj

using namespace lj;

extern "C" {

int lj_compute_list(lj_context* ctx, const float* x, const float* y, const float* z, int64_t n, const lj_params* p,
                    const unsigned long long* row_offsets, const uint32_t* cols, float* fx, float* fy, float* fz,
                    float* e, lj_result* result, void* stream) {
    if (!ctx) return LJ_ERR_INVALID_ARG;
    GridGeom g;
    PairConst c;
    LJ_TRY(make_geom(ctx, p, n, &g, &c));
    if (n > 0 && (!x || !y || !z || !fx || !fy || !fz || !row_offsets || !cols))
        return fail(ctx, LJ_ERR_INVALID_ARG, "NULL pointer argument");
    LJ_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = (hipStream_t)stream;
    lj_result* res = result;
    if (!res) {
        LJ_HIP(ctx, ctx->bin.counters.grow(sizeof(lj_result)));
        res = ctx->bin.counters.as<lj_result>();
    }
    PhaseTimer tf(ctx, LJ_PHASE_FORCE, s);
    // up to 8 sets of rows per workgroup once there are workgroups for every CU
    const int64_t sets = div_up(n > 0 ? n : 1, kListRows);
    const uint32_t turns = (uint32_t)(sets < 2048 ? 1 : sets < 16384 ? sets / 2048 : 8);
    const unsigned nb = div_up(sets, turns);
    LJ_HIP(ctx, ctx->bin.stage.grow((size_t)(n > 0 ? n : 1) * sizeof(float4)));
    float4* pos = ctx->bin.stage.as<float4>();
    const float4* order = nullptr;
    const OrderIf want{row_offsets + n, (unsigned long long)n * kOrderEntries};
    if ((uint64_t)n * sizeof(float4) > kOrderBytes) {
        LJ_TRY(sort_particles(ctx, x, y, z, n, ListOrderOp(p, want), 3 * kOrderBits, s));
        order = ctx->bin.pos.as<float4>();
    }
    if (n > 0) hipLaunchKernelGGL(k_pack_positions, dim3(div_up(n, 256)), dim3(256), 0, s, x, y, z, (uint32_t)n, pos);
    BlockSums* sums;
    LJ_TRY(grow_block_sums(ctx, nb, &sums));
    const bool vir = !(p->flags & LJ_FLAG_NO_VIRIAL);
    const uint32_t nn = (uint32_t)n;
#define LJ_LF(PRED, PREC, VIR)                                                                                    \
    hipLaunchKernelGGL((k_list_force<PRED, PREC, VIR>), dim3(nb), dim3(256), 0, s, (const float4*)pos, nn, order, want, row_offsets, \
                       cols, c, turns, fx, fy, fz, e, sums)
#define LJ_LF_V(PRED, PREC)            \
    do {                               \
        if (vir) LJ_LF(PRED, PREC, true); \
        else LJ_LF(PRED, PREC, false); \
    } while (0)
#define LJ_LF_P(PRED)                                          \
    switch (p->precision) {                                    \
    case LJ_PREC_MIXED: LJ_LF_V(PRED, LJ_PREC_MIXED); break;   \
    case LJ_PREC_FP32: LJ_LF_V(PRED, LJ_PREC_FP32); break;     \
    default: LJ_LF_V(PRED, LJ_PREC_FP32_COMP); break;          \
    }
    switch (p->predicate) {
    case LJ_PRED_AABB: LJ_LF_P(LJ_PRED_AABB); break;
    case LJ_PRED_CUSTOM: LJ_LF_P(LJ_PRED_CUSTOM); break;
    case LJ_PRED_CUDALJ: LJ_LF_P(LJ_PRED_CUDALJ); break;
    case LJ_PRED_SPHERE: LJ_LF_P(LJ_PRED_SPHERE); break;
    case LJ_PRED_TRIANGLE: LJ_LF_P(LJ_PRED_TRIANGLE); break;
    }
#undef LJ_LF_P
#undef LJ_LF_V
#undef LJ_LF
    return finalize_totals(ctx, nb, nullptr, 0u, nullptr, res, s);
}

int lj_max_displacement(lj_context* ctx, const float* x, const float* y, const float* z, const float* x0,
                        const float* y0, const float* z0, int64_t n, float* max2, void* stream) {
    if (!ctx) return LJ_ERR_INVALID_ARG;
    if (n < 0 || n > 0x7fffffffll) return fail(ctx, LJ_ERR_INVALID_ARG, "particle count out of range");
    if (!max2 || (n > 0 && (!x || !y || !z || !x0 || !y0 || !z0)))
        return fail(ctx, LJ_ERR_INVALID_ARG, "NULL pointer argument");
    LJ_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = (hipStream_t)stream;
    unsigned int* m = reinterpret_cast<unsigned int*>(max2);
    // a fill kernel, not hipMemsetAsync: the call may be captured in a graph
    hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(1), 0, s, m);
    if (n > 0)
        hipLaunchKernelGGL(k_max_disp, dim3(n > (int64_t)kDispBlocks * 256 ? kDispBlocks : div_up(n, 256)), dim3(256), 0, s,
                           x, y, z, x0, y0, z0, (uint32_t)n, m);
    LJ_HIP(ctx, hipGetLastError());
    return LJ_OK;
}

}  // extern "C"
