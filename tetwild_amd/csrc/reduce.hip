// reduce.hip -- the energy reductions that drive pass termination in
// MeshRefinement (src/tetwild/MeshRefinement.cpp:185-206, 285-292):
// getAvgMaxEnergy, getMaxEnergy, getSecondMaxEnergy and the histogram of
// getFilterEnergy (src/tetwild/LocalOperations.cpp:605-693), in one pass over
// the per-tet slim energies resident in HBM.
//
// Each block walks a contiguous range of the tets; waves reduce by shuffles in
// a fixed tree, a block's four waves in order, and one block reduces the blocks'
// partials the same way.  Bound by the latency of the locked flags' gathers
// (ids, then four bytes each), so all flags of a thread's four tets are read
// before any is used (four blocks a CU; two and eight 60 and 70 us against 57).
// 3.1 M tets with locks 75 -> 57 us a call, 24 tets 43 -> 30: the flags tested
// one after another, an LDS tree over 128-byte records and a copy of the
// result after the kernels took the difference.  The result is deterministic for a given device (the grid depends
// only on the CU count).  Max, second max, counts and the histogram are exact;
// the sum differs from the reference's sequential loop by rounding only.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "twg_internal.hpp"
#include "twg_math.hpp"

namespace twg {
namespace {

struct Partial {
    double sum, max, second;
    unsigned long long count, bad;
    unsigned long long buckets[11];
};

constexpr int kUnroll = 4;

struct ReduceArgs {
    const double* __restrict__ e;
    int64_t n;
    const uint8_t* __restrict__ removed;
    const int4* __restrict__ tets;
    const uint8_t* __restrict__ locked;
    int64_t nv;
    double lim[11];  // filter_energy_thres - 1 + 10^j, j = 0..10
    Partial* part;
};

__device__ __forceinline__ void combine(Partial& a, const Partial& b)
{
    a.sum += b.sum;
    a.max = b.max > a.max ? b.max : a.max;
    a.second = b.second > a.second ? b.second : a.second;
    a.count += b.count;
    a.bad += b.bad;
#pragma unroll
    for (int k = 0; k < 11; ++k) a.buckets[k] += b.buckets[k];
}

// the wave's partials into every lane (a fixed tree: lanes 32 apart first)
__device__ __forceinline__ void wave_combine(Partial& p)
{
    for (int off = 32; off > 0; off >>= 1) {
        Partial q;
        q.sum = __shfl_xor(p.sum, off, 64);
        q.max = __shfl_xor(p.max, off, 64);
        q.second = __shfl_xor(p.second, off, 64);
        q.count = __shfl_xor(p.count, off, 64);
        q.bad = __shfl_xor(p.bad, off, 64);
#pragma unroll
        for (int k = 0; k < 11; ++k) q.buckets[k] = __shfl_xor(p.buckets[k], off, 64);
        combine(p, q);
    }
}

// the block's partials, its waves' in order, in thread 0
__device__ void block_reduce(Partial& p, Partial* lds)
{
    wave_combine(p);
    if (threadIdx.x % 64 == 0) lds[threadIdx.x / 64] = p;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int w = 1; w < kBlock / 64; ++w) combine(p, lds[w]);
}

__global__ __launch_bounds__(kBlock) void energy_partial_kernel(ReduceArgs A)
{
    __shared__ Partial lds[kBlock / 64];
    Partial p;
    p.sum = 0.0;
    p.max = 0.0;
    p.second = 0.0;
    p.count = 0;
    p.bad = 0;
#pragma unroll
    for (int k = 0; k < 11; ++k) p.buckets[k] = 0;
    // counts of one thread: far below 2^32
    unsigned count = 0, bad = 0, bucket[11] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    // Each block walks its own contiguous range (blocks in XCD order, so the
    // vertex flags its tets read stay in one L2), kUnroll coalesced elements
    // per thread per step with their loads issued before any is used.
    const int64_t step = (int64_t)kBlock * kUnroll;
    const int64_t per = ((A.n + gridDim.x - 1) / gridDim.x + step - 1) / step * step;
    const int64_t lo = xcd_block() * per;
    const int64_t hi = lo + per < A.n ? lo + per : A.n;
    const bool use_locks = A.tets && A.locked;
    for (int64_t base = lo + threadIdx.x; base < hi; base += step) {
        uint8_t rm[kUnroll];
        double ev[kUnroll];
        int4 tv[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const int64_t i = base + (int64_t)u * kBlock;
            const bool in = i < hi;
            rm[u] = in ? (A.removed ? A.removed[i] : 0) : 1;
            ev[u] = in ? A.e[i] : 0.0;
            tv[u] = in && use_locks ? A.tets[i] : make_int4(0, 0, 0, 0);
        }
        // isTetLocked_ui (:1377-1384): bit 0 locked, bit 1 an id out of range
        unsigned lk[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            lk[u] = 0u;
            if (!use_locks) continue;
            const int4 t = tv[u];
            const int id[4] = {t.x, t.y, t.z, t.w};
            unsigned out = 0u, any = 0u;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool in = id[j] >= 0 && id[j] < A.nv;
                out |= in ? 0u : 2u;
                any |= A.nv > 0 ? (unsigned)A.locked[in ? id[j] : 0] : 0u;
            }
            lk[u] = out ? out : (any ? 1u : 0u);
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            if (rm[u]) continue;
            const double e = ev[u];
            // getFilterEnergy: non-removed tets, locks ignored (:656-671); the
            // bucket index first, then an unrolled update (no run-time indexing)
            int bk = -1;
            if (e > A.lim[10]) {
                bk = 10;
            } else {
#pragma unroll
                for (int j = 9; j >= 0; --j)
                    if (e > A.lim[j] && e <= A.lim[j + 1]) bk = j;
            }
#pragma unroll
            for (int k = 0; k < 11; ++k) bucket[k] += (bk == k) ? 1u : 0u;
            if (lk[u] & 2u) bad++;
            if (lk[u]) continue;
            // getAvgMaxEnergy / getMaxEnergy (:605-635), getSecondMaxEnergy (:637-650)
            p.max = e > p.max ? e : p.max;
            if (e != kMaxEnergy) p.second = e > p.second ? e : p.second;
            p.sum += e;
            count++;
        }
    }
    p.count = count;
    p.bad = bad;
#pragma unroll
    for (int k = 0; k < 11; ++k) p.buckets[k] = bucket[k];
    block_reduce(p, lds);
    if (threadIdx.x == 0) A.part[blockIdx.x] = p;
}

__global__ __launch_bounds__(kBlock) void energy_final_kernel(Partial* part, int nblocks,
                                                              Partial* out)
{
    __shared__ Partial lds[kBlock / 64];
    Partial p;
    p.sum = 0.0;
    p.max = 0.0;
    p.second = 0.0;
    p.count = 0;
    p.bad = 0;
#pragma unroll
    for (int k = 0; k < 11; ++k) p.buckets[k] = 0;
    for (int b = threadIdx.x; b < nblocks; b += kBlock) combine(p, part[b]);
    block_reduce(p, lds);
    if (threadIdx.x == 0) *out = p;
}

}  // namespace
}  // namespace twg

using namespace twg;

extern "C" int twg_energy_stats(twg_ctx* ctx, const double* slim_energy, int64_t n,
                                const uint8_t* t_is_removed, const int32_t* tets,
                                const uint8_t* v_is_locked, int64_t nv,
                                double filter_energy_thres, twg_energy_summary* out)
{
    TWG_REQUIRE(ctx != nullptr && out != nullptr, "twg_energy_stats: NULL argument");
    TWG_REQUIRE(n >= 0 && nv >= 0, "twg_energy_stats: negative size");
    TWG_REQUIRE(n == 0 || slim_energy, "twg_energy_stats: NULL slim_energy");
    TWG_REQUIRE(!tets || ((uintptr_t)tets & 15) == 0, "twg_energy_stats: tets must be 16-byte aligned");
    ReduceArgs A;
    A.e = slim_energy;
    A.n = n;
    A.removed = t_is_removed;
    A.tets = reinterpret_cast<const int4*>(tets);
    A.locked = v_is_locked;
    A.nv = nv;
    // the bucket limits as the reference forms them: thres - 1 + pow(10, j)
    for (int j = 0; j <= 10; ++j) A.lim[j] = filter_energy_thres - 1 + std::pow(10.0, (double)j);
    if (int r = bind(ctx)) return r;
    const int nblocks = (int)std::max<int64_t>(1, std::min<int64_t>(grid_for(n), (int64_t)ctx->num_cus * 4));
    // the result goes to pinned host memory: no copy after the kernels, and one
    // block is its own final pass
    static_assert(sizeof(Partial) <= kHostOutBytes, "room for the result");
    if (!ctx->host_out) TWG_HIP(hipHostMalloc(&ctx->host_out, kHostOutBytes, hipHostMallocDefault));
    void* dout = nullptr;
    TWG_HIP(hipHostGetDevicePointer(&dout, ctx->host_out, 0));
    if (int r = ensure_scratch(ctx, sizeof(Partial) * (size_t)nblocks)) return r;
    A.part = nblocks == 1 ? static_cast<Partial*>(dout) : static_cast<Partial*>(ctx->scratch.p);
    hipLaunchKernelGGL(energy_partial_kernel, dim3(nblocks), dim3(kBlock), 0, ctx->cur, A);
    TWG_LAUNCHED();
    if (nblocks > 1) {
        hipLaunchKernelGGL(energy_final_kernel, dim3(1), dim3(kBlock), 0, ctx->cur, A.part, nblocks,
                           static_cast<Partial*>(dout));
        TWG_LAUNCHED();
    }
    TWG_HIP(hipStreamSynchronize(ctx->cur));
    Partial h;
    std::memcpy(&h, ctx->host_out, sizeof h);
    TWG_REQUIRE(h.bad == 0, "twg_energy_stats: %llu tets with vertex ids outside [0, nv)",
                (unsigned long long)h.bad);
    out->sum = h.sum;
    out->max = h.max;
    out->second_max = h.second;
    out->count = (int64_t)h.count;
    for (int k = 0; k < 11; ++k) out->buckets[k] = (int64_t)h.buckets[k];
    return TWG_OK;
}
