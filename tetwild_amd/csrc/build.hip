// build.hip -- the envelope tree built on the device: the facets' Morton
// order, the boxes of the implicit tree (twg_bvh.hpp) and the facets in tree
// order.  Every value is the host build's
// (envelope.hip), bit for bit: the same expressions in the same order, a
// stable sort, exact minima and maxima.
//
// Bound by the copy of the caller's arrays and a few dozen short launches;
// the host build spends its time in comparison sorts.  246 k facets:
// 121 ms on the host, 0.96 ms here (0.7 of it copies and allocations).
#include <cmath>

#include "build.hpp"
#include "twg_internal.hpp"

namespace twg {
namespace {

// what the whole build reduces to; doubles as ordered unsigned integers
struct BuildScalars {
    unsigned long long lo[3], hi[3];  // of the centroids
    unsigned long long rmax;          // bits of the longest edge
    unsigned long long bad;           // first corner with an id out of range
    unsigned crowded[2 * kCrowdLevels];  // facets by crowd_level to the kCrowd-th after them
};

__device__ __forceinline__ unsigned long long ordered(double x)
{
    const unsigned long long b = f2u(x);
    return b >> 63 ? ~b : b | 0x8000000000000000ull;
}
TWG_HD double unordered(unsigned long long u)
{
    return u2f(u >> 63 ? u & 0x7FFFFFFFFFFFFFFFull : ~u);
}

struct BuildArgs {
    const double* __restrict__ V;
    const int32_t* __restrict__ F;
    int64_t nv, nf;
    BuildScalars* sc;
    double* __restrict__ tri;
    int32_t* __restrict__ order;
};

// an id made safe to read with (build_check reports it)
__device__ __forceinline__ int64_t vid(const BuildArgs& A, int64_t c)
{
    const int64_t v = A.F[c];
    return v < 0 ? 0 : (v < A.nv ? v : A.nv - 1);
}

__global__ void build_init(BuildArgs A)
{
    for (int k = 0; k < 3; ++k) {
        A.sc->lo[k] = ordered(__builtin_inf());
        A.sc->hi[k] = ordered(-__builtin_inf());
    }
    A.sc->rmax = 0ull;
    A.sc->bad = ~0ull;
    for (int k = 0; k < 2 * kCrowdLevels; ++k) A.sc->crowded[k] = 0u;
}

__device__ __forceinline__ double centroid(const BuildArgs& A, int64_t f, int c)
{
    return (A.V[3 * vid(A, 3 * f) + c] + A.V[3 * vid(A, 3 * f + 1) + c] + A.V[3 * vid(A, 3 * f + 2) + c]) / 3.0;
}

__device__ __forceinline__ unsigned long long wave_max(unsigned long long v)
{
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned long long o = __shfl_xor(v, off, 64);
        v = o > v ? o : v;
    }
    return v;
}

// the block's largest v (every thread calls it), in thread 0
__device__ __forceinline__ unsigned long long block_max(unsigned long long v)
{
    __shared__ unsigned long long w[kBlock / 64];
    v = wave_max(v);
    if (threadIdx.x % 64 == 0) w[threadIdx.x / 64] = v;
    __syncthreads();
    for (int k = 1; k < kBlock / 64; ++k) v = threadIdx.x == 0 && w[k] > v ? w[k] : v;
    __syncthreads();
    return v;
}

// the centroids' box, and the first id out of range: few blocks, an atomic of
// each on the scalars (an atomic per wave of a full grid took 260 us)
constexpr unsigned kCheckBlocks = 256;
__global__ __launch_bounds__(kBlock) void build_check(BuildArgs A)
{
    unsigned long long lo[3], hi[3], bad = ~0ull;
    for (int c = 0; c < 3; ++c) {
        lo[c] = ~ordered(__builtin_inf());
        hi[c] = ordered(-__builtin_inf());
    }
    for (int64_t f = (int64_t)blockIdx.x * kBlock + threadIdx.x; f < A.nf; f += (int64_t)gridDim.x * kBlock) {
        for (int k = 2; k >= 0; --k)
            if ((A.F[3 * f + k] < 0 || A.F[3 * f + k] >= A.nv) && (unsigned long long)(3 * f + k) < bad)
                bad = 3 * f + k;
        for (int c = 0; c < 3; ++c) {
            const double v = centroid(A, f, c);
            if (v != v) continue;  // std::min and std::max pass over NaN
            const unsigned long long o = ordered(v);
            lo[c] = ~o > lo[c] ? ~o : lo[c];
            hi[c] = o > hi[c] ? o : hi[c];
        }
    }
    bad = ~block_max(~bad);
    for (int c = 0; c < 3; ++c) {
        lo[c] = block_max(lo[c]);
        hi[c] = block_max(hi[c]);
    }
    if (threadIdx.x) return;
    if (bad != ~0ull) atomicMin(&A.sc->bad, bad);
    for (int c = 0; c < 3; ++c) {
        atomicMin(&A.sc->lo[c], ~lo[c]);
        atomicMax(&A.sc->hi[c], hi[c]);
    }
}

__global__ __launch_bounds__(kBlock) void build_keys(BuildArgs A, ulonglong2* __restrict__ kv)
{
    const int64_t f = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (f >= A.nf) return;
    uint64_t key = 0;
    for (int c = 0; c < 3; ++c) {
        const double lo = unordered(A.sc->lo[c]), span = unordered(A.sc->hi[c]) - lo;
        const double q = span > 0 ? (centroid(A, f, c) - lo) / span * 2097152.0 : 0.0;
        const uint64_t qi = !(q > 0) ? 0 : (q >= 2097151.0 ? 2097151 : (uint64_t)q);
        key |= spread3d(qi) << c;
    }
    ulonglong2 r;
    r.x = key;
    r.y = (unsigned long long)f;
    kv[f] = r;
}

// twg_bvh::crowded by level, not summed yet
__global__ __launch_bounds__(kBlock) void build_crowded(BuildArgs A, const ulonglong2* __restrict__ sorted)
{
    __shared__ unsigned n[2 * kCrowdLevels];
    if (threadIdx.x < 2 * kCrowdLevels) n[threadIdx.x] = 0u;
    __syncthreads();
    for (int64_t b = (int64_t)blockIdx.x * kBlock + threadIdx.x; b < A.nf; b += (int64_t)gridDim.x * kBlock)
#pragma unroll
        for (int j = 0; j < 2; ++j)
            if (b + kCrowd[j] < A.nf)
                atomicAdd(&n[j * kCrowdLevels + crowd_level(sorted[b].x, sorted[b + kCrowd[j]].x)], 1u);
    __syncthreads();
    if (threadIdx.x < 2 * kCrowdLevels && n[threadIdx.x]) atomicAdd(&A.sc->crowded[threadIdx.x], n[threadIdx.x]);
}

// tree position b: the facet's corners, its order entry, its longest edge
__global__ __launch_bounds__(kBlock) void build_facets(BuildArgs A, const ulonglong2* __restrict__ sorted)
{
    const int64_t b = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    double r = 0.0;
    if (b < A.nf) {
        const int64_t f = (int64_t)sorted[b].y;
        A.order[b] = (int32_t)f;
        double t[9];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int64_t v = vid(A, 3 * f + k);
#pragma unroll
            for (int c = 0; c < 3; ++c) A.tri[9 * b + 3 * k + c] = t[3 * k + c] = A.V[3 * v + c];
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const double *a = t + 3 * k, *e = t + 3 * ((k + 1) % 3);
            const double l = __builtin_sqrt((a[0] - e[0]) * (a[0] - e[0]) + (a[1] - e[1]) * (a[1] - e[1]) +
                                            (a[2] - e[2]) * (a[2] - e[2]));
            r = r < l ? l : r;
        }
    }
    const unsigned long long m = block_max(f2u(r));  // not negative: its bits order it
    if (threadIdx.x == 0 && m) atomicMax(&A.sc->rmax, m);
}

// Node n at depth d of the tree over nf facets: from its children, its facet
// or, below a leaf, empty
__device__ __forceinline__ void build_node(BvhNode64* n64, BvhNode32* n32, const double* __restrict__ tri,
                                           int64_t nf, int64_t n, int d)
{
    int64_t b = 0, e = nf;
    bool none = false;
    for (int bit = d - 1; bit >= 0; --bit) {
        none = none || e - b <= 1;
        const int64_t m = b + (e - b) / 2;
        if ((n >> bit) & 1) b = m;
        else e = m;
    }
    BvhNode64 N;
    for (int c = 0; c < 3; ++c) {
        N.lo[c] = __builtin_inf();
        N.hi[c] = -__builtin_inf();
        N.pad[c] = 0;
    }
    N.leaf = -2;
    if (!none && e - b == 1) {
        const double* t = tri + 9 * b;
        for (int c = 0; c < 3; ++c) {
            N.lo[c] = N.hi[c] = t[c];
            for (int k = 1; k < 3; ++k) {
                N.lo[c] = t[3 * k + c] < N.lo[c] ? t[3 * k + c] : N.lo[c];
                N.hi[c] = N.hi[c] < t[3 * k + c] ? t[3 * k + c] : N.hi[c];
            }
        }
        N.leaf = (int32_t)b;
    } else if (!none) {
        const BvhNode64 L = n64[2 * n], R = n64[2 * n + 1];
        for (int c = 0; c < 3; ++c) {
            N.lo[c] = R.lo[c] < L.lo[c] ? R.lo[c] : L.lo[c];
            N.hi[c] = L.hi[c] < R.hi[c] ? R.hi[c] : L.hi[c];
        }
        N.leaf = -1;
    }
    n64[n] = N;
    BvhNode32 M;
    for (int c = 0; c < 3; ++c) {
        M.lo[c] = f32_down(N.lo[c]);
        M.hi[c] = f32_up(N.hi[c]);
    }
    M.leaf = N.leaf;
    M.pad = 0;
    n32[n] = M;
}

// Depths bottom .. top, a block per node at depth top: a level at a time,
// each from the level below it (the block's own, or an earlier launch's)
__global__ __launch_bounds__(kBlock) void build_levels(BvhNode64* n64, BvhNode32* n32,
                                                       const double* __restrict__ tri, int64_t nf, int top,
                                                       int bottom)
{
    const int64_t root = ((int64_t)1 << top) + blockIdx.x;
    for (int d = bottom; d >= top; --d) {
        const int64_t cnt = (int64_t)1 << (d - top);
        for (int64_t j = threadIdx.x; j < cnt; j += kBlock)
            build_node(n64, n32, tri, nf, (root << (d - top)) + j, d);
        __syncthreads();
    }
    if (top == 0 && threadIdx.x == 0) {  // slot 0 holds no node
        BvhNode64 N = {};
        BvhNode32 M = {};
        for (int c = 0; c < 3; ++c) {
            N.lo[c] = __builtin_inf();
            N.hi[c] = -__builtin_inf();
            M.lo[c] = __builtin_inff();
            M.hi[c] = -__builtin_inff();
        }
        N.leaf = M.leaf = -2;
        n64[0] = N;
        n32[0] = M;
    }
}

struct DeviceBlock {
    char* p = nullptr;
    ~DeviceBlock()
    {
        if (p) (void)hipFree(p);
    }
};

int bits_of(uint64_t x)
{
    int b = 0;
    while (x >> b) ++b;
    return b;
}

}  // namespace

int bvh_build_device(twg_ctx* ctx, const double* V, int64_t nv, const int32_t* F, int64_t nf, twg_bvh* B,
                     int64_t* bad)
{
    hipStream_t s = ctx->cur;
    const int depth = nf > 1 ? bits_of((uint64_t)(nf - 1)) : 0;
    B->depth = depth;
    B->nnode = (int64_t)2 << depth;  // the rightmost path is as deep as any
    auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
    const size_t b64 = up(sizeof(BvhNode64) * B->nnode), b32 = up(sizeof(BvhNode32) * B->nnode),
                 btri = up(72 * (size_t)nf);
    TWG_HIP(hipMalloc(&B->mem, b64 + b32 + btri));
    char* m = static_cast<char*>(B->mem);
    B->node64 = reinterpret_cast<BvhNode64*>(m);
    B->node32 = reinterpret_cast<BvhNode32*>(m + b64);
    B->tri = reinterpret_cast<double*>(m + b64 + b32);
    // working memory, freed before the call returns
    const size_t bV = up(24 * (size_t)nv), bF = up(12 * (size_t)nf), bO = up(4 * (size_t)nf),
                 bK = up(16 * (size_t)nf), bW = up(sort_pairs_bytes(nf));
    DeviceBlock W;
    TWG_HIP(hipMalloc(&W.p, 256 + bV + bF + bO + 2 * bK + bW));
    char* q = W.p;
    auto take = [&](size_t b) {
        char* r = q;
        q += b;
        return r;
    };
    BuildArgs A;
    A.nv = nv;
    A.nf = nf;
    A.sc = reinterpret_cast<BuildScalars*>(take(256));
    char* dV = take(bV);
    char* dF = take(bF);
    A.V = reinterpret_cast<const double*>(dV);
    A.F = reinterpret_cast<const int32_t*>(dF);
    A.order = reinterpret_cast<int32_t*>(take(bO));
    ulonglong2* kv[2] = {reinterpret_cast<ulonglong2*>(take(bK)), nullptr};
    kv[1] = reinterpret_cast<ulonglong2*>(take(bK));
    void* work = take(bW);
    A.tri = B->tri;
    TWG_HIP(hipMemcpyAsync(dV, V, 24 * (size_t)nv, hipMemcpyHostToDevice, s));
    TWG_HIP(hipMemcpyAsync(dF, F, 12 * (size_t)nf, hipMemcpyHostToDevice, s));
    const dim3 b(kBlock), gf(grid_for(nf));
    hipLaunchKernelGGL(build_init, dim3(1), dim3(1), 0, s, A);
    TWG_LAUNCHED();
    hipLaunchKernelGGL(build_check, dim3(std::min<unsigned>(grid_for(nf), kCheckBlocks)), b, 0, s, A);
    TWG_LAUNCHED();
    hipLaunchKernelGGL(build_keys, gf, b, 0, s, A, kv[0]);
    TWG_LAUNCHED();
    if (int r = sort_pairs(kv, nf, 63, work, s)) return r;
    hipLaunchKernelGGL(build_crowded, dim3(std::min<unsigned>(grid_for(nf), kCheckBlocks)), b, 0, s, A, kv[0]);
    TWG_LAUNCHED();
    hipLaunchKernelGGL(build_facets, gf, b, 0, s, A, kv[0]);
    TWG_LAUNCHED();
    for (int bottom = depth;;) {
        const int top = bottom > 9 ? bottom - 9 : 0;
        hipLaunchKernelGGL(build_levels, dim3(1u << top), b, 0, s, B->node64, B->node32, B->tri, nf, top, bottom);
        TWG_LAUNCHED();
        if (top == 0) break;
        bottom = top - 1;
    }
    BuildScalars h;
    BvhNode64 root;
    B->order.resize(nf);
    TWG_HIP(hipMemcpyAsync(B->order.data(), A.order, 4 * (size_t)nf, hipMemcpyDeviceToHost, s));
    TWG_HIP(hipMemcpyAsync(&root, B->node64 + 1, sizeof root, hipMemcpyDeviceToHost, s));
    TWG_HIP(hipMemcpyAsync(&h, A.sc, sizeof h, hipMemcpyDeviceToHost, s));
    TWG_HIP(hipStreamSynchronize(s));
    *bad = h.bad == ~0ull ? -1 : (int64_t)h.bad;
    B->rmax = u2f(h.rmax);
    for (int c = 0; c < 3; ++c) B->side = std::max(B->side, unordered(h.hi[c]) - unordered(h.lo[c]));
    for (int j = 0; j < 2; ++j) {
        int64_t n = 0;
        for (int l = kCrowdLevels - 1; l >= 0; --l) B->crowded[j][l] = n += h.crowded[j * kCrowdLevels + l];
    }
    for (int c = 0; c < 3; ++c) {
        B->lo[c] = root.lo[c];
        B->hi[c] = root.hi[c];
    }
    return TWG_OK;
}

}  // namespace twg
