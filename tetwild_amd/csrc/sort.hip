// sort.hip -- Morton ordering of query batches.  Envelope queries arrive in
// whatever order the caller produced them; walking them in Morton order makes
// neighbouring threads (and, through the XCD-aware block order, each XCD's
// L2) visit the same tree paths.  Results never depend on the order.
#include <cmath>
#include <utility>

#include "twg_bvh.hpp"
#include "twg_internal.hpp"

namespace twg {
namespace {

// the item's place: a point, or a triangle's centroid
__device__ __forceinline__ void item_place(const double* __restrict__ p, int stride, double c[3])
{
    for (int k = 0; k < 3; ++k) c[k] = stride == 9 ? (p[k] + p[3 + k] + p[6 + k]) * (1.0 / 3.0) : p[k];
}

// The box the keys divide: that of up to kBoxThreads items spread over the
// batch (a triangle's first corner), a sixteenth wider, within the tree's box
// [lo, hi] (which it is when the two do not meet).  One block; box[0..2] the
// corner, box[3..5] cells per unit length.
constexpr int kBoxThreads = 1024;
struct Box6 {
    double lo[3], hi[3];
};
__global__ __launch_bounds__(kBoxThreads) void query_box(const double* __restrict__ items, int64_t n,
                                                         int stride, Box6 tree, double* __restrict__ box)
{
    __shared__ double red[6][kBoxThreads / 64];
    double v[6] = {INFINITY, INFINITY, INFINITY, INFINITY, INFINITY, INFINITY};
    const int64_t k = threadIdx.x;
    const int64_t i = n > kBoxThreads ? (int64_t)((double)k * ((double)n / kBoxThreads)) : k;
    if (i < n) {
        const double* c = items + (int64_t)stride * i;
        for (int q = 0; q < 3; ++q)
            if (is_finite(c[q])) {
                v[q] = c[q];
                v[3 + q] = -c[q];
            }
    }
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        for (int off = 32; off > 0; off >>= 1) v[q] = fmin(v[q], __shfl_xor(v[q], off, 64));
        if (threadIdx.x % 64 == 0) red[q][threadIdx.x / 64] = v[q];
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        const int q = threadIdx.x;
        double lo = INFINITY, hi = -INFINITY;
#pragma unroll
        for (int w = 0; w < kBoxThreads / 64; ++w) {
            lo = fmin(lo, red[q][w]);
            hi = fmax(hi, -red[3 + q][w]);
        }
        const double m = (hi - lo) * (1.0 / 16);
        lo = fmax(lo - m, tree.lo[q]);
        hi = fmin(hi + m, tree.hi[q]);
        if (!(lo < hi)) {
            lo = tree.lo[q];
            hi = tree.hi[q];
        }
        box[q] = lo;
        box[3 + q] = hi > lo ? 2097152.0 / (hi - lo) : 0.0;
    }
}

// ---- the sort ---------------------------------------------------------------
// Least digit first over kDigitBits-bit digits, stable, in three launches a
// pass: every block of kSortTile items counts its digits (count[digit][block];
// the first pass counts as it makes the keys), a block per digit scans its row
// and leaves the digit's total, and the items go to their places.  Nothing
// waits on another block.  27 bits, nine an axis, order 3 M items into cells of
// about four along a closed surface; below kTwoPassMax items 18 bits do, and a
// graded surface takes more (morton_bits).  Bound
// by its launches up to about 1 M items, by the scattered 8-byte writes
// beyond.  A library radix sort of 63-bit keys, with seventeen memory fills
// among its launches, took 440 us for 3 M triangles and 200 us for 1 M points;
// this takes 175 and 80 (4 M points a call: 829 -> 562 us).
constexpr int kDigitBits = 9;
constexpr int kDigits = 1 << kDigitBits;
constexpr int kSortItems = 16;  // per thread
constexpr int kSortTile = kBlock * kSortItems;
constexpr int64_t kTwoPassMax = 1 << 18;

// the item's sort key: the leading `bits` bits of its 63-bit Morton code in the box
__device__ __forceinline__ uint64_t morton_key(const double* __restrict__ p, int stride,
                                               const double* __restrict__ box, int bits)
{
    double c[3];
    item_place(p, stride, c);
    uint64_t key = 0;
    for (int k = 0; k < 3; ++k) {
        const double q = (c[k] - box[k]) * box[3 + k];
        const uint64_t qi = !(q > 0.0) ? 0 : (q >= 2097151.0 ? 2097151 : (uint64_t)q);
        key |= spread3d(qi) << k;
    }
    return key >> (63 - bits);
}

// keys (first pass) and the block's digit counts; KV: a (key, item) pair
template <class KV, bool FIRST>
__global__ __launch_bounds__(kBlock) void digit_count(const double* __restrict__ items, int64_t n,
                                                      int stride, const double* __restrict__ box,
                                                      int bits, int shift, KV* __restrict__ kv,
                                                      unsigned* __restrict__ count)
{
    __shared__ unsigned h[kDigits];
    for (int d = threadIdx.x; d < kDigits; d += kBlock) h[d] = 0u;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * kSortTile;
#pragma unroll 4
    for (int r = 0; r < kSortItems; ++r) {
        const int64_t i = base + r * kBlock + threadIdx.x;
        if (i >= n) break;
        KV v;
        if (FIRST) {
            v.x = (decltype(v.x))morton_key(items + (int64_t)stride * i, stride, box, bits);
            v.y = (uint32_t)i;
            kv[i] = v;
        } else {
            v.x = kv[i].x;
        }
        atomicAdd(&h[(unsigned)(v.x >> shift) & (kDigits - 1)], 1u);
    }
    __syncthreads();
    for (int d = threadIdx.x; d < kDigits; d += kBlock) count[(int64_t)d * gridDim.x + blockIdx.x] = h[d];
}

// exclusive scan of the block's 256 values; total: their sum
__device__ __forceinline__ unsigned block_scan(unsigned v, unsigned* wsum, unsigned& total)
{
    const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
    unsigned incl = v;
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned o = __shfl_up(incl, off, 64);
        if (lane >= off) incl += o;
    }
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    unsigned before = 0, all = 0;
#pragma unroll
    for (int k = 0; k < kBlock / 64; ++k) {
        before += k < w ? wsum[k] : 0u;
        all += wsum[k];
    }
    __syncthreads();
    total = all;
    return before + incl - v;
}

// the wave's LDS accesses so far come before its later ones
__device__ __forceinline__ void wave_order()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// block d: the exclusive scan of digit d's counts over the nb blocks, in place
__global__ __launch_bounds__(kBlock) void digit_scan(unsigned* __restrict__ count, int nb,
                                                     unsigned* __restrict__ total)
{
    __shared__ unsigned wsum[kBlock / 64];
    unsigned* row = count + (int64_t)blockIdx.x * nb;
    unsigned run = 0;
    for (int b0 = 0; b0 < nb; b0 += kBlock) {
        const int b = b0 + threadIdx.x;
        const unsigned v = b < nb ? row[b] : 0u;
        unsigned all;
        const unsigned ex = block_scan(v, wsum, all);
        if (b < nb) row[b] = run + ex;
        run += all;
    }
    if (threadIdx.x == 0) total[blockIdx.x] = run;
}

// Every item of the block's tile to its place: digit start + the block's start
// in the digit + its rank among the block's items of the digit, which keeps
// their order -- wave w holds items [1024 w, 1024 w + 1024) of the tile, 64 a
// round; the lanes of a round that share a digit find each other by ballots
// over its bits, and the wave's LDS counters carry the rounds.  LAST: only the
// item ids are written.
template <class KV, bool LAST>
__global__ __launch_bounds__(kBlock) void digit_place(const KV* __restrict__ in, int64_t n, int shift,
                                                      const unsigned* __restrict__ count,
                                                      const unsigned* __restrict__ total,
                                                      KV* __restrict__ out, int32_t* __restrict__ order)
{
    constexpr int W = kBlock / 64;
    __shared__ unsigned at[W][kDigits];
    __shared__ unsigned wsum[W];
    const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
    for (int d = threadIdx.x; d < W * kDigits; d += kBlock) (&at[0][0])[d] = 0u;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * kSortTile + w * (64 * kSortItems);
    const unsigned long long below = (1ull << lane) - 1ull;
    KV kv[kSortItems];
    unsigned rank[kSortItems];
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        const int64_t i = base + r * 64 + lane;
        kv[r].x = kv[r].y = 0;
        if (i < n) kv[r] = in[i];
    }
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        const bool ok = base + r * 64 + lane < n;
        const unsigned d = (unsigned)(kv[r].x >> shift) & (kDigits - 1);
        unsigned long long same = __ballot(ok);
#pragma unroll
        for (int b = 0; b < kDigitBits; ++b) {
            const unsigned long long m = __ballot((d >> b) & 1u);
            same &= (d >> b) & 1u ? m : ~m;
        }
        const unsigned before = at[w][d];
        rank[r] = before + (unsigned)__popcll(same & below);
        wave_order();
        if (ok && (same & below) == 0ull) at[w][d] = before + (unsigned)__popcll(same);
        wave_order();
    }
    __syncthreads();
    // at[w][d]: where the wave's items of digit d start
    unsigned run = 0;
    for (int d0 = 0; d0 < kDigits; d0 += kBlock) {
        const int d = d0 + threadIdx.x;
        unsigned all;
        const unsigned start = run + block_scan(total[d], wsum, all);
        run += all;
        unsigned p = start + count[(int64_t)d * gridDim.x + blockIdx.x];
#pragma unroll
        for (int k = 0; k < W; ++k) {
            const unsigned c = at[k][d];
            at[k][d] = p;
            p += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        if (base + r * 64 + lane >= n) continue;
        const unsigned p = at[w][(unsigned)(kv[r].x >> shift) & (kDigits - 1)] + rank[r];
        if (LAST) order[p] = (int32_t)kv[r].y;
        else out[p] = kv[r];
    }
}

}  // namespace

size_t sort_pairs_bytes(int64_t n)
{
    return (size_t)((n + kSortTile - 1) / kSortTile) * kDigits * 4 + kDigits * 4;
}

int sort_pairs(ulonglong2* kv[2], int64_t n, int bits, void* work, hipStream_t s)
{
    unsigned* total = static_cast<unsigned*>(work);
    unsigned* count = total + kDigits;
    const unsigned nb = (unsigned)((n + kSortTile - 1) / kSortTile);
    for (int shift = 0; shift < bits; shift += kDigitBits) {
        hipLaunchKernelGGL((digit_count<ulonglong2, false>), dim3(nb), dim3(kBlock), 0, s, nullptr, n, 0, nullptr,
                           0, shift, kv[0], count);
        TWG_LAUNCHED();
        hipLaunchKernelGGL(digit_scan, dim3(kDigits), dim3(kBlock), 0, s, count, (int)nb, total);
        TWG_LAUNCHED();
        hipLaunchKernelGGL((digit_place<ulonglong2, false>), dim3(nb), dim3(kBlock), 0, s, kv[0], n, shift, count,
                           total, kv[1], nullptr);
        TWG_LAUNCHED();
        std::swap(kv[0], kv[1]);
    }
    return TWG_OK;
}

// Bits of the query order.  Two passes of the sort up to kTwoPassMax items,
// three beyond, and more where the surface is graded: as many as leave no more
// than one facet in kCrowdShare in a crowded cell.  (3 M triangles on 246 k
// facets, 30 and 300 times smaller towards one side: with 27 bits the facets of a
// wave's queries overflow its list, 8452 and 10780 us a call, with 36 and 45 bits
// 1414 and 1484.)
constexpr int64_t kCrowdShare = 64;
static int default_passes(int64_t n) { return n < kTwoPassMax ? 2 : 3; }
static int morton_bits(const twg_bvh* B, int64_t n)
{
    constexpr int kLevels = kDigitBits / 3;  // a pass
    int passes = default_passes(n);
    while (passes * kLevels < kCrowdLevels - 1 && B->crowded[0][passes * kLevels] * kCrowdShare > B->nf) ++passes;
    return passes * kDigitBits;
}

bool morton_refined(const twg_bvh* B, int64_t n) { return morton_bits(B, n) > default_passes(n) * kDigitBits; }

// KV: a (key, item) pair that holds the key's bits
template <class KV>
static int order_items(twg_ctx* ctx, int slot, const double* items, int64_t n, int stride, const Box6& tree,
                       int bits, const int32_t** order)
{
    const size_t nb = (size_t)((n + kSortTile - 1) / kSortTile);
    // the box, the digits' totals, two buffers of (key, item), the order, the counts
    if (int r = ensure_slot(ctx, slot, 4096 + (size_t)n * (2 * sizeof(KV) + 4) + nb * kDigits * 4)) return r;
    char* base = (char*)ctx->slot[slot].p;
    double* box = (double*)base;
    unsigned* total = (unsigned*)(base + 1024);
    KV* kv[2] = {(KV*)(base + 4096), (KV*)(base + 4096) + n};
    int32_t* out = (int32_t*)(kv[1] + n);
    unsigned* count = (unsigned*)(out + n);
    static_assert(kDigits * 4 <= 4096 - 1024, "room for the totals");
    hipStream_t s = ctx->cur;
    hipLaunchKernelGGL(query_box, dim3(1), dim3(kBoxThreads), 0, s, items, n, stride, tree, box);
    TWG_LAUNCHED();
    const int passes = bits / kDigitBits;
    const dim3 g((unsigned)nb), b(kBlock);
    for (int p = 0; p < passes; ++p) {
        KV *from = kv[p % 2], *to = kv[1 - p % 2];
        const int shift = p * kDigitBits;
        if (p == 0) hipLaunchKernelGGL((digit_count<KV, true>), g, b, 0, s, items, n, stride, box, bits, shift, from, count);
        else hipLaunchKernelGGL((digit_count<KV, false>), g, b, 0, s, items, n, stride, box, bits, shift, from, count);
        TWG_LAUNCHED();
        hipLaunchKernelGGL(digit_scan, dim3(kDigits), b, 0, s, count, (int)nb, total);
        TWG_LAUNCHED();
        if (p + 1 < passes) hipLaunchKernelGGL((digit_place<KV, false>), g, b, 0, s, from, n, shift, count, total, to, out);
        else hipLaunchKernelGGL((digit_place<KV, true>), g, b, 0, s, from, n, shift, count, total, to, out);
        TWG_LAUNCHED();
    }
    *order = out;
    return TWG_OK;
}

int morton_order(twg_ctx* ctx, int slot, const double* items, int64_t n, int stride, const twg_bvh* B,
                 const int32_t** order)
{
    TWG_REQUIRE(n < (int64_t(1) << 31), "morton_order: too many items");
    Box6 tree;
    for (int k = 0; k < 3; ++k) {
        tree.lo[k] = B->lo[k];
        tree.hi[k] = B->hi[k];
    }
    const int bits = morton_bits(B, n);
    return bits <= 32 ? order_items<uint2>(ctx, slot, items, n, stride, tree, bits, order)
                      : order_items<ulonglong2>(ctx, slot, items, n, stride, tree, bits, order);
}

}  // namespace twg
