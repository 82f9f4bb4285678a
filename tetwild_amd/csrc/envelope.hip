// envelope.hip -- (b) the envelope test: isFaceOutEnvelop_sampling,
// isPointOutEnvelop, nearest_facet and sampleTriangle, over a flattened
// implicit AABB tree resident in HBM.
//
// The tree layout and the decision rule are described in twg_bvh.hpp.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <vector>

#include "build.hpp"
#include "twg_bvh.hpp"
#include "twg_internal.hpp"

namespace twg {
namespace {

__device__ __forceinline__ void flush_stats(const Stats& st, unsigned long long* out)
{
    unsigned long long v[4] = {st.samples, st.traversals, st.boxes, st.leaves};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        unsigned long long s = v[k];
        for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
        if ((threadIdx.x & 63) == 0 && s) atomicAdd(&out[k], s);
    }
}

// LDS copy of the tree top for the point kernel (its registers allow more
// resident blocks than 32 KB of LDS per block would)
constexpr int kPointCacheBytes = 16384;

template <bool F32, bool STATS>
__global__ __launch_bounds__(kBlock) void points_kernel(BvhView B, const double* __restrict__ p3,
                                                        int64_t n, double eps2, double T,
                                                        double sqrtT, uint8_t* __restrict__ out,
                                                        unsigned long long* stats,
                                                        const int32_t* __restrict__ order)
{
    __shared__ __align__(16) unsigned char cache[kPointCacheBytes];
    const BvhWalk W = cache_tree_top<F32, kPointCacheBytes>(B, cache);
    int64_t i = xcd_block() * kBlock + threadIdx.x;
    Stats st;
    if (i < n) {
        if (order) i = order[i];
        int hint = -1;
        V3<double> p = ld3(p3 + 3 * i);
        if (STATS) st.samples++;
        out[i] = in_envelope<F32, STATS>(W, p, eps2, T, sqrtT, hint, st) ? 0 : 1;
    }
    if (STATS) flush_stats(st, stats);
}

// Waves whose facets do not fit their list take their items in halves, down to
// this many lanes.
constexpr int kListSplit = 8;
// ... and only while the box is so many times as wide as one query's (`one`: its
// own extent and the envelope's on both sides): where the envelope is about as
// wide as the box, a half meets nearly the same facets.  Lanes may hold different
// boxes where a coordinate is not finite: one answer for the wave.  (Points, 3 M and 1 M of
// them with an envelope of two facets and 1 M of three: 1849, 1323 and 1774 us a
// call at 1.5, 2475, 1370 and 1666 at 2.0.  Triangles, 2 M with an envelope of one
// and a half facets and 106 k with 0.6: 4323 and 1300 us at 2.0, 5243 and 1396 at
// 1.5.)
constexpr double kHalvePoints = 1.5, kHalveFaces = 2.0;
__device__ __forceinline__ bool halves_help(const double lo[3], const double hi[3], double one)
{
    return __ballot(fmax(hi[0] - lo[0], fmax(hi[1] - lo[1], hi[2] - lo[2])) >= one) != 0ull;
}

// points_kernel for small batches: sixteen lanes per point, which list the
// facets within reach (collect_facets) and test one each -- a chain of a few
// reads instead of a walk's, with lanes to spare, in the caller's order.  On
// 246 k facets 4,096 points 143 -> 17 us, 65 k 169 -> 53, 400 k 282 -> 240, but
// 1 M 451 -> 563 (there the sort pays, and from two points a facet on the wave
// lists).  Dense batches of 65 k points and more keep the wave lists too, and
// where the envelope is wide (reach_wide) most lists overflow and sixteen lanes
// walk one point's way: an envelope of three facets, 5 k points 445 -> 222 us, but
// 60 k 443 -> 670 and 450 k 1003 -> 3965, so from kPointGroupWide points on those
// keep points_kernel.
// (Eight and thirty-two lanes: 58 and 61 us for 65 k.)
constexpr int kPointGroup = 16;
constexpr int kPointGroupCap = 32;
constexpr int64_t kPointGroupMax = 1 << 19;
constexpr int64_t kPointGroupDensity = 8;
constexpr int64_t kPointGroupWide = 1 << 15;
template <bool F32>
__global__ __launch_bounds__(kBlock) void points_group_kernel(BvhView B, const double* __restrict__ p3,
                                                              int64_t n, double eps2, double T,
                                                              double sqrtT, uint8_t* __restrict__ out)
{
    constexpr int G = kPointGroup;
    __shared__ __align__(16) unsigned char lists[(kBlock / G) * kPointGroupCap * 40];
    const BvhWalk W = walk(B);
    const int gl = threadIdx.x % G, gbase = (threadIdx.x % 64) - gl;
    const int64_t i = (int64_t)blockIdx.x * (kBlock / G) + threadIdx.x / G;
    if (i >= n) return;
    unsigned char* mine = lists + (threadIdx.x / G) * (kPointGroupCap * 40);
    LdsNode32W* lst = (LdsNode32W*)mine;
    const V3<double> p = ld3(p3 + 3 * i);
    const double pad = 1.0001 * sqrtT + 1e-9 * fmax(fabs(p.x), fmax(fabs(p.y), fabs(p.z)));
    const double lo[3] = {p.x - pad, p.y - pad, p.z - pad}, hi[3] = {p.x + pad, p.y + pad, p.z + pad};
    const int nl = collect_facets<G>(W, lo, hi, lst, (LdsU32*)(mine + kPointGroupCap * 32), kPointGroupCap,
                                     gl, gbase);
    bool in = false;
    if (nl >= 0) {
        for (int e = gl; e < nl && !in; e += G) in = facet_d2(W, lst[e].leaf, p) <= eps2;
        const unsigned long long gm = (G == 64 ? ~0ull : (1ull << (G & 63)) - 1ull) << gbase;
        in = (__ballot(in) & gm) != 0ull;
    } else {
        int hint = -1;
        Stats st;
        in = in_envelope<F32, false>(W, p, eps2, T, sqrtT, hint, st);
    }
    if (gl == 0) out[i] = in ? 0 : 1;
}

// points_kernel for batches walked in Morton order with many points per
// facet: the wave's 64 consecutive points lie close together, so the wave
// lists once (collect_facets, LDS) the facets whose boxes meet the box of its
// points padded by more than sqrt(T), with their certificates, and each lane
// tests its point against the list (in_envelope_cert).  Blocks of one wave and
// split waves as faces_list_kernel; lanes that no list serves, or that hold a
// coordinate that is not finite, walk the tree, all at once at the end.
template <bool F32, int CAP>
__global__ __launch_bounds__(64) void points_list_kernel(BvhView B, const double* __restrict__ p3,
                                                         int64_t n, double eps2, double T,
                                                         double sqrtT, uint8_t* __restrict__ out,
                                                         const int32_t* __restrict__ order,
                                                         unsigned long long* lstat)
{
    __shared__ __align__(16) unsigned char mine[CAP * kCertEntryBytes];
    const BvhWalk W = walk(B);
    const int lane = threadIdx.x;
    LdsNode32W* lst = (LdsNode32W*)mine;
    LdsU32* fr = (LdsU32*)(mine + CAP * 32);  // the work lists, then the certificates
    LdsF32* cert = (LdsF32*)(mine + CAP * 32);
    int64_t i = xcd_run_block() * 64 + lane;
    const bool have = i < n;
    V3<double> p = mk3(0.0, 0.0, 0.0);
    if (have) {
        if (order) i = order[i];
        p = ld3(p3 + 3 * i);
    }
    const bool fin = is_finite(p.x) && is_finite(p.y) && is_finite(p.z);
    bool rest = false;
    for (int s = 0, w = 64; s < 64;) {
        const bool act = have && lane >= s && lane < s + w;
        if (__ballot(act)) {
            double lo[3] = {act ? p.x : INFINITY, act ? p.y : INFINITY, act ? p.z : INFINITY};
            double hi[3] = {act ? p.x : -INFINITY, act ? p.y : -INFINITY, act ? p.z : -INFINITY};
            double amax = 0.0;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                for (int off = 32; off > 0; off >>= 1) {
                    const double ol = __shfl_xor(lo[k], off, 64), oh = __shfl_xor(hi[k], off, 64);
                    lo[k] = ol < lo[k] ? ol : lo[k];
                    hi[k] = oh > hi[k] ? oh : hi[k];
                }
                amax = fmax(amax, fmax(fabs(lo[k]), fabs(hi[k])));
            }
            const double pad = 1.0001 * sqrtT + 1e-9 * amax;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                lo[k] -= pad;
                hi[k] += pad;
            }
            // a coordinate that is not finite can leave the lanes with different
            // boxes (min / max ignore NaN): no list for them
            const int nl = __ballot(act && !fin) ? -1 : collect_facets<64>(W, lo, hi, lst, fr, CAP, lane, 0);
            if (nl >= 0) {
                const CertFrame F = cert_frame(lo, hi, amax, eps2, 1.0);
                cert_list<64>(W, lst, cert, nl, F, eps2, lane);
                if (act) {
                    uint64_t mk[2];
                    int hl = -1;
                    bool sure;
                    point_list_mask(lst, nl, p, sqrtT, mk);
                    out[i] = in_envelope_cert(W, lst, cert, nl, mk, p, F, eps2, hl, sure) ? 0 : 1;
                }
                wave_sync();  // the list's last reads
            } else if (w > kListSplit && halves_help(lo, hi, kHalvePoints * 2.0 * pad)) {
                w /= 2;
                continue;
            } else {
                rest = rest || act;
            }
        }
        s += w;
        w = s & -s;
    }
    if (rest) {
        int hint = -1;
        Stats st;
        out[i] = in_envelope<F32, false>(W, p, eps2, T, sqrtT, hint, st) ? 0 : 1;
    }
    if (lstat) {
        const bool any = __ballot(rest) != 0ull;
        if (lane == 0) atomicAdd(lstat + (any ? 1 : 0), 1ull);
    }
}

// Triangles the degeneracy filter cannot settle are queued (pending[],
// *n_pending) for faces_exact_kernel, which keeps the exact predicate -- and its
// register footprint -- out of this kernel.  Capped at 128 VGPRs (4 waves
// per SIMD, a few spills): more waves in flight hide more of the traversal's
// load latency (+18% checks/s on 20 M queries against 1 M facets).
template <bool F32, bool STATS>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4, 8))) void faces_kernel(
    BvhView B, const double* __restrict__ tri9, int64_t n, double eps2, double d, double T,
    double sqrtT, uint8_t* __restrict__ out, unsigned long long* stats, unsigned* n_pending,
    int64_t* pending, const int32_t* __restrict__ order)
{
    __shared__ __align__(16) unsigned char cache[kTreeCacheBytes];
    const BvhWalk W = cache_tree_top<F32>(B, cache);
    int64_t i = xcd_block() * kBlock + threadIdx.x;
    Stats st;
    if (i < n) {
        if (order) i = order[i];
        const double* t = tri9 + 9 * i;
        if (certainly_not_collinear(t, t + 3, t + 6)) {
            out[i] = face_out_sampled<F32, STATS>(W, t, eps2, d, T, sqrtT, st) ? 1 : 0;
        } else {
            unsigned k = atomicAdd(n_pending, 1u);
            pending[k] = i;
        }
    }
    if (STATS) flush_stats(st, stats);
}

// One triangle per lane, as faces_kernel, for batches walked in Morton
// order: the wave's 64 consecutive triangles lie close together, so the wave
// lists once (collect_facets, LDS) the facets whose boxes meet the box of its
// triangles padded by more than sqrt(T), with their certificates, and tests
// its triangles against the list (faces_wave_listed) instead of walking the
// tree per sample.  Blocks of one wave: a block's LDS is free for the next one
// as soon as its wave ends.  Three waves a SIMD hold its 168 registers (four
// spill 70 of them: 1574 us a call against 1423).  3 M triangles on 246 k
// facets: 2.73 -> 1.22 ms for the kernel, with the certificates, the wider tree
// rounds of collect_facets, the rows through LDS, the split waves, the short
// blocks and the open triangles on their own lanes; the VALU is busy for some
// 40 % of it, the rest waits for the list's chain of reads.
template <bool F32, int CAP>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3, 8))) void faces_list_kernel(
    BvhView B, const double* __restrict__ tri9, int64_t n, double eps2, double d, double T_, double sqrtT,
    uint8_t* __restrict__ out, unsigned* n_pending, int64_t* pending, const int32_t* __restrict__ order,
    unsigned long long* lstat)
{
    constexpr int kWaveBytes = CAP * kCertEntryBytes;
    static_assert(CAP <= 128, "two list-mask words");
    __shared__ __align__(16) unsigned char mine[kWaveBytes];
    const BvhWalk W = walk(B);
    const int lane = threadIdx.x;
    LdsNode32W* lst = (LdsNode32W*)mine;
    LdsU32* fr = (LdsU32*)(mine + CAP * 32);  // the work lists, then the certificates
    LdsF32* cert = (LdsF32*)(mine + CAP * 32);
    int64_t i = xcd_run_block() * 64 + threadIdx.x;
    const int row = i < n ? (order ? order[i] : (int)i) : -1;
    if (i < n) i = row;
    // the wave's 64 triangles through LDS, nine lanes to a row: each line of a
    // row comes in once (nine 8-byte loads per lane, a row apart from lane to
    // lane, took 60 k of the wave's 300 k cycles)
    LdsF64* rows = (LdsF64*)mine;
    static_assert(64 * 9 * 8 <= kWaveBytes, "room for the wave's triangles");
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        const int e = 64 * k + lane, src = __shfl(row, e / 9, 64);
        rows[e] = src >= 0 ? tri9[9 * (int64_t)src + e % 9] : 0.0;
    }
    wave_sync();
    double t[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) t[k] = rows[9 * lane + k];
    wave_sync();  // read before the list takes its place
    WaveFace T;
    T.act = false;
    T.first = 0;
    T.t9 = tri9 + 9 * (int64_t)(row >= 0 ? row : 0);
    if (row >= 0) {
        const V3<double> a = ld3(t), b = ld3(t + 3), c = ld3(t + 6);
        if (!certainly_not_collinear(t, t + 3, t + 6)) {
            unsigned k = atomicAdd(n_pending, 1u);
            pending[k] = i;
        } else {
            T.act = wave_face_first(a, b, c, d, T.first);
            if (!T.act) out[i] = 1;
        }
    }
    // The lanes [s, s + w) at a time: all 64, unless their facets do not fit the
    // list -- the Morton order jumps inside the wave, say -- then its halves, down
    // to kListSplit lanes; the lanes whose facets do not fit then walk the tree,
    // all at once at the end.  (Whole waves walking it, 5.8 % of them, ran on
    // alone for half of the kernel's time.  Each last split walking it by itself
    // before the next took 7.7 ms for 1 M triangles whose envelope is three facets
    // wide, this 2.9; a kernel of its own for the lanes left, after this one,
    // costs the ordinary batch its tail: 3 M triangles 1386 -> 1646 us.)
    bool rest = false;
    for (int s = 0, w = 64; s < 64;) {
        WaveFace U = T;
        U.act = T.act && lane >= s && lane < s + w;
        if (__ballot(U.act)) {
            V3<double> a = mk3<double>(INFINITY, INFINITY, INFINITY), b = a, c = a;
            if (U.act) {
                a = ld3(T.t9);
                b = ld3(T.t9 + 3);
                c = ld3(T.t9 + 6);
            }
            const bool fin = !U.act || (is_finite(a.x) && is_finite(a.y) && is_finite(a.z) && is_finite(b.x) &&
                                        is_finite(b.y) && is_finite(b.z) && is_finite(c.x) && is_finite(c.y) &&
                                        is_finite(c.z));
            // the box of the lanes' triangles, padded
            const V3<double> l3 = mk3(fmin(a.x, fmin(b.x, c.x)), fmin(a.y, fmin(b.y, c.y)), fmin(a.z, fmin(b.z, c.z)));
            const V3<double> h3 = mk3(fmax(a.x, fmax(b.x, c.x)), fmax(a.y, fmax(b.y, c.y)), fmax(a.z, fmax(b.z, c.z)));
            double lo[3] = {l3.x, l3.y, l3.z};
            double hi[3] = {U.act ? h3.x : -INFINITY, U.act ? h3.y : -INFINITY, U.act ? h3.z : -INFINITY};
            double amax = 0.0;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                for (int off = 32; off > 0; off >>= 1) {
                    const double ol = __shfl_xor(lo[k], off, 64), oh = __shfl_xor(hi[k], off, 64);
                    lo[k] = ol < lo[k] ? ol : lo[k];
                    hi[k] = oh > hi[k] ? oh : hi[k];
                }
                amax = fmax(amax, fmax(fabs(lo[k]), fabs(hi[k])));
            }
            const double pad = 1.0001 * sqrtT + 1e-9 * amax;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                lo[k] -= pad;
                hi[k] += pad;
            }
            // a coordinate that is not finite can leave the lanes with different
            // boxes (min / max ignore NaN): no list for them
            const int nl = __ballot(!fin) ? -1 : collect_facets<64>(W, lo, hi, lst, fr, CAP, lane, 0);
            if (nl >= 0) {
                const CertFrame F = cert_frame(lo, hi, amax, eps2, d);
                face_mask_box(a, b, c, sqrtT, U.mlo, U.mhi);
                U.q[0] = cert_local(F, sel3(U.first, a, b, c));
                U.q[1] = cert_local(F, sel3(U.first, b, c, a));
                U.q[2] = cert_local(F, sel3(U.first, c, a, b));
                cert_list<64>(W, lst, cert, nl, F, eps2, lane);
                const bool o = faces_wave_listed(W, U, eps2, d, lst, cert, nl, F);
                if (U.act) out[i] = o ? 1 : 0;
                wave_sync();  // the list's last reads
            } else {
                bool halve = w > kListSplit;
                if (halve) {
                    double one = U.act ? fmax(h3.x - l3.x, fmax(h3.y - l3.y, h3.z - l3.z)) : 0.0;
                    for (int off = 32; off > 0; off >>= 1) one = fmax(one, __shfl_xor(one, off, 64));
                    halve = halves_help(lo, hi, kHalveFaces * (one + 2.0 * pad));
                }
                if (halve) {
                    w /= 2;
                    continue;
                }
                rest = rest || U.act;
            }
        }
        s += w;
        w = s & -s;
    }
    if (rest) {
        Stats st;
        out[i] = face_out_sampled<F32, false>(W, T.t9, eps2, d, T_, sqrtT, st) ? 1 : 0;
    }
    if (lstat) {
        const bool any = __ballot(rest) != 0ull;
        if (lane == 0) atomicAdd(lstat + (any ? 1 : 0), 1ull);
    }
}

// A wave per triangle, its samples spread over the lanes (face_out_wave): for
// small batches, so that few triangles with many samples each still fill the
// machine.  Same outputs as faces_kernel; triangles the degeneracy filter cannot
// settle are marked in out for faces_marked_kernel (a queue's counter would
// take a launch of its own to clear).  The tree is read from global memory
// throughout (listing through an LDS copy of its top ran
// ~5 % slower here, and only lists that do not fit walk it).
constexpr uint8_t kFacePending = 2;
constexpr int kWaveListCap = 64;
constexpr int kWaveListBytes = kWaveListCap * kCertEntryBytes;
template <bool F32>
__global__ __launch_bounds__(kBlock) void faces_wave_kernel(BvhView B, const double* __restrict__ tri9,
                                                            int64_t n, double eps2, double d,
                                                            double T, double sqrtT,
                                                            uint8_t* __restrict__ out)
{
    __shared__ __align__(16) unsigned char face_lists[(kBlock / 64) * kWaveListBytes];
    __shared__ double seg[(kBlock / 64) * kWaveSegBytes / 8];
    const BvhWalk W = walk(B);
    const int r = threadIdx.x % 64;
    const int64_t i = (xcd_block() * (int64_t)kBlock + threadIdx.x) / 64;
    if (i >= n) return;
    const double* t = tri9 + 9 * i;
    if (!certainly_not_collinear(t, t + 3, t + 6)) {
        if (r == 0) out[i] = kFacePending;
        return;
    }
    // the facets near the triangle, listed in the wave's LDS (the tree walk
    // when they do not fit or a coordinate is not finite)
    unsigned char* mine = face_lists + (threadIdx.x / 64) * kWaveListBytes;
    LdsNode32W* lst = (LdsNode32W*)mine;
    LdsU32* fr = (LdsU32*)(mine + kWaveListCap * 32);  // the work lists, then the certificates
    LdsF32* cert = (LdsF32*)(mine + kWaveListCap * 32);
    double lo[3], hi[3], amax = 0.0;
    bool fin = true;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        lo[j] = fmin(t[j], fmin(t[3 + j], t[6 + j]));
        hi[j] = fmax(t[j], fmax(t[3 + j], t[6 + j]));
        fin = fin && is_finite(t[j]) && is_finite(t[3 + j]) && is_finite(t[6 + j]);
        amax = fmax(amax, fmax(fabs(lo[j]), fabs(hi[j])));
    }
    const double pad = 1.0001 * sqrtT + 1e-9 * amax;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        lo[j] -= pad;
        hi[j] += pad;
    }
    const int nl = fin ? collect_facets<64>(W, lo, hi, lst, fr, kWaveListCap, r, 0) : -1;
    CertFrame F = {};
    if (nl >= 0) {
        F = cert_frame(lo, hi, amax, eps2, d);
        cert_list<64>(W, lst, cert, nl, F, eps2, r);
    }
    const bool o = face_out_wave<F32>(W, ld3(t), ld3(t + 3), ld3(t + 6), eps2, d, T, sqrtT, r, lst, cert, F, nl,
                                      (LdsF64*)seg + (threadIdx.x / 64) * (kWaveSegBytes / 8));
    if (r == 0) out[i] = o ? 1 : 0;
}

template <bool F32>
__global__ __launch_bounds__(kBlock) void faces_marked_kernel(BvhView B, const double* __restrict__ tri9,
                                                              int64_t n, double eps2, double d, double T,
                                                              double sqrtT, uint8_t* __restrict__ out)
{
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n || out[i] != kFacePending) return;
    Stats st;
    out[i] = face_out<F32, false>(walk(B), tri9 + 9 * i, eps2, d, T, sqrtT, st) ? 1 : 0;
}

template <bool F32>
__global__ __launch_bounds__(kBlock) void faces_exact_kernel(BvhView B,
                                                             const double* __restrict__ tri9,
                                                             double eps2, double d, double T,
                                                             double sqrtT, uint8_t* __restrict__ out,
                                                             const unsigned* n_pending,
                                                             const int64_t* pending)
{
    const unsigned cnt = *n_pending;
    Stats st;
    for (unsigned k = blockIdx.x * kBlock + threadIdx.x; k < cnt; k += gridDim.x * kBlock) {
        int64_t i = pending[k];
        out[i] = face_out<F32, false>(walk(B), tri9 + 9 * i, eps2, d, T, sqrtT, st) ? 1 : 0;
    }
}

__global__ void zero_u32(unsigned* p) { *p = 0u; }
__global__ void zero_u64x2(unsigned long long* p)
{
    p[0] = 0ull;
    p[1] = 0ull;
}

// batches at least this large are walked in Morton order of their queries
constexpr int64_t kSortMin = 1 << 16;
// face batches below this size run a wave per triangle (faces_wave_kernel)
constexpr int64_t kWaveMax = 1 << 16;
// Facets per wave list in faces_list_kernel, and the queries per facet from
// which a wave's 64 triangles (about 64 / density facets apart) fit it whole or
// in halves.  Measured against faces_kernel: 800 k triangles on 246 k facets
// (3.2 a facet) 1629 -> 1027 us with the lists, 200 k on 512 k (0.4) 1082 ->
// 2153, so sparser batches keep faces_kernel.  So do wide envelopes (reach_wide),
// and below kWideDensity queries a facet those 2.5 times less wide: eps two facets,
// 2 M triangles (8 a facet) 4156 us without lists and 4356 with them; eps one
// facet, 560 k (2.3) 1372 and 1779, 2 M (8) 3509 and 3478.  On graded surfaces
// (morton_refined) a wave's queries lie further apart in facets: 72 k facets
// shrinking tenfold, 160 k triangles (2.2) 464 and 558, 290 k (4) 591 and 503, so
// those start at kGradedDensity.
constexpr int kFaceListCap = 80;
constexpr int64_t kFaceListDensity = 2, kGradedDensity = 3, kWideDensity = 8;
// the same for points_list_kernel: 1 M points on 246 k facets (4 a facet) 593
// -> 576 us, 4 M on 72 k (56) 980 -> 829, but 300 k on 512 k (0.6) 418 -> 822;
// eps three facets, 1 M points (4 a facet) 1562 us without lists and 1774 with
// them, eps two facets, 3 M (12) 3033 and 1849
constexpr int kPointListCap = 64;
constexpr int64_t kPointListDensity = 2;

// Nearest facets.  nearest_facet's walk is a chain of some 500 dependent
// reads (2.9 ms for any batch up to 65 k points near 246 k facets, 11 ms a
// third of a radius away from them), so kNearestGroup lanes take a point
// (nearest_facet_try: lists of the facets around it).  Where they cannot be
// sure of the walk's result -- far queries, ties -- the walk runs: in the group
// itself for small batches, which have the lanes (4,096 far points 11 -> 2.2
// ms, 65 k 10.5 -> 14.7), else by nearest_rest_kernel, a point per lane.
// Points near the surface, 4,096 of them 2850 -> 39 us, 1 M 10.5 -> 3.0 ms.  A
// third of a radius off it (and seven tenths, deep inside) the group's lists are
// in vain: 40 k 10.8 -> 11.0 ms (78 -> 80), 300 k on 512 k facets 21.6 -> 25.2 (171
// -> 195), but 1 M in order 41.6 -> 31.8 (303 -> 234).  (8, 16 and 64 lanes a point
// before the order: 65, 45 and 35 us for 4,096, 6.6, 4.7 and 5.7 ms for 1 M,
// against 37 us and 3.7 ms.)
constexpr int kNearestGroup = 32;
constexpr int kNearestCap = 64;  // facets listed per group
constexpr int64_t kNearestWalkMax = 1 << 15;
template <bool WALK>
__global__ __launch_bounds__(kBlock) void nearest_kernel(BvhView B, const double* __restrict__ p3,
                                                         int64_t n, double* __restrict__ cp3,
                                                         double* __restrict__ d2out,
                                                         int32_t* __restrict__ fout,
                                                         const int32_t* __restrict__ order, int64_t base)
{
    constexpr int G = kNearestGroup;
    __shared__ __align__(16) unsigned char cache[kPointCacheBytes];
    __shared__ __align__(16) unsigned char lists[(kBlock / G) * kNearestCap * 40];
    const BvhWalk W = cache_tree_top<false, kPointCacheBytes>(B, cache);
    const int gl = threadIdx.x % G, gbase = (threadIdx.x % 64) - gl;
    int64_t i = base + xcd_block() * (int64_t)(kBlock / G) + threadIdx.x / G;
    if (i >= n) return;
    if (order) i = order[i];
    unsigned char* mine = lists + (threadIdx.x / G) * (kNearestCap * 40);
    LdsNode32W* lst = (LdsNode32W*)mine;
    LdsU32* fr = (LdsU32*)(mine + kNearestCap * 32);
    V3<double> np;
    double sq;
    const int f = WALK ? nearest_facet_group<G>(W, ld3(p3 + 3 * i), np, sq, lst, fr, kNearestCap, gl, gbase)
                       : nearest_facet_try<G>(W, ld3(p3 + 3 * i), np, sq, lst, fr, kNearestCap, gl, gbase);
    if (gl != 0) return;
    fout[i] = f;
    if (!WALK && f < 0) return;
    cp3[3 * i + 0] = np.x;
    cp3[3 * i + 1] = np.y;
    cp3[3 * i + 2] = np.z;
    d2out[i] = sq;
}

// the points nearest_kernel<false> left (facet -1), one per lane
__global__ __launch_bounds__(kBlock) void nearest_rest_kernel(BvhView B, const double* __restrict__ p3,
                                                              int64_t n, double* __restrict__ cp3,
                                                              double* __restrict__ d2out,
                                                              int32_t* __restrict__ fout,
                                                              const int32_t* __restrict__ order)
{
    int64_t i = xcd_block() * kBlock + threadIdx.x;
    if (i < n && order) i = order[i];
    __shared__ __align__(16) unsigned char cache[kPointCacheBytes];
    if (!__syncthreads_or(i < n && fout[i] < 0)) return;
    const BvhWalk W = cache_tree_top<false, kPointCacheBytes>(B, cache);
    if (i >= n || fout[i] >= 0) return;
    V3<double> np;
    double sq;
    fout[i] = nearest_facet(W, ld3(p3 + 3 * i), np, sq);
    cp3[3 * i + 0] = np.x;
    cp3[3 * i + 1] = np.y;
    cp3[3 * i + 2] = np.z;
    d2out[i] = sq;
}

__global__ __launch_bounds__(kBlock) void sample_count_kernel(const double* __restrict__ tri9,
                                                              int64_t n, double d,
                                                              int64_t* __restrict__ counts)
{
    int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const double* t = tri9 + 9 * i;
    int64_t k = 0;
    for_each_sample(ld3(t), ld3(t + 3), ld3(t + 6), d, [&](V3<double>) {
        ++k;
        return false;
    });
    counts[i] = k;
}

__global__ __launch_bounds__(kBlock) void sample_write_kernel(const double* __restrict__ tri9,
                                                              int64_t n, double d,
                                                              const int64_t* __restrict__ offsets,
                                                              int64_t total,
                                                              double* __restrict__ pts)
{
    int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const double* t = tri9 + 9 * i;
    int64_t k = offsets[i];
    for_each_sample(ld3(t), ld3(t + 3), ld3(t + 6), d, [&](V3<double> s) {
        if (k >= 0 && k < total) {
            pts[3 * k + 0] = s.x;
            pts[3 * k + 1] = s.y;
            pts[3 * k + 2] = s.z;
        }
        ++k;
        return false;
    });
}

// ---- host-side build --------------------------------------------------
inline uint64_t spread3(uint64_t v)
{
    v &= 0x1FFFFF;
    v = (v | v << 32) & 0x1F00000000FFFFull;
    v = (v | v << 16) & 0x1F0000FF0000FFull;
    v = (v | v << 8) & 0x100F00F00F00F00Full;
    v = (v | v << 4) & 0x10C30C30C30C30C3ull;
    v = (v | v << 2) & 0x1249249249249249ull;
    return v;
}

int64_t max_node(int64_t n, int64_t b, int64_t e)
{
    if (b + 1 == e) return n;
    int64_t m = b + (e - b) / 2;
    return std::max(max_node(2 * n, b, m), max_node(2 * n + 1, m, e));
}

void fill(std::vector<BvhNode64>& nodes, const std::vector<double>& tri, int64_t n, int64_t b,
          int64_t e, int depth, int& maxdepth)
{
    maxdepth = std::max(maxdepth, depth);
    BvhNode64& N = nodes[n];
    if (b + 1 == e) {
        const double* t = &tri[9 * b];
        for (int c = 0; c < 3; ++c) {
            N.lo[c] = N.hi[c] = t[c];
            for (int k = 1; k < 3; ++k) {
                N.lo[c] = std::min(N.lo[c], t[3 * k + c]);
                N.hi[c] = std::max(N.hi[c], t[3 * k + c]);
            }
        }
        N.leaf = (int32_t)b;
        return;
    }
    int64_t m = b + (e - b) / 2;
    fill(nodes, tri, 2 * n, b, m, depth + 1, maxdepth);
    fill(nodes, tri, 2 * n + 1, m, e, depth + 1, maxdepth);
    const BvhNode64& L = nodes[2 * n];
    const BvhNode64& R = nodes[2 * n + 1];
    for (int c = 0; c < 3; ++c) {
        N.lo[c] = std::min(L.lo[c], R.lo[c]);
        N.hi[c] = std::max(L.hi[c], R.hi[c]);
    }
    N.leaf = -1;
}

float round_down(double v)
{
    float f = (float)v;
    if ((double)f > v) f = std::nextafter(f, -INFINITY);
    return f;
}
float round_up(double v)
{
    float f = (float)v;
    if ((double)f < v) f = std::nextafter(f, INFINITY);
    return f;
}

}  // namespace
}  // namespace twg

using namespace twg;

// Surfaces from this size on are built on the device (build.hip), smaller ones
// on the host: 64 facets take 59 us on the host and 169 on the device, 512 take
// 187 and 180, 5,120 take 2.0 ms and 0.32, 246,420 take 121 ms and 0.96.  The host
// also builds those whose working memory the device does not have.
constexpr int64_t kDeviceBuildMin = 512;

extern "C" {

int twg_bvh_build(twg_ctx* ctx, const double* V, int64_t nv, const int32_t* F, int64_t nf,
                  twg_bvh** out)
{
    TWG_REQUIRE(ctx && out, "twg_bvh_build: NULL argument");
    TWG_REQUIRE(nf >= 1 && nv >= 1 && V && F, "twg_bvh_build: empty surface");
    TWG_REQUIRE(nf < (int64_t(1) << 30), "twg_bvh_build: too many facets (%lld)", (long long)nf);
    if (int r = bind(ctx)) return r;
    if (nf >= kDeviceBuildMin && nv < (int64_t(1) << 31)) {
        std::unique_ptr<twg_bvh, int (*)(twg_bvh*)> B(new twg_bvh(), twg_bvh_destroy);
        B->device = ctx->device;
        B->nf = nf;
        int64_t bad = -1;
        const int r = bvh_build_device(ctx, V, nv, F, nf, B.get(), &bad);
        if (r && r != TWG_ENOMEM) return r;
        if (!r) {
            TWG_REQUIRE(bad < 0, "twg_bvh_build: facet %lld has vertex id %d outside [0, %lld)",
                        (long long)(bad / 3), F[bad], (long long)nv);
            *out = B.release();
            return TWG_OK;
        }
        (void)hipGetLastError();
    }
    for (int64_t f = 0; f < 3 * nf; ++f)
        TWG_REQUIRE(F[f] >= 0 && F[f] < nv, "twg_bvh_build: facet %lld has vertex id %d outside [0, %lld)",
                    (long long)(f / 3), F[f], (long long)nv);
    // Morton order of facet centroids
    std::vector<double> cen(3 * nf);
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int64_t f = 0; f < nf; ++f)
        for (int c = 0; c < 3; ++c) {
            double v = (V[3 * F[3 * f] + c] + V[3 * F[3 * f + 1] + c] + V[3 * F[3 * f + 2] + c]) / 3.0;
            cen[3 * f + c] = v;
            lo[c] = std::min(lo[c], v);
            hi[c] = std::max(hi[c], v);
        }
    std::vector<std::pair<uint64_t, int32_t>> key(nf);
    for (int64_t f = 0; f < nf; ++f) {
        uint64_t k = 0;
        for (int c = 0; c < 3; ++c) {
            double span = hi[c] - lo[c];
            double q = span > 0 ? (cen[3 * f + c] - lo[c]) / span * 2097152.0 : 0.0;
            uint64_t qi = q <= 0 ? 0 : (q >= 2097151.0 ? 2097151 : (uint64_t)q);
            k |= spread3(qi) << c;
        }
        key[f] = {k, (int32_t)f};
    }
    std::stable_sort(key.begin(), key.end(),
                     [](const std::pair<uint64_t, int32_t>& a, const std::pair<uint64_t, int32_t>& b) {
                         return a.first < b.first;
                     });
    twg_bvh* B = new twg_bvh();
    B->device = ctx->device;
    B->nf = nf;
    B->order.resize(nf);
    std::vector<double> tri(9 * nf);
    double rmax = 0.0;
    for (int64_t b = 0; b < nf; ++b) {
        int32_t f = key[b].second;
        B->order[b] = f;
        for (int k = 0; k < 3; ++k)
            for (int c = 0; c < 3; ++c) tri[9 * b + 3 * k + c] = V[3 * F[3 * f + k] + c];
        for (int k = 0; k < 3; ++k) {
            const double* a = &tri[9 * b + 3 * k];
            const double* e = &tri[9 * b + 3 * ((k + 1) % 3)];
            double l = std::sqrt((a[0] - e[0]) * (a[0] - e[0]) + (a[1] - e[1]) * (a[1] - e[1]) +
                                 (a[2] - e[2]) * (a[2] - e[2]));
            rmax = std::max(rmax, l);
        }
    }
    B->rmax = rmax;
    for (int c = 0; c < 3; ++c) B->side = std::max(B->side, hi[c] - lo[c]);
    for (int j = 0; j < 2; ++j)
        for (int64_t b = 0; b + kCrowd[j] < nf; ++b)
            for (int l = crowd_level(key[b].first, key[b + kCrowd[j]].first); l >= 0; --l) B->crowded[j][l]++;
    B->nnode = max_node(1, 0, nf) + 1;
    std::vector<BvhNode64> nodes(B->nnode);
    for (auto& N : nodes) {
        for (int c = 0; c < 3; ++c) {
            N.lo[c] = INFINITY;
            N.hi[c] = -INFINITY;
        }
        N.leaf = -2;
        N.pad[0] = N.pad[1] = N.pad[2] = 0;
    }
    int depth = 0;
    fill(nodes, tri, 1, 0, nf, 0, depth);
    B->depth = depth;
    for (int c = 0; c < 3; ++c) {
        B->lo[c] = nodes[1].lo[c];
        B->hi[c] = nodes[1].hi[c];
    }
    if (depth > 30) {
        delete B;
        set_error("twg_bvh_build: tree depth %d exceeds 30", depth);
        return TWG_EINVAL;
    }
    std::vector<BvhNode32> n32(B->nnode);
    for (int64_t i = 0; i < B->nnode; ++i) {
        for (int c = 0; c < 3; ++c) {
            n32[i].lo[c] = round_down(nodes[i].lo[c]);
            n32[i].hi[c] = round_up(nodes[i].hi[c]);
        }
        n32[i].leaf = nodes[i].leaf;
        n32[i].pad = 0;
    }
    int r = bind(ctx);
    hipError_t e = hipSuccess;
    auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
    const size_t b64 = up(sizeof(BvhNode64) * B->nnode), b32 = up(sizeof(BvhNode32) * B->nnode),
                 btri = up(sizeof(double) * 9 * nf);
    if (!r) e = hipMalloc(&B->mem, b64 + b32 + btri);
    if (!r && e == hipSuccess) {
        char* m = static_cast<char*>(B->mem);
        B->node64 = reinterpret_cast<BvhNode64*>(m);
        B->node32 = reinterpret_cast<BvhNode32*>(m + b64);
        B->tri = reinterpret_cast<double*>(m + b64 + b32);
        e = hipMemcpy(B->node64, nodes.data(), sizeof(BvhNode64) * B->nnode, hipMemcpyHostToDevice);
    }
    if (!r && e == hipSuccess)
        e = hipMemcpy(B->node32, n32.data(), sizeof(BvhNode32) * B->nnode, hipMemcpyHostToDevice);
    if (!r && e == hipSuccess)
        e = hipMemcpy(B->tri, tri.data(), sizeof(double) * 9 * nf, hipMemcpyHostToDevice);
    if (r || e != hipSuccess) {
        if (B->mem) (void)hipFree(B->mem);
        delete B;
        return r ? r : hip_fail(e, "twg_bvh_build upload", __FILE__, __LINE__);
    }
    *out = B;
    return TWG_OK;
}

int twg_bvh_destroy(twg_bvh* B)
{
    if (!B) return TWG_OK;
    (void)hipSetDevice(B->device);
    (void)hipDeviceSynchronize();
    if (B->mem) (void)hipFree(B->mem);
    delete B;
    return TWG_OK;
}

int twg_bvh_info(const twg_bvh* B, int64_t* nf, int64_t* nnode, int32_t* depth, double* rmax)
{
    TWG_REQUIRE(B != nullptr, "twg_bvh_info: NULL bvh");
    if (nf) *nf = B->nf;
    if (nnode) *nnode = B->nnode;
    if (depth) *depth = B->depth;
    if (rmax) *rmax = B->rmax;
    return TWG_OK;
}

int twg_bvh_facet_order(const twg_bvh* B, int32_t* order)
{
    TWG_REQUIRE(B && order, "twg_bvh_facet_order: NULL argument");
    std::memcpy(order, B->order.data(), sizeof(int32_t) * B->nf);
    return TWG_OK;
}

static int check_env(twg_ctx* ctx, const twg_bvh* B, const void* in, int64_t n, const void* out,
                     double eps2, int precision, const char* fn)
{
    TWG_REQUIRE(ctx && B, "%s: NULL ctx or bvh", fn);
    TWG_REQUIRE(n >= 0, "%s: negative size", fn);
    TWG_REQUIRE(n == 0 || (in && out), "%s: NULL array", fn);
    TWG_REQUIRE(eps2 >= 0 && std::isfinite(eps2), "%s: bad eps2", fn);
    TWG_REQUIRE(precision == TWG_FP64 || precision == TWG_MIXED, "%s: bad precision %d", fn,
                precision);
    TWG_REQUIRE(B->device == ctx->device, "%s: bvh lives on device %d, ctx on %d", fn, B->device,
                ctx->device);
    return TWG_OK;
}

int twg_envelope_points(twg_ctx* ctx, const twg_bvh* B, const double* p3, int64_t n, double eps2,
                        int precision, uint8_t* out, unsigned long long* stats)
{
    if (int r = check_env(ctx, B, p3, n, out, eps2, precision, "twg_envelope_points")) return r;
    if (n == 0) return TWG_OK;
    if (int r = bind(ctx)) return r;
    double T = bvh_prune_threshold(B, eps2), sT = std::sqrt(T);
    dim3 g(grid_for(n)), b(kBlock);
    BvhView v = bvh_view(B);
    const bool wide = reach_wide(B, 2.0 * sT);
    const bool group = !stats && (n < kSortMin || (n < kPointGroupMax && n < kPointGroupDensity * B->nf)) &&
                       (n < kPointGroupWide || !wide);
    const int32_t* order = nullptr;
    if (n >= kSortMin && !group)
        if (int r = morton_order(ctx, 1, p3, n, 3, B, &order)) return r;
    if (group) {
        const dim3 gg(grid_for(n * kPointGroup));
        if (precision == TWG_FP64) hipLaunchKernelGGL(points_group_kernel<false>, gg, b, 0, ctx->cur, v, p3, n, eps2, T, sT, out);
        else hipLaunchKernelGGL(points_group_kernel<true>, gg, b, 0, ctx->cur, v, p3, n, eps2, T, sT, out);
    } else if (order && !stats && n >= (wide ? kWideDensity : kPointListDensity) * B->nf) {
        if (precision == TWG_FP64)
            hipLaunchKernelGGL((points_list_kernel<false, kPointListCap>), dim3(4 * grid_for(n)), dim3(64), 0, ctx->cur, v, p3, n, eps2, T, sT, out, order, ctx->list_stats_on ? ctx->list_stats : nullptr);
        else
            hipLaunchKernelGGL((points_list_kernel<true, kPointListCap>), dim3(4 * grid_for(n)), dim3(64), 0, ctx->cur, v, p3, n, eps2, T, sT, out, order, ctx->list_stats_on ? ctx->list_stats : nullptr);
    } else if (precision == TWG_FP64) {
        if (stats) hipLaunchKernelGGL((points_kernel<false, true>), g, b, 0, ctx->cur, v, p3, n, eps2, T, sT, out, stats, order);
        else hipLaunchKernelGGL((points_kernel<false, false>), g, b, 0, ctx->cur, v, p3, n, eps2, T, sT, out, stats, order);
    } else {
        if (stats) hipLaunchKernelGGL((points_kernel<true, true>), g, b, 0, ctx->cur, v, p3, n, eps2, T, sT, out, stats, order);
        else hipLaunchKernelGGL((points_kernel<true, false>), g, b, 0, ctx->cur, v, p3, n, eps2, T, sT, out, stats, order);
    }
    TWG_LAUNCHED();
    return TWG_OK;
}

int twg_envelope_faces(twg_ctx* ctx, const twg_bvh* B, const double* tri9, int64_t n, double eps2,
                       double sampling_dist, int precision, uint8_t* out,
                       unsigned long long* stats)
{
    if (int r = check_env(ctx, B, tri9, n, out, eps2, precision, "twg_envelope_faces")) return r;
    TWG_REQUIRE(sampling_dist > 0 && std::isfinite(sampling_dist),
                "twg_envelope_faces: sampling_dist must be positive");
    if (n == 0) return TWG_OK;
    if (int r = bind(ctx)) return r;
    double T = bvh_prune_threshold(B, eps2), sT = std::sqrt(T);
    dim3 g(grid_for(n)), b(kBlock);
    BvhView v = bvh_view(B);
    if (n < kWaveMax && !stats) {
        const dim3 gw(grid_for(n * 64));
        if (precision == TWG_FP64) {
            hipLaunchKernelGGL(faces_wave_kernel<false>, gw, b, 0, ctx->cur, v, tri9, n, eps2, sampling_dist, T, sT, out);
            TWG_LAUNCHED();
            hipLaunchKernelGGL(faces_marked_kernel<false>, g, b, 0, ctx->cur, v, tri9, n, eps2, sampling_dist, T, sT, out);
        } else {
            hipLaunchKernelGGL(faces_wave_kernel<true>, gw, b, 0, ctx->cur, v, tri9, n, eps2, sampling_dist, T, sT, out);
            TWG_LAUNCHED();
            hipLaunchKernelGGL(faces_marked_kernel<true>, g, b, 0, ctx->cur, v, tri9, n, eps2, sampling_dist, T, sT, out);
        }
        TWG_LAUNCHED();
        return TWG_OK;
    }
    if (int r = ensure_scratch(ctx, 256 + sizeof(int64_t) * (size_t)n)) return r;
    unsigned* n_pending = (unsigned*)ctx->scratch.p;
    int64_t* pending = (int64_t*)((char*)ctx->scratch.p + 256);
    const int32_t* order = nullptr;
    if (n >= kSortMin)
        if (int r = morton_order(ctx, 1, tri9, n, 9, B, &order)) return r;
    hipLaunchKernelGGL(zero_u32, dim3(1), dim3(1), 0, ctx->cur, n_pending);
    TWG_LAUNCHED();
    const bool wide = reach_wide(B, (n < kWideDensity * B->nf ? 5.0 : 2.0) * sT);
    const int64_t density = morton_refined(B, n) ? kGradedDensity : kFaceListDensity;
    if (order && !stats && !wide && n >= density * B->nf) {
        if (precision == TWG_FP64)
            hipLaunchKernelGGL((faces_list_kernel<false, kFaceListCap>), dim3(4 * grid_for(n)), dim3(64), 0, ctx->cur, v, tri9, n, eps2, sampling_dist, T, sT, out, n_pending, pending, order, ctx->list_stats_on ? ctx->list_stats : nullptr);
        else
            hipLaunchKernelGGL((faces_list_kernel<true, kFaceListCap>), dim3(4 * grid_for(n)), dim3(64), 0, ctx->cur, v, tri9, n, eps2, sampling_dist, T, sT, out, n_pending, pending, order, ctx->list_stats_on ? ctx->list_stats : nullptr);
    } else if (precision == TWG_FP64) {
        if (stats) hipLaunchKernelGGL((faces_kernel<false, true>), g, b, 0, ctx->cur, v, tri9, n, eps2, sampling_dist, T, sT, out, stats, n_pending, pending, order);
        else hipLaunchKernelGGL((faces_kernel<false, false>), g, b, 0, ctx->cur, v, tri9, n, eps2, sampling_dist, T, sT, out, stats, n_pending, pending, order);
    } else {
        if (stats) hipLaunchKernelGGL((faces_kernel<true, true>), g, b, 0, ctx->cur, v, tri9, n, eps2, sampling_dist, T, sT, out, stats, n_pending, pending, order);
        else hipLaunchKernelGGL((faces_kernel<true, false>), g, b, 0, ctx->cur, v, tri9, n, eps2, sampling_dist, T, sT, out, stats, n_pending, pending, order);
    }
    TWG_LAUNCHED();
    unsigned eg = (unsigned)std::min<int64_t>(grid_for(n), 64);
    if (precision == TWG_FP64)
        hipLaunchKernelGGL((faces_exact_kernel<false>), dim3(eg), b, 0, ctx->cur, v, tri9, eps2, sampling_dist, T, sT, out, n_pending, pending);
    else
        hipLaunchKernelGGL((faces_exact_kernel<true>), dim3(eg), b, 0, ctx->cur, v, tri9, eps2, sampling_dist, T, sT, out, n_pending, pending);
    TWG_LAUNCHED();
    return TWG_OK;
}

int twg_ctx_list_stats(twg_ctx* ctx, int enable, unsigned long long* out)
{
    TWG_REQUIRE(ctx != nullptr, "twg_ctx_list_stats: ctx is NULL");
    if (int r = bind(ctx)) return r;
    if (enable) {
        if (!ctx->list_stats) TWG_HIP(hipMalloc(&ctx->list_stats, 2 * sizeof(unsigned long long)));
        hipLaunchKernelGGL(zero_u64x2, dim3(1), dim3(1), 0, ctx->cur, ctx->list_stats);
        TWG_LAUNCHED();
        ctx->list_stats_on = true;
        return TWG_OK;
    }
    unsigned long long h[2] = {0, 0};
    if (ctx->list_stats) {
        TWG_HIP(hipStreamSynchronize(ctx->cur));
        TWG_HIP(hipMemcpy(h, ctx->list_stats, sizeof h, hipMemcpyDeviceToHost));
    }
    ctx->list_stats_on = false;
    if (out) {
        out[0] = h[0];
        out[1] = h[1];
    }
    return TWG_OK;
}

int twg_nearest_points(twg_ctx* ctx, const twg_bvh* B, const double* p3, int64_t n, double* cp3,
                       double* d2, int32_t* facet)
{
    if (int r = check_env(ctx, B, p3, n, cp3, 0.0, TWG_FP64, "twg_nearest_points")) return r;
    TWG_REQUIRE(n == 0 || (d2 && facet), "twg_nearest_points: NULL output");
    if (n == 0) return TWG_OK;
    if (int r = bind(ctx)) return r;
    const dim3 b(kBlock);
    BvhView v = bvh_view(B);
    const int32_t* order = nullptr;
    // (a captured graph walks the points as they come, and so does a call that
    // finds no memory for their order)
    if (n >= kSortMin && n < (int64_t(1) << 31) && !capturing(ctx)) {
        const int r = morton_order(ctx, 2, p3, n, 3, B, &order);
        if (r && r != TWG_ENOMEM) return r;
        if (r) (void)hipGetLastError();
    }
    constexpr int64_t kPart = 1 << 26;  // a launch holds fewer than 2^32 threads
    for (int64_t at = 0; at < n; at += kPart) {
        const dim3 g(grid_for(std::min(n - at, kPart) * kNearestGroup));
        if (n < kNearestWalkMax)
            hipLaunchKernelGGL(nearest_kernel<true>, g, b, 0, ctx->cur, v, p3, n, cp3, d2, facet, order, at);
        else
            hipLaunchKernelGGL(nearest_kernel<false>, g, b, 0, ctx->cur, v, p3, n, cp3, d2, facet, order, at);
        TWG_LAUNCHED();
    }
    if (n < kNearestWalkMax) return TWG_OK;
    // (walks far from the surface gain nothing from the order below some 250 k
    // points: 65 k 10.5 ms without and 12.1 with it, 1 M 44 and 31.  At 300 k it
    // depends: a third of a radius outside 246 k facets 15.9 and 16.3, a tenth
    // inside 11.2 and 9.1, outside 5 k facets 3.1 and 2.2)
    hipLaunchKernelGGL(nearest_rest_kernel, dim3(grid_for(n)), b, 0, ctx->cur, v, p3, n, cp3, d2, facet,
                       n < (1 << 18) ? nullptr : order);
    TWG_LAUNCHED();
    return TWG_OK;
}

int twg_sample_count(twg_ctx* ctx, const double* tri9, int64_t n, double d, int64_t* counts)
{
    TWG_REQUIRE(ctx != nullptr, "twg_sample_count: ctx is NULL");
    TWG_REQUIRE(n >= 0 && (n == 0 || (tri9 && counts)), "twg_sample_count: bad arrays");
    TWG_REQUIRE(d > 0 && std::isfinite(d), "twg_sample_count: d must be positive");
    if (n == 0) return TWG_OK;
    if (int r = bind(ctx)) return r;
    hipLaunchKernelGGL(sample_count_kernel, dim3(grid_for(n)), dim3(kBlock), 0, ctx->cur, tri9, n,
                       d, counts);
    TWG_LAUNCHED();
    return TWG_OK;
}

int twg_sample_write(twg_ctx* ctx, const double* tri9, int64_t n, double d,
                     const int64_t* offsets, int64_t total, double* pts)
{
    TWG_REQUIRE(ctx != nullptr, "twg_sample_write: ctx is NULL");
    TWG_REQUIRE(n >= 0 && total >= 0 && (n == 0 || (tri9 && offsets && (total == 0 || pts))),
                "twg_sample_write: bad arrays");
    TWG_REQUIRE(d > 0 && std::isfinite(d), "twg_sample_write: d must be positive");
    if (n == 0) return TWG_OK;
    if (int r = bind(ctx)) return r;
    hipLaunchKernelGGL(sample_write_kernel, dim3(grid_for(n)), dim3(kBlock), 0, ctx->cur, tri9, n,
                       d, offsets, total, pts);
    TWG_LAUNCHED();
    return TWG_OK;
}

}  // extern "C"
