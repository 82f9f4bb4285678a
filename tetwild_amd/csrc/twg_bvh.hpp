// twg_bvh.hpp -- device AABB tree of the envelope surface and its traversals
// (shared by the envelope kernels and the smoothing kernel).
//
// Tree: MeshFacetsAABBWithEps's implicit layout (src/tetwild/geogram/
// mesh_AABB.cpp:356-379): root 1, children 2n and 2n+1, facet range split at
// b + (e-b)/2, one facet per leaf, facets in Morton order.  Node n is a 64-byte
// record (FP64 box + leaf facet id) so that the two children of a node -- the
// pair every traversal step reads -- are one 128-byte line; the mixed path
// reads a 32-byte FP32 copy of the boxes (rounded outward) instead.
//
// Decision: a sample p is in the envelope iff some facet f has
// d2(p, f) <= eps_2 (d2 = the FP64 Eberly distance, bit-identical to the host
// restatement).  The traversal prunes a box only when its squared distance
// exceeds eps_2 by a margin larger than the rounding error of any facet
// distance inside it, so the result does not depend on traversal order, on
// the facet-hint shortcut (src/tetwild/LocalOperations.cpp:1078-1098), or on
// FP32 boxes.  The traversal is stackless (a bit per tree level marks a
// pending far child).
#pragma once

#include <vector>

#include "twg_geom.hpp"

struct BvhNode64 {
    double lo[3];
    double hi[3];
    int32_t leaf;  // facet position for leaves, -1 internal
    int32_t pad[3];
};
struct BvhNode32 {
    float lo[3];
    float hi[3];
    int32_t leaf;
    int32_t pad;
};
static_assert(sizeof(BvhNode64) == 64, "node64");
static_assert(sizeof(BvhNode32) == 32, "node32");

// How the facets crowd, from their 63-bit Morton codes: the dispatch of query
// batches reads it (morton_bits, reach_wide); results never depend on it
constexpr int kCrowdLevels = 22;
constexpr int kCrowd[2] = {24, 48};

// levels at which two codes fall into the same cell
TWG_HD int crowd_level(uint64_t a, uint64_t b) { return a == b ? kCrowdLevels - 1 : (__builtin_clzll(a ^ b) - 1) / 3; }

struct twg_bvh {
    int device = 0;
    double lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};  // root box
    int64_t nf = 0, nnode = 0;
    int depth = 0;
    double rmax = 0.0;
    // crowded[j][l]: facets past the first kCrowd[j] of their cell l times
    // halved, the cell of 0 halvings being the cube of side `side` about the
    // facets' centroids
    int64_t crowded[2][kCrowdLevels] = {};
    double side = 0.0;
    BvhNode64* node64 = nullptr;
    BvhNode32* node32 = nullptr;
    double* tri = nullptr;  // nf x 9, tree order
    std::vector<int32_t> order;  // tree position -> caller's facet id
    void* mem = nullptr;         // the one allocation behind the three arrays
};

namespace twg {

// node records in LDS (address space 3): typed so that the compiler emits LDS
// reads for them (a generic pointer would turn every node read into a flat load)
typedef __attribute__((address_space(3))) const BvhNode64 LdsNode64;
typedef __attribute__((address_space(3))) const BvhNode32 LdsNode32;

// field-wise copies out of LDS (a whole-struct assignment across address
// spaces does not compile)
__device__ __forceinline__ BvhNode32 from_lds(LdsNode32* p)
{
    BvhNode32 r;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        r.lo[k] = p->lo[k];
        r.hi[k] = p->hi[k];
    }
    r.leaf = p->leaf;
    return r;
}
__device__ __forceinline__ BvhNode64 from_lds(LdsNode64* p)
{
    BvhNode64 r;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        r.lo[k] = p->lo[k];
        r.hi[k] = p->hi[k];
    }
    r.leaf = p->leaf;
    return r;
}

// What kernels receive (by value, as a kernel argument or inside one): global
// pointers and sizes only, so that the host and device layouts agree.
struct BvhView {
    const BvhNode64* __restrict__ n64;
    const BvhNode32* __restrict__ n32;
    const double* __restrict__ tri;
    int64_t nf;
    int64_t nnode;  // node slots (array length)
};
static_assert(sizeof(BvhView) == 40, "BvhView: kernel-argument layout");

// What the traversals read: the view plus an optional copy of the top of the
// tree in LDS (node slots [0, ncache), the levels every traversal walks
// first; ncache = 0: none).  LDS pointers are 32-bit in device code and 64-bit
// in the host pass, so a walker is made inside a kernel and never crosses into
// a kernel argument.
struct BvhWalk {
    const BvhNode64* __restrict__ n64;
    const BvhNode32* __restrict__ n32;
    const double* __restrict__ tri;
    int64_t nf;
    int64_t nnode;
    LdsNode64* c64;
    LdsNode32* c32;
    int64_t ncache;
    // which copy holds the cached slots (an LDS pointer cannot say: offset 0,
    // where the copy may sit, is also its null value)
    bool top64;
};

// a walker that reads every node from global memory
__device__ __forceinline__ BvhWalk walk(const BvhView& B)
{
    BvhWalk w;
    w.n64 = B.n64;
    w.n32 = B.n32;
    w.tri = B.tri;
    w.nf = B.nf;
    w.nnode = B.nnode;
    w.c64 = nullptr;
    w.c32 = nullptr;
    w.ncache = 0;
    w.top64 = false;
    return w;
}

// bytes of the per-block LDS copy of the top of the tree: 1024 FP32 nodes
// (10 levels) or 512 FP64 nodes (9 levels)
constexpr int kTreeCacheBytes = 32768;

// Every thread of the block calls this once, before any traversal: copies
// node slots [0, ncache) of the tree (FP32 or FP64 records, BYTES bytes at
// most) into cache and returns a walker that reads them from there.
template <bool F32, int BYTES = kTreeCacheBytes>
__device__ __forceinline__ BvhWalk cache_tree_top(const BvhView& B, void* cache)
{
    static_assert(BYTES % 128 == 0, "cache size: an even number of FP64 nodes");
    const int64_t per = BYTES / (F32 ? (int64_t)sizeof(BvhNode32) : (int64_t)sizeof(BvhNode64));
    const int64_t nc = B.nnode < per ? B.nnode : per;
    const uint4* src = F32 ? reinterpret_cast<const uint4*>(B.n32) : reinterpret_cast<const uint4*>(B.n64);
    uint4* dst = static_cast<uint4*>(cache);
    const int64_t chunks = nc * (F32 ? (int64_t)sizeof(BvhNode32) : (int64_t)sizeof(BvhNode64)) / 16;
    for (int64_t k = threadIdx.x; k < chunks; k += blockDim.x) dst[k] = src[k];
    __syncthreads();
    BvhWalk w = walk(B);
    if (F32) w.c32 = (LdsNode32*)cache;
    else w.c64 = (LdsNode64*)cache;
    w.ncache = nc;
    w.top64 = !F32;
    return w;
}

// the two children c, c + 1 (same level: both cached or neither)
__device__ __forceinline__ void load_pair(const BvhWalk& B, int64_t c, BvhNode32& L, BvhNode32& R)
{
    if (c < B.ncache) {
        L = from_lds(B.c32 + c);
        R = from_lds(B.c32 + c + 1);
    } else {
        L = B.n32[c];
        R = B.n32[c + 1];
    }
}

__device__ __forceinline__ void load_pair(const BvhWalk& B, int64_t c, BvhNode64& L, BvhNode64& R)
{
    if (c < B.ncache) {
        L = from_lds(B.c64 + c);
        R = from_lds(B.c64 + c + 1);
    } else {
        L = B.n64[c];
        R = B.n64[c + 1];
    }
}

__device__ __forceinline__ V3<double> ld3(const double* p) { return mk3(p[0], p[1], p[2]); }

__device__ __forceinline__ double facet_d2(const BvhWalk& B, int f, V3<double> p)
{
    const double* t = B.tri + 9 * (int64_t)f;
    V3<double> cp;
    return point_tri_d2<double, false>(p, ld3(t), ld3(t + 3), ld3(t + 6), cp);
}

struct Stats {
    unsigned long long samples = 0, traversals = 0, boxes = 0, leaves = 0;
};

// Tf: FP32 pruning threshold, conservative for the rounding of p to FP32 and
// of the FP32 box distance (see the header comment of this file).
__device__ __forceinline__ float f32_threshold(V3<double> p, double sqrtT)
{
    double pm = fmax(fabs(p.x), fmax(fabs(p.y), fabs(p.z)));
    double ep = 2.0e-7 * pm;
    double t = (sqrtT + ep) * (sqrtT + ep) * (1.0 + 0x1p-19);
    float tf = (float)t;
    if ((double)tf < t) tf = u2f32(f2u(tf) + 1u);  // t > 0: next float up
    return tf;
}

// Levels above the hint facet's leaf whose subtree is searched first when
// the hint itself misses: consecutive samples of a triangle usually move to a
// nearby facet, which lies in that subtree.  Measured on 20 M query triangles
// against 1 M facets: 3 / 5 / 7 / 10 / 12 levels gave 500 / 513 / 525 / 542 /
// 539 M checks/s.
constexpr int kHintLevels = 10;

// the implicit tree's node holding facet position b: the median splits of
// the tree's build (b + (e - b) / 2), integer work only
__device__ __forceinline__ int64_t leaf_node(int64_t nf, int64_t b)
{
    int64_t n = 1, lo = 0, hi = nf;
    while (hi - lo > 1) {
        const int64_t m = lo + (hi - lo) / 2;
        if (b < m) {
            n = 2 * n;
            hi = m;
        } else {
            n = 2 * n + 1;
            lo = m;
        }
    }
    return n;
}

// SUBTREE: after a hint miss, search the hint's ancestor subtree first
template <bool F32, bool STATS, bool SUBTREE = true>
__device__ bool in_envelope(const BvhWalk& B, V3<double> p, double eps2, double T, double sqrtT,
                            int& hint, Stats& st)
{
    int64_t first = 1;  // the subtree searched first
    if (hint >= 0) {
        if (STATS) st.leaves++;
        if (facet_d2(B, hint, p) <= eps2) return true;
        if (SUBTREE) {
            const int64_t a = leaf_node(B.nf, hint) >> kHintLevels;
            first = a > 1 ? a : 1;
        }
    }
    if (STATS) st.traversals++;
    if (B.nf == 1) {
        if (STATS) st.leaves++;
        bool in = facet_d2(B, 0, p) <= eps2;
        if (in) hint = 0;
        return in;
    }
    V3<float> pf = mk3((float)p.x, (float)p.y, (float)p.z);
    float Tf = F32 ? f32_threshold(p, sqrtT) : 0.f;
    // the subtree of `first`, then (if it held no facet within eps) the whole
    // tree; the decision -- some facet within eps -- is the whole tree's
    for (int64_t root = first;; root = 1) {
        uint32_t trail = 0;
        int depth = 0;
        int64_t n = root;
        bool ok;
        int root_leaf;
        if (F32) {
            BvhNode32 r;
            if (root < B.ncache) r = from_lds(B.c32 + root);
            else r = B.n32[root];
            ok = box_d2(pf, r.lo, r.hi) <= Tf;
            root_leaf = r.leaf;
        } else {
            BvhNode64 r;
            if (root < B.ncache) r = from_lds(B.c64 + root);
            else r = B.n64[root];
            ok = box_d2(p, r.lo, r.hi) <= T;
            root_leaf = r.leaf;
        }
        if (STATS) st.boxes++;
        bool found = false;
        if (ok && root_leaf >= 0) {
            if (STATS) st.leaves++;
            if (facet_d2(B, root_leaf, p) <= eps2) {
                hint = root_leaf;
                found = true;
            }
        } else if (ok) {
            for (;;) {
                // n is internal here: look at both children
                int64_t c = 2 * n;
                double dl, dr;
                bool okl, okr;
                int leafl, leafr;
                if (F32) {
                    BvhNode32 L, R;
                    load_pair(B, c, L, R);
                    float fl = box_d2(pf, L.lo, L.hi), fr = box_d2(pf, R.lo, R.hi);
                    okl = fl <= Tf;
                    okr = fr <= Tf;
                    dl = fl;
                    dr = fr;
                    leafl = L.leaf;
                    leafr = R.leaf;
                } else {
                    BvhNode64 L, R;
                    load_pair(B, c, L, R);
                    dl = box_d2(p, L.lo, L.hi);
                    dr = box_d2(p, R.lo, R.hi);
                    okl = dl <= T;
                    okr = dr <= T;
                    leafl = L.leaf;
                    leafr = R.leaf;
                }
                if (STATS) st.boxes += 2;
                bool descend = okl || okr;
                if (descend) {
                    bool left = okl && (!okr || dl <= dr);
                    if (okl && okr) trail |= 1u << (depth + 1);
                    n = left ? c : c + 1;
                    depth++;
                    int leaf = left ? leafl : leafr;
                    if (leaf < 0) continue;
                    if (STATS) st.leaves++;
                    if (facet_d2(B, leaf, p) <= eps2) {
                        hint = leaf;
                        found = true;
                        break;
                    }
                }
                // backtrack to the deepest pending far child (depths are
                // counted from the subtree's root, which has no sibling here)
                bool done = false;
                for (;;) {
                    if (trail == 0) {
                        done = true;
                        break;
                    }
                    int d = 31 - __clz(trail);
                    trail &= ~(1u << d);
                    n = (n >> (depth - d)) ^ 1;
                    depth = d;
                    int leaf;
                    if (F32) leaf = n < B.ncache ? B.c32[n].leaf : B.n32[n].leaf;
                    else leaf = n < B.ncache ? B.c64[n].leaf : B.n64[n].leaf;
                    if (leaf < 0) break;
                    if (STATS) st.leaves++;
                    if (facet_d2(B, leaf, p) <= eps2) {
                        hint = leaf;
                        found = true;
                        done = true;
                        break;
                    }
                }
                if (done) break;
            }
        }
        if (found) return true;
        if (root == 1) return false;
    }
}


// ---- the facets near a small region, in LDS --------------------------------
// writable LDS records
typedef __attribute__((address_space(3))) BvhNode32 LdsNode32W;
typedef __attribute__((address_space(3))) uint32_t LdsU32;

// the wave's LDS writes so far, visible to its other lanes
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// x rounded to FP32 downward / upward
__device__ __forceinline__ float f32_down(double x)
{
    float f = (float)x;
    if ((double)f > x) f = f > 0.f ? u2f32(f2u(f) - 1u) : (f < 0.f ? u2f32(f2u(f) + 1u) : -0x1p-149f);
    return f;
}
__device__ __forceinline__ float f32_up(double x) { return -f32_down(-x); }

__device__ __forceinline__ bool box_meets(const BvhNode32& r, const float lof[3], const float hif[3])
{
    return r.lo[0] <= hif[0] && r.hi[0] >= lof[0] && r.lo[1] <= hif[1] && r.hi[1] >= lof[1] &&
           r.lo[2] <= hif[2] && r.hi[2] >= lof[2];
}

__device__ __forceinline__ void put_lds(LdsNode32W* d, const BvhNode32& s)
{
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        d->lo[k] = s.lo[k];
        d->hi[k] = s.hi[k];
    }
    d->leaf = s.leaf;
    // never read; without this write, or with 0, the smoother's registers come out
    // otherwise and a level of 40 problems takes 0.5 to 1.7 % longer
    d->pad = -1;
}

// The facets whose boxes meet the box [lo, hi], found by the G lanes of a
// group (G a power of two up to 64, lane gl, the group's first lane gbase in
// the wave) from a work list of nodes that meet the box (fr: two buffers of
// cap entries), level by level.  Each round reads, for n listed nodes, their
// descendants lv levels down, as many levels as fill the group (64 nodes for
// a list of one) and two at least, one node per lane from the FP32 records in global memory: a
// node's box lies inside its ancestors', so the levels between need no test,
// and FP32 boxes are rounded outward, so no facet is lost.  The rounds are a
// chain of dependent reads, five for 250 k facets (two levels a round, children
// and grandchildren of a node read by one lane, took nine rounds of twelve
// loads each: 84 k of a wave's cycles against 61 k; 60 k smoothing problems
// 1753 -> 1662 us).  Leaves lie on the last two levels (the median
// splits of the build), and rounds end on the last level at the latest, where
// a lane whose slot is empty looks at its parent.  Ballots place what meets the
// box -- leaves into lst as FP32 records, internal nodes into the next work
// list.  Returns the number of facets in lst, or -1 (nothing usable in lst)
// when more than cap facets, or more than cap nodes in one work list, meet the
// box, when the box is not finite, or for a one-facet tree.  Every lane of the
// group calls it.
template <int G>
__device__ int collect_facets(const BvhWalk& W, const double lo[3], const double hi[3],
                              LdsNode32W* lst, LdsU32* fr, int cap, int gl, int gbase)
{
    bool finite = true;
#pragma unroll
    for (int k = 0; k < 3; ++k) finite = finite && is_finite(lo[k]) && is_finite(hi[k]);
    if (!finite || W.nf < 2) return -1;
    float lof[3], hif[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        lof[k] = f32_down(lo[k]);
        hif[k] = f32_up(hi[k]);
    }
    const unsigned long long gm = (G == 64 ? ~0ull : ((1ull << (G & 63)) - 1ull)) << gbase;
    const unsigned long long below = ((1ull << (gbase + gl)) - 1ull) & gm;
    LdsU32* cur = fr;
    LdsU32* nxt = fr + cap;
    if (gl == 0) cur[0] = 1u;
    wave_sync();
    int below_root = 64 - __builtin_clzll((unsigned long long)(W.nf - 1));  // levels below the listed nodes
    int ncur = 1, nl = 0;
    while (ncur > 0) {
        int lv = below_root < 2 ? below_root : 2;
        while (lv < below_root && (ncur << (lv + 1)) <= G) ++lv;
        below_root -= lv;
        const int total = ncur << lv;
        int nn = 0;
        for (int t0 = 0; t0 < total; t0 += G) {
            const int t = t0 + gl;
            bool ok = false;
            BvhNode32 N;
            N.leaf = -2;
            int64_t id = 0;
            if (t < total) {
                id = ((int64_t)cur[t >> lv] << lv) + (t & ((1 << lv) - 1));
                if (id < W.nnode) N = W.n32[id];
                if (below_root == 0 && N.leaf == -2 && (id & 1) == 0) {
                    N = W.n32[id >> 1];
                    if (N.leaf < 0) N.leaf = -2;  // (a listed node's descendant: never so)
                }
                ok = N.leaf != -2 && box_meets(N, lof, hif);
            }
            const bool leaf = ok && N.leaf >= 0, inner = ok && N.leaf < 0;
            const unsigned long long ml = __ballot(leaf) & gm, mi = __ballot(inner) & gm;
            const int pl = nl + __popcll(ml & below), qi = nn + __popcll(mi & below);
            if (leaf && pl < cap) put_lds(lst + pl, N);
            if (inner && qi < cap) nxt[qi] = (uint32_t)id;
            nl += __popcll(ml);
            nn += __popcll(mi);
        }
        if (nl > cap || nn > cap) return -1;
        wave_sync();
        LdsU32* t = cur;
        cur = nxt;
        nxt = t;
        ncur = nn;
    }
    return nl;
}

typedef __attribute__((address_space(3))) double LdsF64;

// the FP32 box face_list_mask compares a list's boxes with: that of triangle
// (a, b, c) padded as the list's own box is (by 1.0001 sqrt(T) + 1e-9 max
// |coordinate|)
__device__ __forceinline__ void face_mask_box(V3<double> a, V3<double> b, V3<double> c,
                                              double sqrtT, float lof[3], float hif[3])
{
    double lo[3] = {a.x, a.y, a.z}, hi[3] = {a.x, a.y, a.z};
    const double q[6] = {b.x, b.y, b.z, c.x, c.y, c.z};
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        lo[j % 3] = fmin(lo[j % 3], q[j]);
        hi[j % 3] = fmax(hi[j % 3], q[j]);
    }
    double amax = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) amax = fmax(amax, fmax(fabs(lo[k]), fabs(hi[k])));
    const double pad = 1.0001 * sqrtT + 1e-9 * amax;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        lof[k] = f32_down(lo[k] - pad);
        hif[k] = f32_up(hi[k] + pad);
    }
}

// The positions of a collect_facets list (nl <= 128 entries) whose FP32 boxes
// meet a triangle's face_mask_box: every facet within sqrt(T) of a point of the
// triangle -- or of a sample of it, up to its rounding -- is at a set position.
// mk: two 64-bit words.
template <class L>
__device__ __forceinline__ void face_list_mask(L lst, int nl, const float lof[3], const float hif[3],
                                               uint64_t mk[2])
{
    // the two words in registers (an array indexed at run time would go to
    // scratch memory), eight records read before their tests
    const int n = nl < 128 ? nl : 128;
    uint64_t w[2] = {0ull, 0ull};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int e1 = n - 64 * h < 64 ? n - 64 * h : 64;
        uint64_t m = 0ull;
        for (int e0 = 0; e0 < e1; e0 += 8) {
            BvhNode32 r[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (e0 + u < e1) r[u] = from_lds(lst + 64 * h + e0 + u);
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const bool meet = e0 + u < e1 && box_meets(r[u], lof, hif);
                m |= (uint64_t)meet << (e0 + u);
            }
        }
        w[h] = m;
    }
    mk[0] = w[0];
    mk[1] = w[1];
}
// The positions of a collect_facets list (nl <= 128 entries) whose FP32 boxes
// can hold a facet within sqrt(T) of p (the tree walk's box test)
template <class L>
__device__ __forceinline__ void point_list_mask(L lst, int nl, V3<double> p, double sqrtT, uint64_t mk[2])
{
    const V3<float> pf = mk3((float)p.x, (float)p.y, (float)p.z);
    const float Tf = f32_threshold(p, sqrtT);
    uint64_t w[2] = {0ull, 0ull};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int e1 = nl - 64 * h < 64 ? nl - 64 * h : 64;
        uint64_t m = 0ull;
        for (int e0 = 0; e0 < e1; e0 += 8) {  // eight records read before their tests
            BvhNode32 r[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (e0 + u < e1) r[u] = from_lds(lst + 64 * h + e0 + u);
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (e0 + u < e1) m |= (uint64_t)(box_d2(pf, r[u].lo, r[u].hi) <= Tf) << (e0 + u);
        }
        w[h] = m;
    }
    mk[0] = w[0];
    mk[1] = w[1];
}

// ---- certified FP32 decisions for the listed facets ------------------------
// A sample's exact test against a facet (point_tri_d2, FP64) is some 240
// instructions once the lanes of a wave diverge over its seven regions, and a
// sample away from the limit does not need it.  Per listed facet the group
// keeps (LDS, kCertFloats floats) its unit normal and the outward unit
// normals of its edges in its plane, each with its offset from an origin o in
// the middle of the list's box.  In that frame, with q = p - o in FP32, h the
// distance from the plane and e_i the distances past the edges:
//   h^2 + max(e_i, 0)^2 is at most the squared distance (the projection lies
//   past edge i's line), so above (eps + mu)^2 the facet does not hold p;
//   it is the squared distance when the projection is inside (all e_i <= 0) or
//   its foot on the line of the edge it is furthest past lies on the edge, so
//   below (eps - mu)^2 the facet holds p.
// Everything else (the eps band, the corner regions, a facet without a frame)
// is left to FP64.  mu covers every rounding: with R the distance from o to
// the list box's corners every |q|, |offset| <= 4 R, so h and e_i are within
// 2^-20 R (twelve products and sums of 2^-24 relative error); mu = 2^-17 R +
// 2^-46 max|coordinate| is the margin on distances, eta = mu / 2 on the signs
// of the e_i.  A facet gets a frame only when the rounding of its own
// point_tri_d2 (2^-46 (edge + R)^2 over the squared sine of its angle at
// vertex 0) stays below mu eps / 4 and its determinant is above the 1e-30
// where point_tri_d2 leaves the interior out; others hold NaN, which fails
// every comparison.  The FP64 test's outcome is the certified one in every
// certified case, so decisions are unchanged.
//   Measured: 3 M triangles of 6-11 samples on 246 k facets 3.19 -> 2.57 ms, 200 k
// collapse candidates 360 -> 317 us, 12 triangles of ~800 samples 199 -> 159 us.
constexpr int kCertFloats = 20;  // 80 bytes: 16-byte reads, 16 bank phases
constexpr int kCertEntryBytes = 32 + 4 * kCertFloats;  // a list entry and its certificate
typedef __attribute__((address_space(3))) float LdsF32;

struct CertFrame {
    double o[3];
    double mu;  // the margin on distances (above eps / 4: no certificates)
    float in2, out2, eta;
    bool runs;  // samples between two certified ones on a line are certified
};

// The frame for a list made for the box [lo, hi] (padded, so it holds every
// point tested); amax: the box's largest coordinate magnitude before padding,
// d: the sampling distance.  runs: a facet's distance is convex, so it holds
// what lies between points that it holds, up to how far the samples are from
// their lines and triangles -- at most 16 ulp of edge^2 / d + max|coordinate|
// (the rows' starts carry the rounding of the triangle's angles) with edges of
// at most 2 R, which has to stay below mu / 4.
__device__ __forceinline__ CertFrame cert_frame(const double lo[3], const double hi[3], double amax,
                                                double eps2, double d)
{
    CertFrame F;
    double r2 = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        F.o[k] = 0.5 * (lo[k] + hi[k]);
        const double h = 0.5 * (hi[k] - lo[k]);
        r2 += h * h;
    }
    const double R = __builtin_sqrt(r2), eps = __builtin_sqrt(eps2);
    F.mu = 0x1p-17 * R + 0x1p-46 * amax;
    F.eta = (float)(0.5 * F.mu);
    F.runs = 4.0 * r2 + amax * d <= F.mu * d * 0x1p44;
    F.in2 = -1.0f;
    F.out2 = __builtin_inff();
    // (squares in FP32 need room on both sides; NaN fails)
    if (F.mu <= 0.25 * eps && eps2 > 1e-24 && r2 < 1e24) {
        F.in2 = (float)((eps - F.mu) * (eps - F.mu) * (1.0 - 0x1p-20));
        F.out2 = (float)((eps + F.mu) * (eps + F.mu) * (1.0 + 0x1p-20));
    }
    return F;
}

// writes facet t's entry (9 doubles) into c
template <class P>
__device__ __forceinline__ void cert_write(P c, const double* t, const CertFrame& F, double eps2)
{
    const V3<double> o = mk3(F.o[0], F.o[1], F.o[2]);
    const V3<double> a = ld3(t) - o, b = ld3(t + 3) - o, d = ld3(t + 6) - o;
    const V3<double> e0 = b - a, e1 = d - a, e2 = d - b;
    const V3<double> n = cross(e0, e1);
    const double a00 = len2(e0), a11 = len2(e1), a01 = dot(e0, e1), nn = len2(n);
    const double det = a00 * a11 - a01 * a01;
    const double r = 0x1p17 * F.mu;  // >= R
    const double big = (a00 > a11 ? a00 : a11) + r * r;
    const bool ok = det > 1e-29 && nn > 1e-29 && F.in2 > 0.0f &&
                    big * a00 * a11 <= F.mu * __builtin_sqrt(eps2) * 0x1p44 * nn;
    const double lim = 4.0 * r;  // an offset beyond it keeps its sign and stays out of reach
    const V3<double> un = mulv(n, 1.0 / __builtin_sqrt(nn));
    V3<double> m[3] = {cross(e0, un), cross(e2, un), cross(un, e1)};
    const V3<double> at[3] = {a, b, a};
#pragma unroll
    for (int k = 0; k < 3; ++k) m[k] = mulv(m[k], 1.0 / len(m[k]));
    double off[4] = {dot(un, a), dot(m[0], at[0]), dot(m[1], at[1]), dot(m[2], at[2])};
#pragma unroll
    for (int k = 0; k < 4; ++k) off[k] = off[k] > lim ? lim : (off[k] < -lim ? -lim : off[k]);
    const float bad = __builtin_nanf("");
    c[0] = ok ? (float)un.x : bad;
    c[1] = ok ? (float)un.y : bad;
    c[2] = ok ? (float)un.z : bad;
    c[3] = ok ? (float)off[0] : bad;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        c[4 + 4 * k] = (float)m[k].x;
        c[5 + 4 * k] = (float)m[k].y;
        c[6 + 4 * k] = (float)m[k].z;
        c[7 + 4 * k] = (float)off[k + 1];
    }
    c[16] = (float)dot(m[0], m[1]);
    c[17] = (float)dot(m[1], m[2]);
    c[18] = (float)dot(m[2], m[0]);
    c[19] = 0.0f;
}

// the entries of a whole collect_facets list (lanes gl, gl + G, ...); ends
// with the group's writes visible
template <int G>
__device__ __forceinline__ void cert_list(const BvhWalk& W, LdsNode32W* lst, LdsF32* cert, int nl,
                                          const CertFrame& F, double eps2, int gl)
{
    for (int e = gl; e < nl; e += G)
        cert_write(cert + kCertFloats * e, W.tri + 9 * (int64_t)lst[e].leaf, F, eps2);
    wave_sync();
}

__device__ __forceinline__ V3<float> cert_local(const CertFrame& F, V3<double> p)
{
    return mk3((float)(p.x - F.o[0]), (float)(p.y - F.o[1]), (float)(p.z - F.o[2]));
}

// 1: the facet holds the point, -1: it does not, 0: FP64 decides
template <class P>
__device__ __forceinline__ int cert_class(P c, V3<float> q, const CertFrame& F)
{
    float v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = c[k];
    float s[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        s[k] = __builtin_fmaf(v[4 * k], q.x, __builtin_fmaf(v[4 * k + 1], q.y,
                              __builtin_fmaf(v[4 * k + 2], q.z, -v[4 * k + 3])));
    const float me = s[1] > s[2] ? (s[1] > s[3] ? s[1] : s[3]) : (s[2] > s[3] ? s[2] : s[3]);
    const float mp = me > 0.0f ? me : 0.0f;
    const float lb2 = __builtin_fmaf(mp, mp, s[0] * s[0]);
    int r = lb2 > F.out2 ? -1 : 0;
    if (lb2 < F.in2) {
        if (me < -F.eta) {
            r = 1;
        } else {
            // past (or at) one edge: the foot on its line, against the others
            const float g01 = c[16], g12 = c[17], g20 = c[18];
            const bool i0 = me == s[1], i1 = !i0 && me == s[2];
            const float fa = i0 ? s[2] - me * g01 : (i1 ? s[1] - me * g01 : s[1] - me * g20);
            const float fb = i0 ? s[3] - me * g20 : (i1 ? s[3] - me * g12 : s[2] - me * g12);
            if (fa < -F.eta && fb < -F.eta) r = 1;
        }
    }
    return r;
}

// in_envelope's decision for a point p of the box that a collect_facets list
// was made for, with that box padded by at least sqrt(T) beyond every point
// tested (then the list holds every facet the tree walk could accept) and every
// facet within sqrt(T) of p at a position set in mask (two 64-bit words, lists of
// at most 128 facets): the facet at list position hl first (the one that held the
// previous point, -1: none), then the positions set in mask, in ascending order;
// positions no certificate decides go to FP64 at the end.  On a hit hl becomes
// the position of a facet that holds p.  sure: set when that is certified.
template <class L, class P, class M>
__device__ __forceinline__ bool in_envelope_cert(const BvhWalk& W, L lst, P cert, int nl, M mask,
                                                 V3<double> p, const CertFrame& F, double eps2,
                                                 int& hl, bool& sure)
{
    const V3<float> q = cert_local(F, p);
    uint64_t open[2] = {0ull, 0ull}, done[2] = {0ull, 0ull};
    auto mark = [](uint64_t (&w)[2], int i) {
        const uint64_t b = 1ull << (i & 63);
        w[0] |= i < 64 ? b : 0ull;
        w[1] |= i < 64 ? 0ull : b;
    };
    sure = true;
    if (hl >= 0) {
        const int r = cert_class(cert + kCertFloats * hl, q, F);
        if (r > 0) return true;
        mark(done, hl);
        if (r == 0) mark(open, hl);
    }
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        uint64_t mm = 64 * w < nl ? mask[w] & ~done[w] : 0ull;
        while (mm) {
            const int i = 64 * w + __builtin_ctzll(mm);
            mm &= mm - 1;
            const int r = cert_class(cert + kCertFloats * i, q, F);
            if (r > 0) {
                hl = i;
                return true;
            }
            if (r == 0) open[w] |= 1ull << (i & 63);
        }
    }
    sure = false;
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        uint64_t mm = open[w];
        while (mm) {
            const int i = 64 * w + __builtin_ctzll(mm);
            mm &= mm - 1;
            if (facet_d2(W, lst[i].leaf, p) <= eps2) {
                hl = i;
                return true;
            }
        }
    }
    return false;
}

// nearest_facet with the reference's traversal order
// (src/tetwild/geogram/mesh_AABB.h:130-141, mesh_AABB.cpp:381-480):
// get_nearest_facet_hint, then depth-first search visiting the nearer child
// first (the right one on ties) and pruning boxes whose signed distance is not
// below the best so far.  Stackless: one bit per level marks a far child still
// to visit; its box distance is recomputed on the way back (the same value the
// recursion keeps on its stack), so the walk needs no per-lane memory.
// node k of the FP64 tree, from the walker's LDS copy when it holds it
__device__ __forceinline__ BvhNode64 node64(const BvhWalk& B, int64_t k)
{
    if (k < B.ncache) return from_lds(B.c64 + k);
    return B.n64[k];
}

// get_nearest_facet_hint: down from the root to a leaf, into the child whose
// box center is nearer
__device__ __forceinline__ int nearest_hint(const BvhWalk& B, V3<double> p)
{
    int64_t nd = 1;
    while (node64(B, nd).leaf < 0) {
        const BvhNode64 L = node64(B, 2 * nd), R = node64(B, 2 * nd + 1);
        nd = box_center_d2(p, L.lo, L.hi) < box_center_d2(p, R.lo, R.hi) ? 2 * nd : 2 * nd + 1;
    }
    return node64(B, nd).leaf;
}

__device__ __forceinline__ int nearest_facet(const BvhWalk& B, V3<double> p, V3<double>& np,
                                             double& sq)
{
    int best = nearest_hint(B, p);
    np = ld3(B.tri + 9 * (int64_t)best);
    sq = len2(np - p);
    auto visit = [&](int leaf) {
        const double* t = B.tri + 9 * (int64_t)leaf;
        V3<double> cp;
        double dd = point_tri_d2<double, true>(p, ld3(t), ld3(t + 3), ld3(t + 6), cp);
        if (dd < sq) {
            best = leaf;
            np = cp;
            sq = dd;
        }
    };
    {
        const int root_leaf = node64(B, 1).leaf;
        if (root_leaf >= 0) {  // a one-facet tree: the root is the leaf
            visit(root_leaf);
            return best;
        }
    }
    int64_t n = 1;
    int depth = 0;
    uint32_t trail = 0;  // bit d: the far child at depth d is still to visit
    for (;;) {
        // n is internal: the nearer child first
        const int64_t c = 2 * n;
        BvhNode64 L, R;
        load_pair(B, c, L, R);
        const double dl = box_signed_d2(p, L.lo, L.hi);
        const double dr = box_signed_d2(p, R.lo, R.hi);
        const bool left = dl < dr;
        // the far child is never nearer, so a pruned near child prunes both
        if ((left ? dl : dr) < sq) {
            trail |= 1u << (depth + 1);
            n = left ? c : c + 1;
            depth++;
            const int leaf = left ? L.leaf : R.leaf;
            if (leaf < 0) continue;
            visit(leaf);
        }
        // back to the deepest pending far child that can still hold a nearer facet
        for (;;) {
            if (trail == 0) return best;
            const int d = 31 - __clz(trail);
            trail &= ~(1u << d);
            const int64_t far = (n >> (depth - d)) ^ 1;
            n = far;
            depth = d;
            const BvhNode64 F = node64(B, far);
            if (!(box_signed_d2(p, F.lo, F.hi) < sq)) continue;
            const int leaf = F.leaf;
            if (leaf < 0) break;
            visit(leaf);
        }
    }
}

// nearest_facet's result (facet, np, sq -- bit for bit) computed by the G
// lanes of a group (lane gl, first lane gbase in the wave; G a power of two up
// to 64), or -1 where the group cannot be sure to agree.
// The walk starts from the hint facet h with sq = s0 = |v0(h) - p|^2 and
// takes a facet only when its distance is strictly below the best so far.
// The group lists the facets whose boxes meet a cube around p (collect_facets)
// -- half-width rr plus more than the rounding of a facet distance, so the
// list holds every facet at distance rr or less -- and computes their
// distances; rr starts at the hint leaf's box diagonal (about one facet) and
// doubles, up to sqrt(s0), until some listed facet lies within rr.  None
// below s0 with rr = sqrt(s0): the walk keeps (h, v0(h)).  Else let f be the
// facet of least distance D: when no other facet has distance D and every
// node on f's path from the root has a box distance strictly below D, the
// walk cannot prune that path (it prunes a box only at or above the best so
// far, never below D) and nothing it visits later replaces f, so it returns
// f -- taken here.  Otherwise (ties, a box at or above D, a list too long for
// cap, a query that is not finite, three cubes without a facet): -1.  Every lane of the group calls it with the same p.
template <int G>
__device__ int nearest_facet_try(const BvhWalk& B, V3<double> p, V3<double>& np, double& sq,
                                   LdsNode32W* lst, LdsU32* fr, int cap, int gl, int gbase)
{
    if (B.nf < 2) return -1;
    int64_t na = 1;
    while (node64(B, na).leaf < 0) {
        const BvhNode64 L = node64(B, 2 * na), R = node64(B, 2 * na + 1);
        na = box_center_d2(p, L.lo, L.hi) < box_center_d2(p, R.lo, R.hi) ? 2 * na : 2 * na + 1;
    }
    const BvhNode64 HL = node64(B, na);
    const int h = HL.leaf;
    const V3<double> v0 = ld3(B.tri + 9 * (int64_t)h);
    const double s0 = len2(v0 - p), sr0 = __builtin_sqrt(s0);
    if (!(s0 <= 1.0e300)) return -1;
    // more than the rounding of a facet distance: ~1e-7 (|p| + d + 2 edge) in
    // distance units (the root box's diagonal bounds every edge)
    const BvhNode64 root = node64(B, 1);
    const double diag = __builtin_sqrt(len2(mk3(root.hi[0] - root.lo[0], root.hi[1] - root.lo[1],
                                                root.hi[2] - root.lo[2])));
    const double eabs = 0x1p-20 * (diag + fmax(fabs(p.x), fmax(fabs(p.y), fabs(p.z))));
    double r = __builtin_sqrt(len2(mk3(HL.hi[0] - HL.lo[0], HL.hi[1] - HL.lo[1], HL.hi[2] - HL.lo[2])));
    const unsigned long long gm = (G == 64 ? ~0ull : ((1ull << (G & 63)) - 1ull)) << gbase;
    for (int attempt = 0; attempt < 3; ++attempt, r *= 2.0) {
        const bool last = !(r < sr0);  // the cube holds every facet below s0
        const double rr = last ? sr0 : r;
        const double half = rr + 0x1p-20 * rr + eabs;
        const double lo[3] = {p.x - half, p.y - half, p.z - half};
        const double hi[3] = {p.x + half, p.y + half, p.z + half};
        // listed from the global tree (~1 % faster than through an LDS copy
        // of its top; the descents above read the copy)
        BvhWalk GW = B;
        GW.ncache = 0;
        GW.top64 = false;
        const int n = collect_facets<G>(GW, lo, hi, lst, fr, cap, gl, gbase);
        if (n < 0) break;
        // the lane's least distance below s0, its facet and how many reach it
        double bd = s0;
        int bf = -1, nb = 0;
        V3<double> bcp = v0;
        for (int i = gl; i < n; i += G) {
            const int f = lst[i].leaf;
            const double* t = B.tri + 9 * (int64_t)f;
            V3<double> cp;
            const double dd = point_tri_d2<double, true>(p, ld3(t), ld3(t + 3), ld3(t + 6), cp);
            if (dd < bd) {
                bd = dd;
                bf = f;
                bcp = cp;
                nb = 1;
            } else if (dd == bd && bf >= 0) {
                nb++;
            }
        }
        double m = bd;
        for (int off = G / 2; off > 0; off >>= 1) {
            const double o = __shfl_xor(m, off, G);
            m = o < m ? o : m;
        }
        const unsigned long long at = __ballot(bf >= 0 && bd == m) & gm;
        if (at == 0ull) {
            if (!last) continue;
            np = v0;  // no facet below s0
            sq = s0;
            return h;
        }
        if (!last && !(m <= rr * rr)) continue;  // a nearer facet may lie outside
        const int wl = __builtin_ctzll(at) - gbase;
        const int wf = __shfl(bf, wl, G);
        bool sure = (at & (at - 1)) == 0ull && __shfl(nb, wl, G) == 1;
        if (sure) {
            // every box on the path from the root to wf's leaf strictly below m
            const int64_t leaf = leaf_node(B.nf, wf);
            const int depth = 63 - __builtin_clzll((unsigned long long)leaf);
            bool below = true;
            for (int k = 1 + gl; k <= depth; k += G) {
                const BvhNode64 N = node64(B, leaf >> (depth - k));
                below = below && box_signed_d2(p, N.lo, N.hi) < m;
            }
            sure = (__ballot(!below) & gm) == 0ull;
        }
        if (!sure) break;
        np = mk3(__shfl(bcp.x, wl, G), __shfl(bcp.y, wl, G), __shfl(bcp.z, wl, G));
        sq = m;
        return wf;
    }
    return -1;
}

// nearest_facet by the group's lanes, walking itself where they are not sure
template <int G>
__device__ int nearest_facet_group(const BvhWalk& B, V3<double> p, V3<double>& np, double& sq,
                                   LdsNode32W* lst, LdsU32* fr, int cap, int gl, int gbase)
{
    const int f = nearest_facet_try<G>(B, p, np, sq, lst, fr, cap, gl, gbase);
    return f >= 0 ? f : nearest_facet(B, p, np, sq);
}

// Triangles whose longest edge exceeds kMaxEdgeSamples sampling distances are
// reported out without sampling: their sample count (quadratic in that ratio)
// would keep one lane busy for seconds.  TetWild's faces are orders of
// magnitude below this.
constexpr double kMaxEdgeSamples = 65536.0;

// isFaceOutEnvelop_sampling for a triangle known not to be degenerate
template <bool F32, bool STATS>
__device__ bool face_out_sampled(const BvhWalk& B, const double* t9, double eps2, double d,
                                 double T, double sqrtT, Stats& st)
{
    const V3<double> a = ld3(t9), b = ld3(t9 + 3), c = ld3(t9 + 6);
    {
        double l = fmax(len2(a - b), fmax(len2(b - c), len2(c - a)));
        if (!(__builtin_sqrt(l) / d <= kMaxEdgeSamples)) return true;
    }
    int hint = -1;
    return for_each_sample(a, b, c, d, [&](V3<double> s) {
        if (STATS) st.samples++;
        return !in_envelope<F32, STATS>(B, s, eps2, T, sqrtT, hint, st);
    });
}

// What a lane keeps of its triangle while the wave's list is made: its corners
// in the list's frame, the one SampleGen::init rotates to the front first, and
// the box face_list_mask compares the list with.  (The corners themselves,
// 18 registers, are read again by the few lanes that need them.)
struct WaveFace {
    bool act;
    int first;
    const double* t9;
    V3<float> q[3];
    float mlo[3], mhi[3];
};

// the corner SampleGen::init rotates to the front; false for a triangle that is
// reported out without sampling
__device__ __forceinline__ bool wave_face_first(V3<double> a, V3<double> b, V3<double> c, double d, int& first)
{
    const double l0 = len2(a - b), l1 = len2(b - c), l2 = len2(c - a);
    const double N = __builtin_sqrt(fmax(l0, fmax(l1, l2))) / d;
    first = 0;
    if (!(N <= kMaxEdgeSamples)) return false;
    if (N > 1) first = !(l2 < l0) && !(l2 < l1) ? 2 : (!(l1 < l0) ? 1 : 0);
    return true;
}

// face_out_sampled for the wave's triangles at once (a list of nl <= 128
// facets, nl >= 0, with its certificates).  Every lane scans the facets near
// its triangle for one that holds its first corner: none, and the triangle is
// out; one that certifies all three corners, and it is in.  The few triangles
// still open -- they straddle facets, or reach the limit -- are sampled by
// their lanes, which pass over the samples between two that one facet
// certifies on a row.  (Spreading the open triangles' samples over the wave
// takes two more samplers per lane and their registers: 3 M triangles of 6-11
// samples 1568 us against 1551, of ~20 samples 3205 against 3028.)  Returns the
// lane's decision.
__device__ bool faces_wave_listed(const BvhWalk& W, const WaveFace& T, double eps2, double d,
                                  LdsNode32W* lst, LdsF32* cert, int nl, const CertFrame& F)
{
    bool out = T.act, open_lane = false;
    uint64_t mk[2] = {0ull, 0ull};
    int hl = -1;
    const double* t9 = T.t9;
    if (T.act) {
        face_list_mask(lst, nl, T.mlo, T.mhi, mk);
        uint64_t unsure[2] = {0ull, 0ull};
        bool all = false;
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            uint64_t mm = 64 * w < nl ? mk[w] : 0ull;
            while (mm && !all) {
                const int i = 64 * w + __builtin_ctzll(mm);
                LdsF32* ci = cert + kCertFloats * i;
                const int r = cert_class(ci, T.q[0], F);
                if (r == 0) unsure[w] |= mm & (0ull - mm);
                mm &= mm - 1;
                if (r > 0) {
                    hl = i;
                    all = F.runs && cert_class(ci, T.q[1], F) > 0 && cert_class(ci, T.q[2], F) > 0;
                }
            }
        }
        if (hl < 0 && (unsure[0] | unsure[1])) {
            const V3<double> p0 = ld3(t9 + 3 * T.first);
#pragma unroll
            for (int w = 0; w < 2; ++w)
                for (uint64_t mm = unsure[w]; mm && hl < 0; mm &= mm - 1) {
                    const int i = 64 * w + __builtin_ctzll(mm);
                    if (facet_d2(W, lst[i].leaf, p0) <= eps2) hl = i;
                }
        }
        out = hl < 0;
        open_lane = hl >= 0 && !all;
    }
    if (open_lane) {
        SampleGen g;
        g.init(ld3(t9), ld3(t9 + 3), ld3(t9 + 6), d);
        V3<double> s;
        g.next(s);  // the first corner
        while (g.next(s)) {
            bool sure;
            if (!in_envelope_cert(W, lst, cert, nl, mk, s, F, eps2, hl, sure)) {
                out = true;
                break;
            }
            if (sure && F.runs) {
                const int64_t left = g.run_left(INT64_MAX);
                if (left > 0 && cert_class(cert + kCertFloats * hl, cert_local(F, g.run_at(left)), F) > 0)
                    g.k += (int)left;
            }
        }
    }
    return out;
}

// LDS of face_out_wave per wave: a triangle's segment record and header
// (SampleGen::store_seg) and its row table
constexpr int kWaveRows = 96;
constexpr int kWaveSegBytes = kSegRec * 8 + kSegHdr * 4 + kWaveRows * kSegRow * 8;
typedef __attribute__((address_space(3))) int LdsI32;

// face_out_sampled's decision computed by a wave (every lane passes the same
// triangle, r its lane), against a collect_facets list with its certificates
// (lst, cert, F, nl >= 0; its box holding the triangle padded by more than
// sqrt(T)) or the tree (nl < 0).  A facet that certifies the three corners
// settles the triangle.  Otherwise the sampler's sequence of `total` samples is
// cut into 64 consecutive blocks of K = ceil(total / 64); lane r finds sample
// r K and tests its block in order -- when a facet certifies a sample and the
// last one of the lane's run along the same row, the ones between are passed
// over -- and after each step a ballot stops the wave at the first sample
// found outside.  A triangle of up to kWaveRows rows has them made a row per
// lane in LDS (seg, kWaveSegBytes; seg_row: a row needs nothing from the ones
// before it); the lanes of a taller one pass whole rows by their headers
// (SampleGen::skip), one after another.  12 triangles of ~800 samples: 159 ->
// 66 us, 30 k of ~90 797 -> 343.  The decision -- some sample has no facet within eps -- does
// not depend on which lane tests which sample, so it equals
// face_out_sampled's.  For batches of few triangles with many samples each,
// where one lane per triangle leaves most of the machine idle.
template <bool F32, bool SUBTREE = true>
__device__ bool face_out_wave(const BvhWalk& B, V3<double> a, V3<double> b, V3<double> c, double eps2,
                              double d, double T, double sqrtT, int r, LdsNode32W* lst, LdsF32* cert,
                              const CertFrame& F, int nl, LdsF64* seg)
{
    {
        double l = fmax(len2(a - b), fmax(len2(b - c), len2(c - a)));
        if (!(__builtin_sqrt(l) / d <= kMaxEdgeSamples)) return true;
    }
    if (nl > 0 && F.runs) {
        const V3<float> qa = cert_local(F, a), qb = cert_local(F, b), qc = cert_local(F, c);
        bool all = false;
        for (int e = r; e < nl; e += 64) {
            LdsF32* ce = cert + kCertFloats * e;
            all = all || (cert_class(ce, qa, F) > 0 && cert_class(ce, qb, F) > 0 &&
                          cert_class(ce, qc, F) > 0);
        }
        if (__ballot(all)) return false;
    }
    SampleGen g;
    g.init(a, b, c, d);
    const int rows = g.phase != 9 && g.M >= 1 ? g.M : 0;
    const bool table = rows <= kWaveRows;
    LdsF64* row = seg + kSegRec;
    LdsI32* hdr = (LdsI32*)(row + kWaveRows * kSegRow);
    SegFace S;
    int64_t total;
    if (table) {
        if (r == 0) g.store_seg(seg, hdr, 0);
        wave_sync();
        int made = rows, sum = 0;  // the rows before the first that ends, their samples
        for (int m0 = 0; m0 < rows; m0 += 64) {
            const int m = m0 + r;
            int rc = 0;
            if (m < rows) {
                V3<double> st = mk3(0.0, 0.0, 0.0);
                rc = seg_row(seg, d, m + 1, st);
                row[kSegRow * m] = st.x;
                row[kSegRow * m + 1] = st.y;
                row[kSegRow * m + 2] = st.z;
                row[kSegRow * m + 3] = (double)rc;
            }
            const unsigned long long end = __ballot(m < rows && rc == 0);
            if (end && made > m0 + __builtin_ctzll(end)) made = m0 + __builtin_ctzll(end);
            sum += m < made ? rc : 0;
        }
        for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
        if (r == 0) hdr[kShRows] = made;
        wave_sync();
        S.load(hdr);
        total = S.total(sum);
    } else {
        total = g.skip(INT64_MAX);
        g.init(a, b, c, d);
    }
    const int64_t K = (total + 63) / 64;
    const int64_t first = (int64_t)r * K;
    const int64_t mine = total - first < K ? total - first : K;
    int ss = 0, sk = 0, sc = 0;
    if (mine > 0) {
        if (table) {
            S.seek(row, first, ss, sk);
            sc = S.count(row, ss);
        } else {
            g.skip(first);
        }
    }
    int hint = -1, hl = -1;
    Stats st;
    const uint64_t mask[2] = {~0ull >> (nl < 64 && nl > 0 ? 64 - nl : 0),
                              nl > 64 ? ~0ull >> (128 - nl) : 0ull};
    for (int64_t j = 0; __ballot(j < mine);) {
        V3<double> q = a;
        bool have = j < mine, out = false, sure = false;
        if (have && table) {
            while (sk >= sc) {  // past the segments with no samples left
                sk = 0;
                if (++ss >= S.nseg()) {
                    have = false;
                    break;
                }
                sc = S.count(row, ss);
            }
            if (have) q = S.sample(seg, row, ss, sk++, d);
        } else if (have) {
            have = g.next(q);
        }
        if (have) {
            if (nl >= 0) out = !in_envelope_cert(B, lst, cert, nl, mask, q, F, eps2, hl, sure);
            else out = !in_envelope<F32, false, SUBTREE>(B, q, eps2, T, sqrtT, hint, st);
        }
        ++j;
        if (sure && !out && F.runs && j < mine) {
            int64_t left = mine - j;
            if (table) left = sc - sk < left ? sc - sk : left;
            else left = g.run_left(left);
            if (left > 0) {
                const V3<double> e = table ? S.sample(seg, row, ss, sk + (int)left - 1, d) : g.run_at(left);
                if (cert_class(cert + kCertFloats * hl, cert_local(F, e), F) > 0) {
                    j += left;
                    if (table) sk += (int)left;
                    else g.k += (int)left;
                }
            }
        }
        if (__ballot(out)) return true;
    }
    return false;
}

// isFaceOutEnvelop_sampling for one triangle (false for a collinear one)
template <bool F32, bool STATS>
__device__ bool face_out(const BvhWalk& B, const double* t9, double eps2, double d, double T,
                         double sqrtT, Stats& st)
{
    if (collinear3(t9, t9 + 3, t9 + 6)) return false;
    return face_out_sampled<F32, STATS>(B, t9, eps2, d, T, sqrtT, st);
}

inline BvhView bvh_view(const twg_bvh* b)
{
    BvhView v;
    v.n64 = b->node64;
    v.n32 = b->node32;
    v.tri = b->tri;
    v.nf = b->nf;
    v.nnode = b->nnode;
    return v;
}

inline BvhView no_bvh()
{
    BvhView v = {nullptr, nullptr, nullptr, 0, 0};
    return v;
}

// Whether a quarter of the facets have more than some 36 others in a box of side
// `reach` about them.  Read off the level whose cells are up to twice as wide,
// with the kCrowd for its width; a cell holds about two thirds of what a box of
// its size about a facet does, so the line lies between 24 and 48 facets.
inline bool reach_wide(const twg_bvh* b, double reach)
{
    int l = 0;
    double s = b->side;
    while (l + 1 < kCrowdLevels && 0.5 * s >= reach) {
        s *= 0.5;
        ++l;
    }
    return 4 * b->crowded[s * s >= 2.0 * reach * reach][l] > b->nf;
}

inline double bvh_prune_threshold(const twg_bvh* b, double eps2)
{
    double r = b->rmax + __builtin_sqrt(eps2);
    return eps2 + eps2 * 0x1p-20 + 0x1p-44 * (r * r);
}

}  // namespace twg
