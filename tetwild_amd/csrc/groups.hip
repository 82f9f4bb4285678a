// groups.hip -- isFlip + calTetQualities + getCheckQuality over many small
// groups of tets in one launch: the evaluation step of every configuration
// EdgeRemover tries (src/tetwild/EdgeRemover.cpp:138-174 for 3-2, 327-368 for
// the two rotations of 4-4, 501-575 for the tet pairs of 5-6), and of any
// other caller that checks a handful of candidate tets at a time.
//
// A wave takes up to 64 consecutive groups and evaluates their tets a lane each,
// whatever the groups' sizes; words and qualities meet in LDS, where a lane per
// group reads its verdict.  Small batches are bound by the chain offsets -> ids
// -> coordinates, large ones by the gathers where a batch's groups lie apart and
// by FP64 arithmetic where neighbours share vertices.  One lane per group runs
// the chain once per tet; eight lanes per group leave half of them idle on four
// tets.  us a call with one lane, eight, and this: 150 k groups of 2..6 tets of a
// lattice at random 54, 28, 29; 2.5 M of four 673, 358, 327; 2.5 M of four in the
// lattice's order 120, 298, 124; 300 k of 20 1450, 258, 97.  (The next ids read
// before a tet's arithmetic: 133 -> 118 in order, 317 -> 330 at random.)
// Orientation comes from the floating-point filter; a group with no tet certainly
// flipped but some tet undecided is marked and finished by a second pass with the
// exact predicate, one thread per group, which keeps the exact code's registers
// out of the main kernel.
#include <algorithm>

#include "twg_internal.hpp"
#include "twg_math.hpp"

namespace twg {
namespace {

constexpr uint8_t kGroupPending = 3;

struct GroupArgs {
    const int4* __restrict__ tets;
    const int32_t* __restrict__ off;
    int64_t n_groups, n_tets;
    const double* __restrict__ x;
    const double* __restrict__ y;
    const double* __restrict__ z;
    int64_t nv;
    uint8_t* __restrict__ flipped;
    double* __restrict__ max_q;
    double* __restrict__ q;
};

__device__ __forceinline__ bool load(const GroupArgs& A, int4 t, Tet& T)
{
    const int id[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (id[j] < 0 || id[j] >= A.nv) return false;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        T.p[j][0] = A.x[id[j]];
        T.p[j][1] = A.y[id[j]];
        T.p[j][2] = A.z[id[j]];
    }
    return true;
}

// group g with every orientation decided exactly
__device__ void eval_group_exact(const GroupArgs& A, int64_t g)
{
    const int64_t b = A.off[g], e = A.off[g + 1];
    // isFlip (src/tetwild/LocalOperations.cpp:555-573): any tet not POSITIVE
    bool flip = false, bad = false;
    for (int64_t k = b; k < e && !flip && !bad; ++k) {
        Tet T;
        if (!load(A, A.tets[k], T)) {
            bad = true;
            break;
        }
        flip = orient3d(T.p[0], T.p[1], T.p[2], T.p[3]) != 1;
    }
    if (bad) {
        A.flipped[g] = TWG_GROUP_BAD_INPUT;
        A.max_q[g] = __builtin_nan("");
        return;
    }
    if (flip) {
        A.flipped[g] = 1;
        A.max_q[g] = __builtin_nan("");
        return;
    }
    // calTetQualities of positively oriented tets (src/tetwild/LocalOperations.cpp:
    // 695-773, 862-884) and getCheckQuality's max (:575-588)
    double m = 0.0;
    for (int64_t k = b; k < e; ++k) {
        Tet T;
        load(A, A.tets[k], T);
        double q = amips_energy(T);
        if (is_inf(q) || is_nan(q) || q <= 0) q = kMaxEnergy;
        if (A.q) A.q[k] = q;
        m = q > m ? q : m;
    }
    A.flipped[g] = 0;
    A.max_q[g] = m;
}

// the wave's LDS accesses so far come before its later ones
__device__ __forceinline__ void wave_order()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// what a tet says: kBad and kFlip decide their group (the first of them does),
// kOpen sends it to the exact pass unless one of those does
enum : uint8_t { kFine = 0, kOpen = 1, kFlip = 2, kBad = 3 };

// tet t's word and, unless it is kBad, its quality
__device__ __forceinline__ uint8_t tet_word(const GroupArgs& A, int4 t, double& q)
{
    Tet T;
    if (!load(A, t, T)) return kBad;
    q = amips_energy(T);
    if (is_inf(q) || is_nan(q) || q <= 0) q = kMaxEnergy;
    const int o = orient3d_filter(T.p[0], T.p[1], T.p[2], T.p[3]);
    return o == kUndecided ? kOpen : (o != 1 ? kFlip : kFine);
}

__device__ __forceinline__ void group_out(const GroupArgs& A, int64_t g, uint8_t word, double m)
{
    A.flipped[g] = word == kBad ? TWG_GROUP_BAD_INPUT : (word == kFlip ? 1 : (word == kOpen ? kGroupPending : 0));
    if (word == kBad || word == kFlip) A.max_q[g] = __builtin_nan("");
    else if (word == kFine) A.max_q[g] = m;
}

// lanes per group where groups are taken one by one
constexpr int kGroupLanes = 8;
// tets a wave takes at once: four rounds and, with groups of mixed sizes, a fourth
// more (64 groups of 2..6 pass 256 every other time, and those waves take three
// times as long)
constexpr int kWaveTets = 320;

// group g by eight lanes, eight tets a round (g < 0: none); the wave calls it
__device__ void group_by_lanes(const GroupArgs& A, int64_t g)
{
    constexpr int L = kGroupLanes;
    const int lane = threadIdx.x % L, base = threadIdx.x % 64 - lane;
    const unsigned mask = (1u << L) - 1u;
    const int64_t b = g < 0 ? 0 : A.off[g], e = g < 0 ? 0 : A.off[g + 1];
    uint8_t word = b < 0 || e < b || e > A.n_tets ? kBad : kFine;
    if (word == kFine)
        for (int64_t k = b; k < e; k += L) {
            double v;
            const uint8_t w = k + lane < e ? tet_word(A, A.tets[k + lane], v) : kFine;
            const unsigned stop = (unsigned)(__ballot(w >= kFlip) >> base) & mask;
            const unsigned bad = (unsigned)(__ballot(w == kBad) >> base) & mask;
            if (((unsigned)(__ballot(w == kOpen) >> base) & mask) != 0u) word = kOpen;
            if (stop) {
                word = (stop & -stop & bad) != 0u ? kBad : kFlip;
                break;
            }
        }
    double m = 0.0;
    if (word == kFine)
        for (int64_t k = b + lane; k < e; k += L) {
            double v;
            (void)tet_word(A, A.tets[k], v);
            if (A.q) A.q[k] = v;
            m = v > m ? v : m;
        }
    for (int off = L / 2; off > 0; off >>= 1) {
        const double o = __shfl_xor(m, off, L);
        m = o > m ? o : m;
    }
    if (g >= 0 && lane == 0) group_out(A, g, word, m);
}

// gw (8 .. 64) consecutive groups a wave; where their tets do not fit its LDS, or
// an offset is out of range, eight lanes a group
__global__ __launch_bounds__(kBlock) void groups_kernel(GroupArgs A, int gw)
{
    __shared__ double lq[kBlock / 64][kWaveTets];
    __shared__ uint8_t lw[kBlock / 64][kWaveTets];
    const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
    const int64_t stride = (int64_t)gridDim.x * (kBlock / 64) * gw;
    for (int64_t g0 = (xcd_block() * (int64_t)(kBlock / 64) + w) * gw; g0 < A.n_groups; g0 += stride) {
        const int cnt = A.n_groups - g0 < gw ? (int)(A.n_groups - g0) : gw;
        const bool mine = lane < cnt;
        const int64_t b = mine ? A.off[g0 + lane] : 0, e = mine ? A.off[g0 + lane + 1] : 0;
        const int64_t first = __shfl(b, 0, 64), last = __shfl(e, cnt - 1, 64);
        if (__ballot(mine && (b < 0 || e < b || e > A.n_tets)) || last - first > kWaveTets) {
            for (int k = 0; k < cnt; k += 64 / kGroupLanes) {
                const int j = k + lane / kGroupLanes;
                group_by_lanes(A, j < cnt ? g0 + j : -1);
            }
            continue;
        }
        const int n = (int)(last - first);
        int4 t = make_int4(0, 0, 0, 0);
        if (lane < n) t = A.tets[first + lane];
        for (int k = lane; k < n; k += 64) {
            const int4 c = t;
            if (k + 64 < n) t = A.tets[first + k + 64];
            double v = 0.0;
            lw[w][k] = tet_word(A, c, v);
            lq[w][k] = v;
        }
        wave_order();
        if (mine) {
            const int kb = (int)(b - first), ke = (int)(e - first);
            uint8_t word = kFine;
            double m = 0.0;
            for (int k = kb; k < ke && word < kFlip; ++k) {
                const uint8_t t = lw[w][k];
                word = t > word ? t : word;
                m = lq[w][k] > m ? lq[w][k] : m;
            }
            if (word != kFine)
                for (int k = kb; k < ke; ++k) lw[w][k] = kBad;  // no qualities
            group_out(A, g0 + lane, word, m);
        }
        if (A.q) {
            wave_order();
            for (int k = lane; k < n; k += 64)
                if (lw[w][k] == kFine) A.q[first + k] = lq[w][k];
        }
        wave_order();
    }
}

__global__ __launch_bounds__(kBlock) void groups_exact_kernel(GroupArgs A)
{
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t g = (int64_t)blockIdx.x * kBlock + threadIdx.x; g < A.n_groups; g += stride)
        if (A.flipped[g] == kGroupPending) eval_group_exact(A, g);
}

}  // namespace
}  // namespace twg

using namespace twg;

extern "C" int twg_tet_groups(twg_ctx* ctx, const int32_t* tets, const int32_t* group_off,
                              int64_t n_groups, int64_t n_tets, const double* x, const double* y,
                              const double* z, int64_t nv, uint8_t* flipped, double* max_q,
                              double* q)
{
    TWG_REQUIRE(ctx != nullptr, "twg_tet_groups: NULL context");
    TWG_REQUIRE(n_groups >= 0 && n_tets >= 0 && nv >= 0, "twg_tet_groups: negative size");
    TWG_REQUIRE(n_groups == 0 || (tets && group_off && x && y && z && flipped && max_q),
                "twg_tet_groups: NULL array");
    TWG_REQUIRE(!tets || ((uintptr_t)tets & 15) == 0, "twg_tet_groups: tets must be 16-byte aligned");
    if (n_groups == 0) return TWG_OK;
    if (int r = bind(ctx)) return r;
    GroupArgs A;
    A.tets = reinterpret_cast<const int4*>(tets);
    A.off = group_off;
    A.n_groups = n_groups;
    A.n_tets = n_tets;
    A.x = x;
    A.y = y;
    A.z = z;
    A.nv = nv;
    A.flipped = flipped;
    A.max_q = max_q;
    A.q = q;
    // as many groups a wave as leave four rounds of tets, at the batch's mean, and
    // 16 waves a CU (which holds 20): 150 k groups of 2..6 22.4, 22.3, 21.5 us with
    // 8, 16, 32 a wave; 2.5 M of 4 in order 169, 150, 140 with
    // 16, 32, 64 (124 since)
    int gw = 8;
    while (gw < 64 && 2 * gw * n_tets <= 256 * n_groups && n_groups >= (int64_t)32 * gw * ctx->num_cus) gw *= 2;
    const int64_t per = gw * (kBlock / 64);
    const unsigned gm = (unsigned)std::min<int64_t>((n_groups + per - 1) / per, 1 << 20);
    hipLaunchKernelGGL(groups_kernel, dim3(gm), dim3(kBlock), 0, ctx->cur, A, gw);
    TWG_LAUNCHED();
    const unsigned gx = std::min<unsigned>(grid_for(n_groups), 1024u);
    hipLaunchKernelGGL(groups_exact_kernel, dim3(gx), dim3(kBlock), 0, ctx->cur, A);
    TWG_LAUNCHED();
    return TWG_OK;
}
