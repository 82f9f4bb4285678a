// groups.hip -- isFlip + calTetQualities + getCheckQuality over many small
// groups of tets in one launch: the evaluation step of every configuration
// EdgeRemover tries (src/tetwild/EdgeRemover.cpp:138-174 for 3-2, 327-368 for
// the two rotations of 4-4, 501-575 for the tet pairs of 5-6), and of any
// other caller that checks a handful of candidate tets at a time.
//
// Eight lanes per group, a tet each (configurations hold 2..6): the call is
// bound by the chain offsets -> ids -> coordinates, which one lane per group
// ran through once per tet with a third of the machine's waves (150 k groups of
// 2..6 tets 44 -> 32 us a call, 600 k 178 -> 94).  Orientation comes from the floating-point
// filter; a group with no tet certainly flipped but some tet undecided is
// marked and finished by a second pass with the exact predicate, one thread per
// group, which keeps the exact code's registers out of the main kernel.
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

// lanes per group
constexpr int kGroupLanes = 8;

__global__ __launch_bounds__(kBlock) void groups_kernel(GroupArgs A)
{
    constexpr int L = kGroupLanes;
    const int lane = threadIdx.x % L, base = threadIdx.x % 64 - lane;
    const unsigned mask = (1u << L) - 1u;
    const int64_t stride = (int64_t)gridDim.x * (kBlock / L);
    for (int64_t g = xcd_block() * (int64_t)(kBlock / L) + threadIdx.x / L; g < A.n_groups; g += stride) {
        const int64_t b = A.off[g], e = A.off[g + 1];
        // what the group's tets say in their order: the first bad or flipped
        // one decides (later ones are not looked at), qualities are written
        // once no tet is
        bool bad = b < 0 || e < b || e > A.n_tets, flip = false, undecided = false;
        const bool wide = !bad && e - b > L;  // more than a sweep
        double m = 0.0, q = 0.0;
        if (!bad) {
            for (int64_t k = b; k < e; k += L) {
                bool tb = false, tf = false, tu = false;
                if (k + lane < e) {
                    Tet T;
                    tb = !load(A, A.tets[k + lane], T);
                    if (!tb) {
                        const int o = orient3d_filter(T.p[0], T.p[1], T.p[2], T.p[3]);
                        tu = o == kUndecided;
                        tf = !tu && o != 1;
                        if (!wide) {
                            q = amips_energy(T);
                            if (is_inf(q) || is_nan(q) || q <= 0) q = kMaxEnergy;
                            m = q;
                        }
                    }
                }
                const unsigned mb = (unsigned)(__ballot(tb) >> base) & mask, mf = (unsigned)(__ballot(tf) >> base) & mask;
                undecided = undecided || ((unsigned)(__ballot(tu) >> base) & mask) != 0u;
                if (mb | mf) {
                    bad = ((mb | mf) & -(mb | mf) & mb) != 0u;
                    flip = !bad;
                    break;
                }
            }
        }
        if (wide && !bad && !flip && !undecided)
            for (int64_t k = b + lane; k < e; k += L) {
                Tet T;
                load(A, A.tets[k], T);
                double v = amips_energy(T);
                if (is_inf(v) || is_nan(v) || v <= 0) v = kMaxEnergy;
                if (A.q) A.q[k] = v;
                m = v > m ? v : m;
            }
        for (int off = L / 2; off > 0; off >>= 1) {
            const double o = __shfl_xor(m, off, L);
            m = o > m ? o : m;
        }
        const bool fine = !bad && !flip && !undecided;
        if (fine && !wide && A.q && b + lane < e) A.q[b + lane] = q;
        if (lane == 0) {
            A.flipped[g] = bad ? TWG_GROUP_BAD_INPUT : (flip ? 1 : (undecided ? kGroupPending : 0));
            if (bad || flip) A.max_q[g] = __builtin_nan("");
            else if (fine) A.max_q[g] = m;
        }
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
    const unsigned gm = (unsigned)std::min<int64_t>((n_groups * kGroupLanes + kBlock - 1) / kBlock, 1 << 20);
    hipLaunchKernelGGL(groups_kernel, dim3(gm), dim3(kBlock), 0, ctx->cur, A);
    TWG_LAUNCHED();
    const unsigned gx = std::min<unsigned>(grid_for(n_groups), 1024u);
    hipLaunchKernelGGL(groups_exact_kernel, dim3(gx), dim3(kBlock), 0, ctx->cur, A);
    TWG_LAUNCHED();
    return TWG_OK;
}
