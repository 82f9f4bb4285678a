// twg_internal.hpp -- context, error reporting and launch helpers shared by
// the translation units of libtetwild_amd.so.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cstdio>
#include <map>
#include <mutex>
#include <string>
#include <tuple>

#include "../../include/tetwild_gpu.h"

struct twg_ctx {
    int device = 0;
    hipStream_t own = nullptr;
    hipStream_t cur = nullptr;
    // recorded on the old stream when the caller switches streams, so work on
    // the new one starts after the old one's use of the shared scratch
    hipEvent_t order = nullptr;
    int num_cus = 256;
    // growable device memory owned by the context.  in_graph: a stream was
    // capturing when a call took it, so a graph may hold its address
    struct Block {
        void* p = nullptr;
        size_t bytes = 0;
        bool in_graph = false;
    };
    Block scratch;
    // further blocks: 0 the queue of tets the orientation filter left
    // undecided, 1 the envelope batches' query order, 2 the nearest queries'
    // (which take none under capture, so they never write to a graph's)
    Block slot[3];
    // outgrown blocks that a graph may still use, freed with the context (a
    // block grows by a quarter at least, so they come to less than five times
    // the one in use)
    struct Retired {
        void* p;
        Retired* next;
    };
    Retired* retired = nullptr;
    // device address of smooth.hip's file-scope scratch array on this
    // context's device (twg_smooth_batch_noalloc), looked up at creation
    void* noalloc_scratch = nullptr;
    // debug counters of the envelope list kernels (twg_ctx_list_stats):
    // waves that tested their LDS facet list, waves that walked the tree
    unsigned long long* list_stats = nullptr;
    bool list_stats_on = false;
    // pinned host memory a kernel writes a synchronous call's result to
    void* host_out = nullptr;
};
constexpr size_t kHostOutBytes = 256;

namespace twg {

void set_error(const char* fmt, ...);

// returns nonzero (TWG_EDEVICE) and records the message on failure
int hip_fail(hipError_t e, const char* what, const char* file, int line);

// Whether the context's stream captures a graph (or cannot be asked: the null
// stream beside a capturing one).
bool capturing(twg_ctx* ctx);

int ensure_scratch(twg_ctx* ctx, size_t bytes);
int ensure_slot(twg_ctx* ctx, int i, size_t bytes);

// Morton order of n query items (points: stride 3, triangles: stride 9,
// keyed by their centroids) near tree B: writes a permutation (int32, device)
// into *order (in the context's `slot`).  The order only affects speed: every
// query's result is independent of it.
int morton_order(twg_ctx* ctx, int slot, const double* items, int64_t n, int stride, const twg_bvh* B,
                 const int32_t** order);

// Whether that order takes more bits than its size asks for: the surface is graded.
bool morton_refined(const twg_bvh* B, int64_t n);

// Stable sort of n (key, value) pairs by the low `bits` bits of their keys:
// kv[0] in and, after the call, out; kv[1] as large; work: sort_pairs_bytes(n).
size_t sort_pairs_bytes(int64_t n);
int sort_pairs(ulonglong2* kv[2], int64_t n, int bits, void* work, hipStream_t s);

// Activates ctx->device for the calling thread.
int bind(twg_ctx* ctx);

// With ctx->device current: the device address of the no-allocation
// smoothing entry point's scratch array, into ctx->noalloc_scratch.
int noalloc_scratch_init(twg_ctx* ctx);

constexpr int kBlock = 256;

// Autotuner results: (device, precision flag, size class) -> (tile, chunk),
// shared by every context of the process.  Contexts may live on different
// host threads, so the map is guarded.
class TuneCache {
public:
    bool get(int device, bool flag, int size_class, int& tile, unsigned& chunk)
    {
        std::lock_guard<std::mutex> lock(m_);
        auto it = map_.find(std::make_tuple(device, flag, size_class));
        if (it == map_.end()) return false;
        tile = it->second.first;
        chunk = it->second.second;
        return true;
    }
    void put(int device, bool flag, int size_class, int tile, unsigned chunk)
    {
        std::lock_guard<std::mutex> lock(m_);
        map_[std::make_tuple(device, flag, size_class)] = {tile, chunk};
    }

private:
    std::mutex m_;
    std::map<std::tuple<int, bool, int>, std::pair<int, unsigned>> map_;
};

// The two timing events of an autotuner, destroyed on every path out of the
// scope that owns them (early error returns included).
struct EventPair {
    hipEvent_t e0 = nullptr;
    hipEvent_t e1 = nullptr;
    hipError_t create()
    {
        hipError_t e = hipEventCreate(&e0);
        return e == hipSuccess ? hipEventCreate(&e1) : e;
    }
    ~EventPair()
    {
        if (e0) (void)hipEventDestroy(e0);
        if (e1) (void)hipEventDestroy(e1);
    }
};

// xcd_block (twg_math.hpp) in runs: each XCD takes 64 consecutive blocks in
// turn instead of a contiguous eighth of the grid.  No XCD is left with a long
// eighth of uneven work (sorted queries: 3 M triangles 2187 -> 1812 us with
// one-wave blocks, 31 % of the CU time had been idle), and eight streams a
// gigabyte apart become eight near each other (AMIPS over 10.1 M tets, three
// meshes in turn: 317 -> 291 us; runs of 8 and 512 blocks 292 and 303).
__device__ __forceinline__ int64_t xcd_run_block()
{
    const unsigned g = gridDim.x, b = blockIdx.x;
    const unsigned whole = g / 512 * 512;
    if (b >= whole) return b;
    const unsigned k = b / 8;
    return (int64_t)(k / 64) * 512 + (b % 8) * 64 + k % 64;
}

inline unsigned grid_for(int64_t n, int block = kBlock)
{
    int64_t g = (n + block - 1) / block;
    return (unsigned)(g < 1 ? 1 : g);
}

}  // namespace twg

#define TWG_HIP(expr)                                                    \
    do {                                                                 \
        hipError_t _e = (expr);                                          \
        if (_e != hipSuccess) return twg::hip_fail(_e, #expr, __FILE__, __LINE__); \
    } while (0)

#define TWG_REQUIRE(cond, ...)                       \
    do {                                             \
        if (!(cond)) {                               \
            twg::set_error(__VA_ARGS__);             \
            return TWG_EINVAL;                       \
        }                                            \
    } while (0)

// after a kernel launch
#define TWG_LAUNCHED() TWG_HIP(hipGetLastError())
