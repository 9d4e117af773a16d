// Internal definitions behind the opaque C handles.
#pragma once
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/sortgpu.h"
#include "bvh_build.h"
#include "layout.h"

struct sortgpu_ctx {
    int device = -1;
    bool host_only = true;
    int num_cus = 0;
    size_t hbm_bytes = 0;
    char arch[64] = {0};
    sortgpu_tuning tuning{};
    std::mutex mu;
    std::string err;
    std::atomic<int> refs{1};  // the creator's, plus one per object made from the context
    // stream-ordered device memory for traversal orders (created on first use; released with the
    // context once its last allocation is freed)
    hipMemPool_t order_pool = nullptr;
    ~sortgpu_ctx() {
        if (order_pool) (void)hipMemPoolDestroy(order_pool);
    }
};

namespace sortgpu {
// Work-counter ring: each query takes the next slot so queries on different streams that
// share one accelerator never share a counter (unless more than kCounterSlots are in flight).
constexpr uint32_t kCounterSlots = 256;
constexpr uint32_t kCounterStride = 16;  // 64 B apart
}  // namespace sortgpu

struct sortgpu_accel {
    sortgpu_ctx* ctx = nullptr;
    sortgpu::BuiltTree host;
    sortgpu::TreeView view;
    void* d_nodes = nullptr;
    sortgpu::PrimRec* d_prims = nullptr;
    sortgpu::QuadRec* d_quads = nullptr;
    sortgpu::WalkNode* d_wnodes = nullptr;
    sortgpu::PrimRec* d_wrecs = nullptr;
    sortgpu::WalkAux* d_waux = nullptr;
    uint32_t* d_wgates = nullptr;
    uint32_t* d_counters = nullptr;
    uint32_t* d_error = nullptr;
    unsigned long long* d_stats = nullptr;
    std::atomic<uint32_t> slot{0};
    size_t device_bytes = 0;
    // host copies of the input geometry (shading and hit reconstruction need it by primitive id)
    std::vector<float> pos;
    std::vector<uint32_t> idx;
    std::vector<sortgpu_quad> quads;
};

namespace sortgpu {
void set_error(sortgpu_ctx* ctx, const char* fmt, ...);
int hip_fail(sortgpu_ctx* ctx, hipError_t e, const char* what);
int ctx_bind(sortgpu_ctx* ctx);
// Reference counting of contexts: every object made from a context holds one reference.
void ctx_acquire(sortgpu_ctx* ctx);
void ctx_release(sortgpu_ctx* ctx);
int upload_accel(sortgpu_accel* acc);
// Copies the context's tuning knobs into a launch.
void apply_tuning(const sortgpu_ctx* ctx, struct TraceArgs& a);
void free_accel_device(sortgpu_accel* acc);
// Which batches are traced in traversal order by default (order.hip). Sorting costs 0.15 ms for 4M
// rays, and a sorted batch reads its rays and writes its results scattered; what it saves is
// traffic past the caches. Measured on rays in random order, sorted against index order:
//   walk tree (closest, any): pays once the tree outgrows the caches and the batch is large. 4M rays
//     through 1M triangles (58 MB of nodes and records) 2.36 against 2.21 ms, 3.6M triangles (209 MB)
//     2.46 / 2.91, 8M 2.68 / 3.43, 16M 2.67 / 3.76; shadow segments 1M 2.33 / 2.47, 3.6M 2.47 / 3.52,
//     16M 2.78 / 4.68; 2M rays: 1M triangles 1.35 / 1.26 (shadow 1.35 / 1.39), 3.6M 1.51 / 1.66 (shadow
//     1.43 / 1.93), 16M 1.59 / 2.13; 1M rays: 1M 0.99 / 0.84, 3.6M 0.97 / 0.95 (shadow 1.02 / 1.16), 8M
//     1.11 / 1.15 (no line at 1M rays serves both kinds on such trees);
//   transparent shadows: 524K rays through 200K triangles 1.99 / 1.90 ms, through 1M 2.63 / 2.75; 1M
//     rays 2.96 / 2.97 and 3.80 / 4.10; 2M 4.94 / 5.11 and 6.38 / 6.82 (the line looks at the rays alone: at
//     524K it costs the smaller of these trees 5% and gives the larger 4%);
//   multi-hit probes: 524K into 200K triangles 0.45 / 0.38, into 1M 0.56 / 0.51; 1M 0.62 / 0.69 and
//     0.84 / 0.95; 4M 1.80 / 2.58 and 2.62 / 3.50;
//   Fast-BVH walk (trees without a walk tree): batches of 256K rays and more.
constexpr uint32_t kReorderMinRays = 1u << 18;
constexpr uint32_t kReorderMinWalkRays = 1u << 21;
constexpr size_t kReorderMinWalkBytes = (size_t)192 << 20;
constexpr uint32_t kReorderMinAttenuation = 1u << 19;
constexpr uint32_t kReorderMinMulti = 1u << 20;
// Bytes a walk reads of a tree's walk tree (0: it has none).
inline size_t walk_bytes(const BuiltTree& t) {
    return t.walk.nodes.size() * sizeof(WalkNode) + t.walk.recs.size() * sizeof(PrimRec);
}
// The same of an accelerator as it lies on the device (its upload may have left the walk tree out).
inline size_t walked_bytes(const sortgpu_accel* a) { return a->view.walk_stack ? walk_bytes(a->host) : 0; }
// The default for closest- and any-hit batches on walk trees of `bytes` together (0: no walk tree).
inline bool reorder_pays(uint32_t n, size_t bytes) {
    return bytes ? n >= kReorderMinWalkRays && bytes >= kReorderMinWalkBytes : n >= kReorderMinRays;
}
// Waves of at least this many paths shade each bounce's hits in spatial order (tuning shade_order:
// 0 = this default, 1 = never (0 returned), 2 = always).
inline uint32_t shade_sort_min(const sortgpu_tuning& t) {
    return t.shade_order == 1 ? 0u : t.shade_order == 2 ? 1u : (1u << 18);
}
// The context's stream-ordered pool for traversal-order buffers (made on first use), or null.
hipMemPool_t order_pool(sortgpu_ctx* ctx);
// Takes (and clears) the error flags at d_flags after the work queued on `s`; returns SORTGPU_OK
// when none was raised, else SORTGPU_ERR_STATE with a message naming each flag ("who: ...").
int report_flags(sortgpu_ctx* ctx, uint32_t* d_flags, hipStream_t s, const char* who, uint32_t* flags_out);
}  // namespace sortgpu
