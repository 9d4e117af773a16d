// The walk tree only makes queries faster: a build short of host memory, an upload and a pool short of device
// memory go without it. The library's sources are built here against a device whose memory is a number.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <random>
#include <string>
#include <vector>

#include "api_internal.h"
#include "trace_launch.h"

using namespace sortgpu;

// ---- host memory: the n-th allocation from now on fails -------------------------------------------
static std::atomic<long> g_until{-1};
static void* take(size_t n) {
    if (g_until >= 0 && g_until-- == 0) throw std::bad_alloc();
    void* p = std::malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void* operator new(size_t n) { return take(n); }
void* operator new[](size_t n) { return take(n); }
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }
void operator delete[](void* p) noexcept { std::free(p); }
void operator delete[](void* p, size_t) noexcept { std::free(p); }

// ---- the device --------------------------------------------------------------------------------------
static size_t g_room = SIZE_MAX, g_held = 0;
extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    if (n > g_room - g_held) return hipErrorOutOfMemory;
    char* b = static_cast<char*>(std::malloc(n + 64));
    std::memcpy(b, &n, sizeof(n));
    g_held += n;
    *p = b + 64;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    size_t n;
    std::memcpy(&n, static_cast<char*>(p) - 64, sizeof(n));
    g_held -= n;
    std::free(static_cast<char*>(p) - 64);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) {
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMemPoolDestroy(hipMemPool_t) { return hipSuccess; }
}
namespace sortgpu {
void set_error(sortgpu_ctx*, const char*, ...) {}
int hip_fail(sortgpu_ctx*, hipError_t e, const char*) { return e == hipErrorOutOfMemory ? SORTGPU_ERR_OOM : SORTGPU_ERR_HIP; }
int ctx_bind(sortgpu_ctx*) { return 0; }
void ctx_acquire(sortgpu_ctx*) {}
void ctx_release(sortgpu_ctx*) {}
void apply_tuning(const sortgpu_ctx*, TraceArgs&) {}
int report_flags(sortgpu_ctx*, uint32_t*, hipStream_t, const char*, uint32_t*) { return 0; }
hipMemPool_t order_pool(sortgpu_ctx*) { return nullptr; }
uint32_t trace_max_stack_supported() { return 1024; }
hipError_t launch_trace(const TraceArgs&, bool, bool, hipStream_t, int) { return hipSuccess; }
hipError_t order_rays_multi(hipMemPool_t, const void*, const uint32_t*, uint32_t, const TreeView*, uint32_t, hipStream_t, RayOrder&) {
    return hipErrorOutOfMemory;
}
void release_order(RayOrder&, hipStream_t) {}
}  // namespace sortgpu

static int fail(const char* what, long at) {
    std::printf("FAIL %s (%ld)\n", what, at);
    return 1;
}

int main() {
    // a tree of 20,000 primitives: eight children to a node, up to 16 primitives to a leaf
    std::mt19937 g(5);
    std::uniform_real_distribution<float> u(0.f, 1.f);
    const uint32_t n = 20000;
    std::vector<float> pos(9 * (size_t)n);
    std::vector<uint32_t> idx(3 * (size_t)n);
    for (uint32_t t = 0; t < n; t++)
        for (int v = 0; v < 9; v++) pos[9 * (size_t)t + v] = (v % 3 ? u(g) * 0.01f : (float)t / n) + 0.01f * u(g);
    for (uint32_t i = 0; i < 3 * n; i++) idx[i] = i;
    BuildInput in;
    in.pos = pos.data();
    in.nverts = 3 * n;
    in.idx = idx.data();
    in.ntris = n;
    in.quads = nullptr;
    in.nquads = 0;
    in.width = 8;
    in.max_leaf = 16;
    in.max_depth = 28;
    in.threads = 4;
    std::vector<BuildPrim> prims(n);
    float box[6] = {1e30f, 1e30f, 1e30f, -1e30f, -1e30f, -1e30f};
    for (uint32_t t = 0; t < n; t++) {
        BuildPrim& p = prims[t];
        p.id = t;
        for (int k = 0; k < 3; k++) {
            const float* f = &pos[9 * (size_t)t + k];
            p.mn[k] = std::min(f[0], std::min(f[3], f[6]));
            p.mx[k] = std::max(f[0], std::max(f[3], f[6]));
            p.c[k] = (p.mn[k] + p.mx[k]) * 0.5f;
            box[k] = std::min(box[k], p.mn[k]);
            box[3 + k] = std::max(box[3 + k], p.mx[k]);
        }
    }
    std::vector<SrcNode> src = {{0, n, 0, 0}};
    for (size_t i = 0; i < src.size(); i++) {
        if (src[i].cnt <= 16) continue;
        src[i].first = (uint32_t)src.size();
        src[i].nchild = 8;
        const SrcNode s = src[i];
        for (uint32_t j = 0; j < 8; j++) {
            const uint32_t a = s.off + s.cnt * j / 8, b = s.off + s.cnt * (j + 1) / 8;
            src.push_back({a, b - a, 0, 0});
        }
    }
    bool whole = false, none = false;
    for (long at = 0; !whole; at += 1 + at / 4) {
        WalkTree w;
        g_until = at;
        build_walk_tree(in, prims, src, box, 4, w);
        whole = g_until >= 0;
        g_until = -1;
        if (whole != (w.stack != 0) && !(w.stack != 0 && !whole)) return fail("walk tree without memory", at);
        if (!w.stack && (!w.nodes.empty() || !w.recs.empty() || !w.gates.empty())) return fail("a part of a walk tree", at);
        none |= !w.stack;
    }
    if (!none) return fail("no allocation failed", 0);

    // a device with room for everything, for the Fast-BVH and part of the walk tree, and for less
    sortgpu_ctx ctx;
    ctx.host_only = false;
    sortgpu_accel acc;
    acc.ctx = &ctx;
    std::string err;
    if (!build_tree(in, acc.host, err) || !acc.host.walk.stack) return fail("build", 0);
    std::memset(&acc.view, 0, sizeof(acc.view));
    if (upload_accel(&acc) || !acc.view.walk_stack || acc.device_bytes > g_held) return fail("upload", 0);
    const size_t all = g_held, walk = acc.host.walk.nodes.size() * sizeof(WalkNode) + acc.host.walk.recs.size() * sizeof(PrimRec) +
                                      acc.host.walk.aux.size() * sizeof(WalkAux) + acc.host.walk.gates.size() * sizeof(uint32_t);
    sortgpu_accel* list[2] = {&acc, &acc};
    sortgpu_pool* pool = nullptr;
    uint64_t info[4];
    if (sortgpu_pool_create(&ctx, list, 2, &pool)) return fail("pool", 0);
    const size_t pool_all = g_held - all;
    sortgpu_pool_destroy(pool);
    for (size_t less : {walk / 8, walk / 2, walk - 1024}) {
        g_room = all + pool_all - 2 * less;
        if (sortgpu_pool_create(&ctx, list, 2, &pool)) return fail("pool without walk trees", (long)less);
        sortgpu_pool_info(pool, info);
        if (info[2] > g_held - all) return fail("pool bytes", (long)less);
        sortgpu_pool_destroy(pool);
        if (g_held != all) return fail("pool memory", (long)less);
    }
    g_room = all + 1024;
    if (sortgpu_pool_create(&ctx, list, 2, &pool) != SORTGPU_ERR_OOM || g_held != all) return fail("pool without memory", 0);
    free_accel_device(&acc);
    if (g_held) return fail("accelerator memory", 0);
    for (size_t less : {(size_t)1, walk / 8, walk / 2, walk - 1024}) {
        g_room = all - less;
        std::memset(&acc.view, 0, sizeof(acc.view));
        if (upload_accel(&acc)) return fail("upload without the walk tree", (long)less);
        if (acc.view.walk_stack || acc.view.wnodes || acc.view.wgates || acc.device_bytes > all - walk) return fail("walk tree kept", (long)less);
        free_accel_device(&acc);
        if (g_held) return fail("accelerator memory", (long)less);
    }
    g_room = all - walk - 1;
    if (upload_accel(&acc) != SORTGPU_ERR_OOM || g_held) return fail("upload without memory", 0);
    std::printf("ok\n");
    return 0;
}
