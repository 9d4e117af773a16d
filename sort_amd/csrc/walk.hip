// Closest-hit and any-hit queries over the walk tree (walk_tree.h), with the Fast-BVH's results.
//
// What a query returns is defined by the Fast-BVH walk of trace.hip: hits count only in leaves
// whose box the ray's slab test accepts, leaves are pruned by their entry distance, and equal hits
// go to the one met first. This kernel finds candidates in a tree of its own (4-wide nodes of 48
// bytes, at most two triangles to a leaf) and then shows that the walk would have returned the same:
//
//   * The candidates are complete. A walk node's boxes are quantised outwards, and every slab is
//     widened by kPad = 2^-19 of the largest coordinate in play, more than the rounding of the slab
//     distances (4 units of 2^-24 of it) and of the triangle test (18 units) put together. So a
//     triangle that the triangle test accepts is always reached, unless its t is past the pruning bound.
//   * Slab distances grow monotonically from a box to a box inside it, in floating point too (each
//     is one product and one sum), and a Fast-BVH node's box holds its children's exactly. So the
//     walk may take hits from a leaf when the leaf's own box passes, and the leaf is pruned only by
//     a hit nearer than the leaf's own entry distance.
//   * Let (t, leaf) be the nearest candidate whose leaf passes, and e that leaf's entry distance.
//     Only a hit at a distance in [t, e] can tie with it or prune it. The walk here keeps looking up
//     to `lim`, a little past t, and remembers the second nearest distance it met: if that lies past
//     max(t, e) and e does not lie past lim, the walk returns this candidate.
//
// A ray for which this cannot be shown (a tie across leaves, a leaf box missed by rounding), or whose
// numbers leave the bounds above (NaN, infinities, a negative tmin, an origin very far out), is walked
// again through the Fast-BVH by its lane, in `exact_walk`. Any hit needs less: the first candidate
// whose leaf box passes.
//
// What it saves: on the benchmark's 4,194,304 bounce rays through 2^20 triangles a ray of the
// Fast-BVH walk tests 14.8 nodes and 81.5 triangles, reading 391 chunks of 16 bytes; here it tests 30.4
// nodes and 11.6 triangles, reading 123 chunks, with about half the arithmetic. The call takes 2.09 ms
// instead of 4.35; 1.5M shadow segments through 300K triangles 0.97 instead of 1.79; 2M camera rays on
// 768K triangles of spheres 0.70 instead of 0.80. Leaves of one triangle instead of two: 2 to 3 steps
// more per ray on meshes. 8-wide nodes: 20.7 steps instead of 30.4, each with twice the arithmetic.
#include <hip/hip_runtime.h>

#include "trace_launch.h"
#include "traverse.h"

#pragma clang fp contract(off)

namespace sortgpu {
namespace {

constexpr int kBlock = 256;
constexpr uint32_t kNone = 0xffffffffu;
constexpr float kPad = 1.9073486328125e-6f;  // 2^-19

// What the walk keeps of a ray besides the triangle test's constants: reciprocal directions (true
// ones, at most 1e18) and plane offsets widened outwards (near: a, far: b).
struct Slabs {
    float rx, ry, rz, ax, ay, az, bx, by, bz;
};

__device__ __forceinline__ float recip(float d) {
    const float a = fmaxf(fabsf(d), 1e-18f);
    return copysignf(1.0f / a, d);
}

// ray_setup's shear constants and traverse.h's root test, from the reciprocals above: 1 / d is the
// same number wherever |d| >= 1e-18. (The Fast-BVH's own slab constants are not set.)
__device__ __forceinline__ void shear_setup(RayK& r, const Slabs& s) {
    const float ax = fabsf(r.dx), ay = fabsf(r.dy), az = fabsf(r.dz);
    int ky;
    if (ax > ay && ax > az) ky = 0;
    else ky = ay > az ? 1 : 2;
    const int kz = ky == 2 ? 0 : ky + 1;
    const int kx = kz == 2 ? 0 : kz + 1;
    r.kx = kx; r.ky = ky; r.kz = kz;
    const float px = sel3(r.dx, r.dy, r.dz, kx);
    const float py = sel3(r.dx, r.dy, r.dz, ky);
    const float pz = sel3(r.dx, r.dy, r.dz, kz);
    r.sx = -px / py;
    r.sz = -pz / py;
    r.sy = sel3(s.rx, s.ry, s.rz, ky);
    r.okx = sel3(r.ox, r.oy, r.oz, kx);
    r.oky = sel3(r.ox, r.oy, r.oz, ky);
    r.okz = sel3(r.ox, r.oy, r.oz, kz);
}
__device__ __forceinline__ bool root_test(const RayK& r, const Slabs& s, const float* bb) {
    float tmax = r.tmax, tmin = r.tmin;
    const float o[3] = {r.ox, r.oy, r.oz};
    const float d[3] = {r.dx, r.dy, r.dz};
    const float q[3] = {s.rx, s.ry, s.rz};
    bool ok = true;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        if (d[a] < 0.00001f && d[a] > -0.00001f) {
            ok &= !(o[a] > bb[3 + a] || o[a] < bb[a]);
        } else {
            const float t1 = (bb[3 + a] - o[a]) * q[a], t2 = (bb[a] - o[a]) * q[a];
            const bool swap = t1 > t2;
            tmin = smax(swap ? t2 : t1, tmin);
            tmax = smin(swap ? t1 : t2, tmax);
            ok &= !(tmin > tmax);
        }
    }
    return ok && tmin >= 0.0f;
}

// Whether the error bounds above hold for this ray; fills `s` and the search slack.
__device__ __forceinline__ bool slabs_setup(const RayK& r, const float* bb, Slabs& s, float& slack) {
    const float mo = fmaxf(fmaxf(fabsf(r.ox), fabsf(r.oy)), fabsf(r.oz));
    const float md = fmaxf(fmaxf(fabsf(r.dx), fabsf(r.dy)), fabsf(r.dz));
    float mb = 0.0f, ext = 0.0f;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        mb = fmaxf(mb, fmaxf(fabsf(bb[k]), fabsf(bb[3 + k])));
        ext = fmaxf(ext, bb[3 + k] - bb[k]);
    }
    const float pad = kPad * (mo + mb);
    s.rx = recip(r.dx);
    s.ry = recip(r.dy);
    s.rz = recip(r.dz);
    const float ox = -r.ox * s.rx, oy = -r.oy * s.ry, oz = -r.oz * s.rz;
    const float px = pad * fabsf(s.rx), py = pad * fabsf(s.ry), pz = pad * fabsf(s.rz);
    s.ax = ox - px;
    s.ay = oy - py;
    s.az = oz - pz;
    s.bx = ox + px;
    s.by = oy + py;
    s.bz = oz + pz;
    slack = 2.0f * pad * fminf(fminf(fabsf(s.rx), fabsf(s.ry)), fabsf(s.rz));
    // comparisons with a NaN are false; fmaxf drops one, so every component is tested
    return __builtin_isfinite(r.ox) & __builtin_isfinite(r.oy) & __builtin_isfinite(r.oz) &
           __builtin_isfinite(r.dx) & __builtin_isfinite(r.dy) & __builtin_isfinite(r.dz) & (r.tmin >= 0.0f) &
           !__builtin_isnan(r.tmax) & (mo <= 1e12f) & (mo <= 4096.0f * ext) & (md >= 1e-12f) & (md <= 1e12f);
}

// The Fast-BVH's slab test of one box in the x86-select form (traverse.h node_test).
__device__ __forceinline__ bool box_test(const RayK& r, float lx, float hx, float ly, float hy, float lz, float hz,
                                         float& entry) {
    float fmn = r.tmin, fmx = r.tmax;
    float t1 = r.odx + r.rcx * hx, t2 = r.odx + r.rcx * lx;
    fmn = xmax(fmn, xmin(t1, t2));
    fmx = xmin(fmx, xmax(t1, t2));
    t1 = r.ody + r.rcy * hy;
    t2 = r.ody + r.rcy * ly;
    fmn = xmax(fmn, xmin(t1, t2));
    fmx = xmin(fmx, xmax(t1, t2));
    t1 = r.odz + r.rcz * hz;
    t2 = r.odz + r.rcz * lz;
    fmn = xmax(fmn, xmin(t1, t2));
    fmx = xmin(fmx, xmax(t1, t2));
    entry = fmn;
    return fmn <= fmx;
}

__device__ __forceinline__ void load_ray(const void* rays, uint32_t i, RayK& r) {
    const float4* rp = reinterpret_cast<const float4*>(rays) + 2 * (size_t)i;
    const float4 q0 = rp[0], q1 = rp[1];
    r.ox = q0.x; r.oy = q0.y; r.oz = q0.z; r.tmin = q0.w;
    r.dx = q1.x; r.dy = q1.y; r.dz = q1.z; r.tmax = q1.w;
}

struct Best {
    float t, u, v;
    uint32_t prim;  // kNone: nothing found
    bool any;
};

// The Fast-BVH walk of one ray (trace.hip's, a box and a triangle at a time), for the rays that the
// walk tree leaves open. `st`: the lane's own stack, at least the tree's max_stack entries.
template <bool ANY>
__device__ __forceinline__ void exact_walk(const TreeView& tv, RayK& r, uint2* st, Best& best) {
    best.t = FLT_MAX;
    best.u = best.v = 0.f;
    best.prim = kNone;
    best.any = false;
    ray_setup(r);
    const float rmin = root_slab(r, tv.bbox);
    if (!(rmin >= 0.0f)) return;
    const uint32_t W = tv.width;
    int sp = 0;
    st[sp++] = make_uint2(tv.root, __float_as_uint(rmin));
    while (sp > 0) {
        const uint2 e = st[--sp];
        if (best.t < __uint_as_float(e.y)) continue;
        if (e.x & REF_LEAF) {
            uint32_t li = e.x & ~REF_LEAF;
            while (true) {
                const PrimRec pr = load_prim(tv.prims, li);
                if (pr.id_a & PR_FLAG) {
                    float t;
                    if (quad_test(r, tv.quads[__float_as_uint(pr.a.p0x)], best.t, t)) {
                        best.t = t;
                        best.prim = pr.id_a & PR_ID;
                        best.u = best.v = 0.f;
                        best.any = true;
                    }
                } else {
#pragma unroll 1
                    for (int k = 0; k < 2; k++) {
                        const uint32_t id = (k ? pr.id_b : pr.id_a) & PR_ID;
                        if (id == PR_NONE) break;
                        float t, u, v;
                        const Tri x = k ? pr.b : pr.a;
                        if (tri_test(r, x, t, u, v) && t < best.t) {
                            best.t = t;
                            best.prim = id;
                            best.u = u;
                            best.v = v;
                            best.any = true;
                        }
                    }
                }
                if ((ANY && best.any) || (pr.id_b & PR_FLAG)) break;
                ++li;
            }
            if (ANY && best.any) return;
            continue;
        }
        const float* nd = static_cast<const float*>(tv.nodes) + (size_t)e.x * (W == 8 ? 64 : 32);
        const int base = sp;
#pragma unroll 1
        for (uint32_t j = 0; j < W; j++) {
            const uint32_t ref = __float_as_uint(nd[6 * W + j]);
            float f;
            if (ref == REF_EMPTY ||
                !box_test(r, nd[j], nd[W + j], nd[2 * W + j], nd[3 * W + j], nd[4 * W + j], nd[5 * W + j], f))
                continue;
            // farther below nearer; of equal ones the lower slot below
            int k = sp++;
            while (k > base && __uint_as_float(st[k - 1].y) < f) {
                st[k] = st[k - 1];
                k--;
            }
            st[k] = make_uint2(ref, __float_as_uint(f));
        }
        // three or more hits: only those with an entry distance above -1 (fast_bvh.hpp:438-453)
        if (sp - base >= 3)
            while (sp > base && !(__uint_as_float(st[sp - 1].y) > -1.0f)) sp--;
    }
}

template <bool ANY, bool MULTI, int LDS, int SPILL>
__global__ __launch_bounds__(kBlock) void k_walk(TraceArgs a) {
    __shared__ uint2 s_st[LDS * kBlock];  // (reference, entry distance), [entry][thread]
    constexpr int CAP = LDS + SPILL;
    uint2 sp_st[SPILL];  // deeper entries; also the stack of exact_walk, whose lane has none of its own left

    const uint32_t tid = threadIdx.x;
    const uint32_t lane = __lane_id();
    const uint32_t n_rays = a.n_dev ? *a.n_dev : a.n;
    const uint32_t refill = a.refill ? a.refill : 16u;
    const uint32_t leaf_batch = a.leaf_batch ? a.leaf_batch : 16u;
    const WalkNode* __restrict__ nodes = a.tree.wnodes;
    const PrimRec* __restrict__ recs = a.tree.wrecs;

    RayK r;
    Slabs s;
    uint32_t cur = kNone;  // node or leaf to visit next; kNone: pop the stack
    uint32_t ray_id = kNone;
    uint32_t hit = kNone;  // nearest candidate: record * 2 + (0: A or the quad, 1: B)
    float bt = FLT_MAX, bu = 0.f, bv = 0.f;
    float lim = FLT_MAX;     // search bound: bt and the slack above it
    float second = FLT_MAX;  // second nearest distance met
    float slack = 0.f;
    int sp = 0;
    bool more = true, overflow = false, open = false;  // open: exact_walk has to answer
    // Rays are handed to a wave `chunk` at a time, [own, own_end) still to be started: one atomic on
    // the launch's counter takes about 8.5 ns of the whole chip's time.
    const uint32_t chunk = min(max(n_rays / (gridDim.x * (kBlock / 64) * 8u), 64u), 512u);
    uint32_t own = 0, own_end = 0;

    auto push = [&](uint32_t ref, uint32_t t) {
        if (sp < LDS) s_st[sp * kBlock + tid] = make_uint2(ref, t);
        else if (sp < CAP) sp_st[sp - LDS] = make_uint2(ref, t);
        else overflow = true;
        sp++;
    };

    while (true) {
        const bool idle = cur == kNone && sp == 0;
        const uint64_t want = __ballot(idle && (more || ray_id != kNone));
        const uint64_t busy = __ballot(!idle);
        if (want == 0 && busy == 0) break;
        if (want != 0 && (busy == 0 || (uint32_t)__popcll(want) >= refill)) {
            // ---- answer the rays that are through ----
            if (idle && ray_id != kNone) {
                Best best{bt, bu, bv, kNone, false};
                {
                    if (!open && hit != kNone) {
                        const TreeView& tv = MULTI ? a.trees[a.ray_scene[ray_id]] : a.tree;
                        const float4* xp = reinterpret_cast<const float4*>(tv.waux + (hit >> 1));
                        const float4 x0 = xp[0], x1 = xp[1];
                        best.any = true;
                        if (!ANY) {
                            const uint32_t* rw = reinterpret_cast<const uint32_t*>(tv.wrecs + (hit >> 1));
                            best.prim = rw[18 + (hit & 1u)] & PR_ID;
                        }
                        // the leaf box shrunk by the padding: if even that one is hit, the exact test
                        // passes too, with an entry distance no larger than this one
                        const bool px = s.rx >= 0.0f, py = s.ry >= 0.0f, pz = s.rz >= 0.0f;
                        float entry = fmaxf(fmaxf((px ? x0.x : x0.w) * s.rx + s.bx, (py ? x0.y : x1.x) * s.ry + s.by),
                                            fmaxf((pz ? x0.z : x1.y) * s.rz + s.bz, r.tmin));
                        const float exit = fminf(fminf((px ? x0.w : x0.x) * s.rx + s.ax, (py ? x1.x : x0.y) * s.ry + s.ay),
                                                 fminf((pz ? x1.y : x0.z) * s.rz + s.az, r.tmax));
                        // (beyond 1e5 the exact test steps along another line: it clamps the direction)
                        const bool clamped = fmaxf(fmaxf(fabsf(s.rx), fabsf(s.ry)), fabsf(s.rz)) > 1e5f;
                        const bool inside = entry <= exit && !clamped;
                        auto alone = [&](float e) { return ANY || e <= bt || (e < second && e <= lim); };
                        if (!(second > bt) && !ANY) {
                            open = true;  // a tie
                        } else if (!(inside && alone(entry))) {
                            load_ray(a.rays, ray_id, r);
                            ray_setup(r);
                            open = !box_test(r, x0.x, x0.w, x0.y, x1.x, x0.z, x1.y, entry) || !alone(entry);
                        }
                    }
                    if (open) {
                        const TreeView& tv = MULTI ? a.trees[a.ray_scene[ray_id]] : a.tree;
                        load_ray(a.rays, ray_id, r);
                        exact_walk<ANY>(tv, r, sp_st, best);
                    }
                }
                if (!ANY) {
                    reinterpret_cast<float4*>(a.out)[ray_id] = make_float4(best.t, __uint_as_float(best.prim), best.u, best.v);
                } else if (!a.occ_slot) {
                    static_cast<uint8_t*>(a.out)[ray_id] = best.any ? 1 : 0;
                } else if (best.any) {  // the shadow ray's contribution is cleared here (w kept)
                    const uint32_t slot = a.occ_slot[ray_id];
                    float* c = reinterpret_cast<float*>(a.occ_rec + 4 * (size_t)(slot >> 1) + 2 + (slot & 1u));
                    c[0] = 0.f;
                    c[1] = 0.f;
                    c[2] = 0.f;
                }
                ray_id = kNone;
            }
            // ---- take new ones ----
            const uint64_t take = __ballot(idle && more);
            if (take != 0) {
                const uint32_t cnt = (uint32_t)__popcll(take), left = own_end - own;
                uint32_t next = 0;
                if (cnt > left) {
                    if (lane == 0) next = atomicAdd(a.counter, chunk);
                    next = __builtin_amdgcn_readfirstlane(next);
                }
                const uint32_t rank = (uint32_t)__popcll(take & ((1ull << lane) - 1ull));
                const uint32_t k = rank < left ? own + rank : next + (rank - left);
                if (cnt > left) {
                    own = next + (cnt - left);
                    own_end = next + chunk;
                } else {
                    own += cnt;
                }
                if (idle && more) {
                    if (k < n_rays) {
                        const uint32_t my = a.order ? a.order[k] : k;
                        load_ray(a.rays, my, r);
                        bt = lim = second = FLT_MAX;
                        bu = bv = 0.f;
                        hit = kNone;
                        open = false;
                        bool known = true;  // the scene id is one of the table's
                        const TreeView* tv = &a.tree;
                        if (MULTI) {
                            const uint32_t sid = a.ray_scene[my];
                            known = sid < a.n_trees;
                            if (!known) atomicOr(a.error, kFlagBadScene);
                            tv = a.trees + (known ? sid : 0u);
                            nodes = tv->wnodes;
                            recs = tv->wrecs;
                        }
                        const bool fits = slabs_setup(r, tv->bbox, s, slack);
                        shear_setup(r, s);
                        // a ray outside the bounds goes to the exact walk, with its root test
                        if (known && tv->valid && (!fits || root_test(r, s, tv->bbox))) {
                            ray_id = my;
                            if (fits) cur = 0;
                            else open = true;
                        } else if (!ANY) {
                            reinterpret_cast<float4*>(a.out)[my] = make_float4(FLT_MAX, __uint_as_float(kNone), 0.f, 0.f);
                        } else if (!a.occ_slot) {
                            static_cast<uint8_t*>(a.out)[my] = 0;
                        }
                    } else {
                        more = false;
                    }
                }
            }
            continue;
        }
        // ---- node phase: lanes that hold no leaf step through inner nodes ----
        while (true) {
            const bool walk = (int32_t)cur >= 0 || (cur == kNone && sp > 0);
            if (__ballot(walk) == 0 || (uint32_t)__popcll(__ballot(cur != kNone && (int32_t)cur < 0)) >= leaf_batch) break;
            if (walk && cur == kNone) {
                --sp;
                // the LDS read is unconditional (clamped index) so that it stays an LDS access
                uint2 e = s_st[(sp < LDS ? sp : LDS - 1) * kBlock + tid];
                if (sp >= LDS) e = sp_st[sp - LDS < SPILL ? sp - LDS : 0];
                if (__uint_as_float(e.y) <= lim) cur = e.x;
            }
            if (walk && (int32_t)cur >= 0) {
                const uint4* np = reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(nodes) + cur * 48u);
                const uint4 q0 = np[0], q1 = np[1], q2 = np[2];
                const uint32_t meta = q0.w;
                const uint32_t ni = (meta >> 24) & 15u, nc = meta >> 28;
                const float gx = __uint_as_float((meta & 0xffu) << 23) * s.rx;
                const float gy = __uint_as_float(((meta >> 8) & 0xffu) << 23) * s.ry;
                const float gz = __uint_as_float(((meta >> 16) & 0xffu) << 23) * s.rz;
                const float bx = __uint_as_float(q0.x) * s.rx, by = __uint_as_float(q0.y) * s.ry,
                            bz = __uint_as_float(q0.z) * s.rz;
                const float nx = bx + s.ax, ny = by + s.ay, nz = bz + s.az;
                const float fx = bx + s.bx, fy = by + s.by, fz = bz + s.bz;
                const bool px = s.rx >= 0.0f, py = s.ry >= 0.0f, pz = s.rz >= 0.0f;
                const uint32_t wnx = px ? q1.z : q1.w, wfx = px ? q1.w : q1.z;
                const uint32_t wny = py ? q2.x : q2.y, wfy = py ? q2.y : q2.x;
                const uint32_t wnz = pz ? q2.z : q2.w, wfz = pz ? q2.w : q2.z;
                const float hi = fminf(r.tmax, lim);
                uint32_t key[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    auto q = [&](uint32_t w) { return (float)((w >> (8 * j)) & 0xffu); };
                    const float t0 = fmaxf(fmaxf(__builtin_fmaf(q(wnx), gx, nx), __builtin_fmaf(q(wny), gy, ny)),
                                           fmaxf(__builtin_fmaf(q(wnz), gz, nz), r.tmin));
                    const float t1 = fminf(fminf(__builtin_fmaf(q(wfx), gx, fx), __builtin_fmaf(q(wfy), gy, fy)),
                                           fminf(__builtin_fmaf(q(wfz), gz, fz), hi));
                    // distances are not negative: their bits order as they do; the slot rides in the last two
                    const bool in = (t0 <= t1) & ((uint32_t)j < nc);
                    key[j] = in ? ((__float_as_uint(t0) & ~3u) | (uint32_t)j) : kNone;
                }
                const uint32_t leaf_at = (q1.y | REF_LEAF) - ni;
                auto ref = [&](uint32_t k) {
                    const uint32_t j = k & 3u;
                    return (j < ni ? q1.x : leaf_at) + j;
                };
                auto order = [&](uint32_t& x, uint32_t& y) {
                    const uint32_t lo = min(x, y), up = max(x, y);
                    x = lo;
                    y = up;
                };
                order(key[0], key[1]);
                order(key[2], key[3]);
                order(key[0], key[2]);
                order(key[1], key[3]);
                order(key[1], key[2]);
                if (key[3] != kNone) push(ref(key[3]), key[3]);
                if (key[2] != kNone) push(ref(key[2]), key[2]);
                if (key[1] != kNone) push(ref(key[1]), key[1]);
                cur = key[0] != kNone ? ref(key[0]) : kNone;
                // only reachable on overflow (the host sizes the stack for the tree)
                if (sp > CAP) sp = CAP;
            }
        }
        // ---- leaf phase: every lane that holds a leaf tests its record ----
        if (cur != kNone && (int32_t)cur < 0) {
            const uint32_t ri = cur & ~REF_LEAF;
            const PrimRec pr = load_prim(recs, ri);
            cur = kNone;
            // A tie of two triangles of one Fast-BVH leaf (a mesh with doubled faces has one at every
            // hit): the one that comes first there wins. False: not such a tie.
            float tie_u = 0.f, tie_v = 0.f;
            auto same_leaf_order = [&](uint32_t rec, uint32_t which) {
                if (rec == hit >> 1) return (pr.id_a & PR_FLAG) == 0;  // A and B of one record: A comes first
                const TreeView& tv = MULTI ? a.trees[a.ray_scene[ray_id]] : a.tree;
                const WalkAux &x = tv.waux[rec], &y = tv.waux[hit >> 1];
                const uint32_t px = (x.places >> (16u * which)) & 0xffffu, py = (y.places >> (16u * (hit & 1u))) & 0xffffu;
                if (x.leaf != y.leaf || px == 0xffffu || py == 0xffffu || (pr.id_a & PR_FLAG) ||
                    (recs[hit >> 1].id_a & PR_FLAG))
                    return false;
                if (px < py) {
                    hit = 2 * rec + which;
                    bu = tie_u;
                    bv = tie_v;
                }
                return true;
            };
            auto found = [&](float t, float u, float v, uint32_t which) {
                tie_u = u;
                tie_v = v;
                if (t < bt) {
                    second = bt;
                    bt = t;
                    bu = u;
                    bv = v;
                    hit = 2 * ri + which;
                    lim = t + (slack + 4e-7f * t);
                } else if (!ANY) {
                    if (t == bt && same_leaf_order(ri, which)) return;
                    second = fminf(second, t);
                }
            };
            if (pr.id_a & PR_FLAG) {
                const TreeView& tv = MULTI ? a.trees[a.ray_scene[ray_id]] : a.tree;
                RayK w;
                load_ray(a.rays, ray_id, w);
                float t;
                if (quad_test(w, tv.quads[__float_as_uint(pr.a.p0x)], FLT_MAX, t)) found(t, 0.f, 0.f, 0u);
            } else {
                float t, u, v;
                if (tri_test(r, pr.a, t, u, v)) found(t, u, v, 0u);
                if ((pr.id_b & PR_ID) != PR_NONE && tri_test(r, pr.b, t, u, v)) found(t, u, v, 1u);
            }
            if (ANY && hit != kNone) sp = 0;
        }
    }
    if (overflow) atomicOr(a.error, kFlagStackOverflow);
}

__global__ void k_walk_reset(uint32_t* counter) {
    if (threadIdx.x == 0) *counter = 0;
}

template <bool ANY, bool MULTI, int LDS, int SPILL>
hipError_t launch(const TraceArgs& a, hipStream_t stream, int num_cus) {
    auto kern = k_walk<ANY, MULTI, LDS, SPILL>;
    int per_cu = 0;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, kBlock, 0);
    if (e != hipSuccess) return e;
    if (per_cu < 1) per_cu = 1;
    if (a.blocks_per_cu && (int)a.blocks_per_cu < per_cu) per_cu = (int)a.blocks_per_cu;
    const uint64_t want = ((uint64_t)a.n + kBlock - 1) / kBlock;
    uint64_t grid = (uint64_t)num_cus * (uint64_t)per_cu;
    if (want < grid) grid = want;
    if (grid < 1) grid = 1;
    hipLaunchKernelGGL(k_walk_reset, dim3(1), dim3(64), 0, stream, a.counter);
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(kBlock), 0, stream, a);
    return hipGetLastError();
}

template <bool ANY, bool MULTI, int LDS>
hipError_t launch_spill(const TraceArgs& a, hipStream_t stream, int num_cus) {
    const uint32_t walk = MULTI ? a.walk_stack : a.tree.walk_stack;
    const uint32_t exact = MULTI ? a.max_stack : a.tree.max_stack;
    if (walk <= LDS + 64 && exact <= 64) return launch<ANY, MULTI, LDS, 64>(a, stream, num_cus);
    if (walk <= LDS + 256 && exact <= 256) return launch<ANY, MULTI, LDS, 256>(a, stream, num_cus);
    return hipErrorInvalidValue;
}

template <bool ANY, bool MULTI>
hipError_t launch_lds(const TraceArgs& a, hipStream_t stream, int num_cus) {
    return a.lds_entries == 8 ? launch_spill<ANY, MULTI, 8>(a, stream, num_cus)
                              : launch_spill<ANY, MULTI, 16>(a, stream, num_cus);
}

}  // namespace

hipError_t launch_walk(const TraceArgs& a, bool any, hipStream_t stream, int num_cus) {
    if (a.trees) return any ? launch_lds<true, true>(a, stream, num_cus) : launch_lds<false, true>(a, stream, num_cus);
    return any ? launch_lds<true, false>(a, stream, num_cus) : launch_lds<false, false>(a, stream, num_cus);
}

}  // namespace sortgpu
