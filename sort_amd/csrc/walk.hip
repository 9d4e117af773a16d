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

constexpr float FLT_INF = __builtin_inff();

// Three floats at any word, as one load.
struct __attribute__((packed, aligned(4))) Float3 {
    float x, y, z;
};

// The value of the even lane of this lane's pair; the value of the pair's other lane.
__device__ __forceinline__ uint32_t quad_even(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xA0, 0xf, 0xf, true);  // quad_perm [0, 0, 2, 2]
}
__device__ __forceinline__ float quad_swap(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xB1, 0xf, 0xf, true));  // [1, 0, 3, 2]
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
// 4 waves per SIMD (128 VGPRs): 5 spilled in the rarely taken parts and gained nothing.
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4))) void k_walk(TraceArgs a) {
    __shared__ uint2 s_st[LDS * kBlock];  // (reference, entry distance), [entry][thread]
    constexpr int CAP = LDS + SPILL;
    uint2 sp_st[SPILL];  // deeper entries; also the stack of exact_walk, whose lane has none of its own left

    const uint32_t tid = threadIdx.x;
    const uint32_t lane = __lane_id();
    const uint32_t n_rays = a.n_dev ? *a.n_dev : a.n;
    const uint32_t refill = a.refill ? a.refill : 16u;
    const uint32_t leaf_batch = a.leaf_batch ? a.leaf_batch : 24u;
    const WalkNode* __restrict__ nodes = a.tree.wnodes;
    const PrimRec* __restrict__ recs = a.tree.wrecs;

    RayK r;
    Slabs s;
    uint32_t cur = kNone;   // node to visit next (or the next leaf, while `leaf` is taken); kNone: pop the stack
    uint32_t leaf = kNone;  // leaf waiting for the wave's leaf phase
    uint32_t ray_id = kNone;
    uint32_t hit = kNone;  // nearest candidate: record * 2 + (0: A or the quad, 1: B)
    float bt = FLT_MAX, bu = 0.f, bv = 0.f;
    float lim = FLT_MAX;     // search bound: the window's end, then bt and the slack above it
    float second = FLT_MAX;  // second nearest distance met
    float slack = 0.f;
    int sp = 0;
    bool more = true, overflow = false, open = false;  // open: exact_walk has to answer
    // Handing out the rays. One atomic on the launch's counter takes about 8.5 ns of the whole chip's
    // time (measured: 4.19M rays, 16 at a time, spent 2.2 ms there), so every workgroup has a share of
    // its own that its waves take from through LDS. Of a large batch only three quarters are shares,
    // dealt 64 rays at a time so that all workgroups move through the order together (a contiguous
    // share each has them all over the tree at once: 2.05 instead of 1.87 ms for 4.19M
    // bounce rays); the rest goes out
    // through the counter, in chunks that shrink with what is left, so that the workgroups end
    // together. A batch with less than a full wave of rays for each wave spreads over all of them, on
    // the first `seats` lanes of each.
    const uint32_t waves = gridDim.x * (kBlock / 64);
    const uint32_t seats = min((n_rays + waves - 1) / waves, 64u);
    const bool dealt = n_rays >= 128u * waves;
    const uint32_t share = dealt ? (n_rays - n_rays / 4u) / (gridDim.x * 64u) * 64u : (n_rays + gridDim.x - 1) / gridDim.x;
    const uint32_t pooled = min(share * gridDim.x, n_rays);  // first ray that the counter hands out
    __shared__ uint32_t s_next, s_out;  // rays of the share taken; whether the counter has run out
    if (tid == 0) {
        s_next = 0;
        s_out = pooled >= n_rays ? 1u : 0u;
    }
    __syncthreads();
    bool sharing = true;             // the share may have rays left
    uint32_t own = 0, own_end = 0;   // this wave's chunk of the rest
    more = lane < seats;


    while (true) {
        const bool idle = cur == kNone && leaf == kNone && sp == 0;
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
                const uint32_t cnt = (uint32_t)__popcll(take);
                const uint32_t rank = (uint32_t)__popcll(take & ((1ull << lane) - 1ull));
                uint32_t k = 0;
                bool given = false, out = false;  // a lane without a ray waits for the next refill; out: there is none
                if (sharing) {
                    uint32_t v = 0;
                    if (lane == 0) v = atomicAdd(&s_next, cnt);
                    v = __builtin_amdgcn_readfirstlane(v);
                    sharing = v + cnt < share;
                    v += rank;
                    k = dealt ? ((((v >> 6) * gridDim.x + blockIdx.x) << 6) | (v & 63u)) : blockIdx.x * share + v;
                    given = v < share && k < pooled;
                } else {
                    if (own == own_end) {
                        uint32_t done = 0;
                        if (lane == 0) done = __hip_atomic_load(&s_out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                        out = __builtin_amdgcn_readfirstlane(done) != 0;
                        if (!out) {
                            const uint32_t rest = n_rays - max(own_end, pooled);
                            const uint32_t chunk = max(min(rest / (2u * waves), 256u), 32u);
                            if (lane == 0) own = atomicAdd(a.counter, chunk);
                            own = pooled + __builtin_amdgcn_readfirstlane(own);
                            own_end = min(own + chunk, n_rays);
                            out = own >= n_rays;
                            if (out && lane == 0)
                                __hip_atomic_store(&s_out, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                        }
                    }
                    k = own + rank;
                    given = k < own_end;
                    own = min(own + cnt, own_end);
                }
                if (out) more = false;
                if (idle && more) {
                    if (given) {
                        const uint32_t my = a.order ? a.order[k] : k;
                        load_ray(a.rays, my, r);
                        bt = second = FLT_MAX;
                        lim = r.tmax;
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
                    }
                }
            }
            continue;
        }
        // ---- node phase: lanes step through inner nodes; the first leaf that one meets waits while it
        // walks on, the second stops it ----
        // `leaf_batch` of 64 lanes at work, in proportion of fewer (a fixed number has a thinly filled
        // wave walk on and on past the leaves that would have ended its rays: 1.87 -> 1.74 ms for 4.19M
        // bounce rays, 0.47 -> 0.44 for 2.07M camera rays)
        const uint32_t batch = (leaf_batch * (uint32_t)__popcll(busy) + 63u) / 64u;
        while (true) {
            const bool walk = (int32_t)cur >= 0 || (cur == kNone && sp > 0);
            if (__ballot(walk) == 0 || (uint32_t)__popcll(__ballot(leaf != kNone)) >= batch) break;
            const bool pop = walk && cur == kNone;
            // Stack accesses are LDS ones unless some lane of the wave is past the entries there: a
            // choice per lane would make every access a generic one.
            if (__ballot(pop && sp > LDS) == 0) {
                if (pop) {
                    --sp;
                    const uint2 e = s_st[sp * kBlock + tid];
                    if (__uint_as_float(e.y) <= lim) cur = e.x;
                }
            } else if (pop) {
                --sp;
                uint2 e;
                if (sp < LDS) e = s_st[sp * kBlock + tid];
                else e = sp_st[min(sp - LDS, SPILL - 1)];
                if (__uint_as_float(e.y) <= lim) cur = e.x;
            }
            if (walk && (int32_t)cur >= 0) {
                const uint4* np = reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(nodes) + (((cur << 1) + cur) << 4));
                const uint4 q0 = np[0], q1 = np[1], q2 = np[2];
                const uint32_t meta = q0.w;
                const uint32_t ni = (meta >> 24) & 15u;
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
                uint32_t key[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    auto q = [&](uint32_t w) { return (float)((w >> (8 * j)) & 0xffu); };
                    const float t0 = fmaxf(fmaxf(__builtin_fmaf(q(wnx), gx, nx), __builtin_fmaf(q(wny), gy, ny)),
                                           fmaxf(__builtin_fmaf(q(wnz), gz, nz), r.tmin));
                    const float t1 = fminf(fminf(__builtin_fmaf(q(wfx), gx, fx), __builtin_fmaf(q(wfy), gy, fy)),
                                           fminf(__builtin_fmaf(q(wfz), gz, fz), lim));
                    // distances are not negative: their bits order as they do; the slot rides in the last two
                    key[j] = t0 <= t1 ? ((__float_as_uint(t0) & ~3u) | (uint32_t)j) : kNone;
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
                // Farthest first. An entry that is no hit is written as well and then written over:
                // the slot above the top is free.
                if (__ballot(sp + 3 > LDS) == 0) {
#pragma unroll
                    for (int i = 3; i >= 1; i--) {
                        s_st[sp * kBlock + tid] = make_uint2(ref(key[i]), key[i]);
                        sp += key[i] != kNone ? 1 : 0;
                    }
                } else {
#pragma unroll
                    for (int i = 3; i >= 1; i--) {
                        if (key[i] == kNone) continue;
                        const uint2 e = make_uint2(ref(key[i]), key[i]);
                        if (sp < LDS) s_st[sp * kBlock + tid] = e;
                        else if (sp < CAP) sp_st[sp - LDS] = e;
                        // not reached: the host sizes the stack for the tree
                        if (sp < CAP) sp++;
                        else overflow = true;
                    }
                }
                cur = key[0] != kNone ? ref(key[0]) : kNone;
            }
            if (cur != kNone && (int32_t)cur < 0 && leaf == kNone) {
                leaf = cur;
                cur = kNone;
            }
        }
        // ---- leaf phase: the waiting leaves' triangles, one to a lane ----
        // Leaf number i of the wave has its A tested by lane 2i and its B by lane 2i + 1, with the ray
        // fetched from the lane that owns it: twenty leaves keep forty lanes busy for one triangle's
        // time, where their owners would take two. At most 32 leaves a round; others wait.
        const uint64_t holders = __ballot(leaf != kNone);
        if (holders == 0) continue;
        const uint32_t rank = (uint32_t)__popcll(holders & ((1ull << lane) - 1ull));
        const bool mine = leaf != kNone && rank < 32u;
        // lane 2i learns which lane owns leaf i; lane 2i + 1 has it from its neighbour
        int owner = __builtin_amdgcn_ds_permute((int)((mine ? 2u * rank : 63u) << 2), mine ? (int)lane : -1);
        owner = (int)quad_even((uint32_t)owner);
        const bool tester = (lane >> 1) < (uint32_t)__popcll(holders);
        const int from = owner << 2;
        auto fetch = [&](float x) { return __int_as_float(__builtin_amdgcn_ds_bpermute(from, __float_as_int(x))); };
        RayK w;
        w.okx = fetch(r.okx); w.oky = fetch(r.oky); w.okz = fetch(r.okz);
        w.sx = fetch(r.sx); w.sy = fetch(r.sy); w.sz = fetch(r.sz);
        w.tmin = fetch(r.tmin);
        w.tmax = fetch(r.tmax);
        w.ky = __builtin_amdgcn_ds_bpermute(from, r.ky);
        const uint32_t ri = leaf & ~REF_LEAF;
        const char* tp = nullptr;
        if (MULTI) {
            const uint64_t at = reinterpret_cast<uint64_t>(recs + ri);
            const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)(uint32_t)at);
            const uint32_t up = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)(uint32_t)(at >> 32));
            tp = reinterpret_cast<const char*>(((uint64_t)up << 32) | lo);
        } else {
            const uint32_t at = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)(ri * (uint32_t)sizeof(PrimRec)));
            tp = reinterpret_cast<const char*>(recs) + at;
        }
        float t = FLT_INF, u = 0.f, v = 0.f;
        bool quad = false;
        if (tester) {
            w.kz = w.ky == 2 ? 0 : w.ky + 1;
            w.kx = w.kz == 2 ? 0 : w.kz + 1;
            const Float3* vp = reinterpret_cast<const Float3*>(tp + (lane & 1u) * sizeof(Tri));
            const Float3 p0 = vp[0], p1 = vp[1], p2 = vp[2];
            const Tri x{p0.x, p0.y, p0.z, p1.x, p1.y, p1.z, p2.x, p2.y, p2.z};
            quad = __builtin_isnan(p1.x);  // a quad's record (no triangle of a walk tree holds a NaN)
            float tt, uu, vv;
            if (tri_test(w, x, tt, uu, vv)) {
                t = tt;
                u = uu;
                v = vv;
            }
        }
        // the nearer of A and B (A where they are equal), and the other one's distance
        const float to = quad_swap(t), uo = quad_swap(u), vo = quad_swap(v);
        const bool take_b = to < t;  // as lane 2i sees it
        float other = take_b ? t : (to == t ? FLT_INF : to);
        if (quad) other = -1.0f;
        const int back = (int)((2u * min(rank, 31u)) << 2);
        auto result = [&](float x) { return __int_as_float(__builtin_amdgcn_ds_bpermute(back, __float_as_int(x))); };
        const float rt = result(take_b ? to : t), ru = result(take_b ? uo : u), rv = result(take_b ? vo : v);
        const float ro = result(other);
        const bool rb = __builtin_amdgcn_ds_bpermute(back, take_b ? 1 : 0) != 0;
        if (mine) {
            leaf = kNone;
            if (cur != kNone && (int32_t)cur < 0) {
                leaf = cur;
                cur = kNone;
            }
            // A tie of two triangles of one Fast-BVH leaf (a mesh with doubled faces has one at every
            // hit): the one that comes first there wins. False: not such a tie.
            auto same_leaf_order = [&](uint32_t which, float tie_u, float tie_v) {
                const TreeView& tv = MULTI ? a.trees[a.ray_scene[ray_id]] : a.tree;
                if ((recs[ri].id_a & PR_FLAG) || (recs[hit >> 1].id_a & PR_FLAG)) return false;
                if (ri == hit >> 1) return true;  // the same record again
                const WalkAux &x = tv.waux[ri], &y = tv.waux[hit >> 1];
                const uint32_t px = (x.places >> (16u * which)) & 0xffffu, py = (y.places >> (16u * (hit & 1u))) & 0xffffu;
                if (x.leaf != y.leaf || px == 0xffffu || py == 0xffffu) return false;
                if (px < py) {
                    hit = 2 * ri + which;
                    bu = tie_u;
                    bv = tie_v;
                }
                return true;
            };
            auto found = [&](float ft, float fu, float fv, uint32_t which) {
                if (ft < bt) {
                    second = bt;
                    bt = ft;
                    bu = fu;
                    bv = fv;
                    hit = 2 * ri + which;
                    lim = ft + (slack + 4e-7f * ft);
                } else if (!ANY && !(ft == bt && same_leaf_order(which, fu, fv))) {
                    second = fminf(second, ft);
                }
            };
            if (ro < 0.0f) {
                const TreeView& tv = MULTI ? a.trees[a.ray_scene[ray_id]] : a.tree;
                RayK q;
                load_ray(a.rays, ray_id, q);
                float ft;
                if (quad_test(q, tv.quads[__float_as_uint(recs[ri].a.p0x)], FLT_MAX, ft)) found(ft, 0.f, 0.f, 0u);
            } else if (rt < FLT_INF) {
                found(rt, ru, rv, rb ? 1u : 0u);
                second = fminf(second, ro);
            }
            if (ANY && hit != kNone) {
                sp = 0;
                cur = leaf = kNone;
            }
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
    // as many waves as run at once, down to four rays each
    const uint64_t want = ((uint64_t)a.n + 15) / 16;
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
