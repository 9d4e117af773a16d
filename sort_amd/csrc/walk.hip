// Closest-hit and any-hit queries over the walk tree (walk_tree.h), with the Fast-BVH's results.
//
// What a query returns is defined by the Fast-BVH walk of trace.hip: hits count only in leaves
// whose box the ray's slab test accepts, leaves are pruned by their entry distance, and equal hits
// go to the one met first. This kernel finds candidates in a tree of its own (4-wide nodes of 48
// bytes, at most two triangles to a leaf) and then shows that the walk would have returned the same:
//
//   * The candidates are complete: below.
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
// numbers leave the bounds below (NaN, infinities, a negative tmin, an origin very far out), is walked
// again through the Fast-BVH by its lane, in `exact_walk`. Any hit needs less: the first candidate
// whose leaf box passes.
//
// Why the candidates are complete. Let u = 2^-24, M the largest coordinate of origin and scene, D that of a
// vertex relative to the origin. Take a triangle with longest edge L and height H over it, in a leaf whose box
// the exact test passes, at R at most across (times sqrt(3), for the shear), and accepted by the triangle test
// at t. The test sees its corners projected along the ray, wrong by e = 5.7 u D + u R; it takes the signs of the
// three products of two corners, and a sign is right unless the ray sees the two within an angle of u (or
// pi - u). So either the ray passes within rounding of the triangle, or it sees all of it within 2 u, however
// far beside it: a flat sheet edge-on, a needle, a triangle of the rounding's own size. The Fast-BVH has such
// hits all over the leaf's box (at up to 16 triangles to a leaf), where no box of the triangle's reaches.
//   - Beside: all three corners lie within u R + e of one plane through the ray, so the ray's direction lies
//     within 2.83 (u R + e) / H of the triangle's plane. Within 8 e / H of it, too, rounding may take half of the
//     projected area. Such triangles are the gates' matter: each Fast-BVH leaf's part of the walk tree starts
//     at a node of its own (a gated node) with all its triangles' normals in four bytes each, and a ray that
//     comes there is tested against each triangle whose plane it is that near to, whatever its box says
//     (kGateReach, kGateLeaf; normals in 127ths add 0.0137).
//   - Otherwise t is a mean of the corners' distances with weights that are off by 6 u R R over the projected
//     area, so that the ray's point at t lies within 36 u L L / (H s) + e of the triangle where its direction is
//     more than s off the plane. What of this is more than L / 256, by which a triangle's box is widened, is again
//     the gates' matter (kGateShape). The rest, with the rounding of the slab distances (10 u M, the Fast-BVH's own
//     4 among them) and of t (8 u M), is below the 32 u M that every slab is widened by.
//   - So a leaf's boxes are met where they matter, and the node at its top wherever the exact test passes the
//     leaf's box. That test steps along a direction with no component below 1e-5: slabs of smaller ones are
//     widened by what that strays. And a gate's hit may lie before its leaf's entry, so that no box is left out
//     for its entry distance but only where it starts past `lim` on the ray's main axis: t is a mean of
//     distances on that axis.
// Scenes below 1e-8 have no walk tree: products would be lost to underflow. A quad is tested in its own space:
// its rounding there, and what its two matrices disagree by, are in the tree's padding (walk_tree.cpp).
// tests/native/walk_complete_check.cpp looks for counterexamples with this arithmetic on the CPU.
//
// What it costs and saves: on the benchmark's 4,194,304 bounce rays through 2^20 triangles a ray of the
// Fast-BVH walk tests 14.8 nodes and 81.5 triangles, reading 391 chunks of 16 bytes; here it tests 35.7
// nodes, the boxed triangles of 6.2 records, 46 records' normals at 7.6 gates and two triangles behind them.
// The call takes 2.19 instead of 4.35 ms; 1.5M shadow segments through 300K triangles 0.91 instead of 1.79, 2M camera
// rays on 768K triangles of spheres 0.36 instead of 0.80. Without the gates and with boxes left out for their
// entry distances, and other answers for the rays above, it was 1.57, 0.69 and 0.30. Gates seen to by each ray's
// own lane in the node step took 3.04, 1.23 and 0.40: one node in five has one. (The figures beside the choices
// further down are from before the gates.)
// Leaves of one triangle instead of two: 2 to 3 steps more per ray on meshes. 8-wide nodes: a third of the steps
// less, each with twice the arithmetic.
#include <hip/hip_runtime.h>

#include <atomic>

#include "trace_launch.h"
#include "traverse.h"
#include "walk_step.h"

#pragma clang fp contract(off)

namespace sortgpu {
namespace {

constexpr int kBlock = 256;
constexpr uint32_t kDealtPerWave = 128;  // rays per wave from which part of a batch goes out through the counter
constexpr uint32_t kQuadsPerWave = 28;   // rays per wave up to which four lanes take a ray together

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

// The value of the even lane of this lane's pair; of the pair's other lane; of another lane of its four.
__device__ __forceinline__ uint32_t pair_even(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xA0, 0xf, 0xf, true);  // quad_perm [0, 0, 2, 2]
}
__device__ __forceinline__ float pair_swap(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xB1, 0xf, 0xf, true));  // [1, 0, 3, 2]
}
template <int PERM>
__device__ __forceinline__ uint32_t quad_rot(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, PERM, 0xf, 0xf, true);
}
template <int PERM>
__device__ __forceinline__ float quad_rot_f(float x) { return __uint_as_float(quad_rot<PERM>(__float_as_uint(x))); }

// How many lanes below this one are in `m`.
__device__ __forceinline__ uint32_t rank_in(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
// Another lane's value.
__device__ __forceinline__ uint32_t of_lane(uint32_t lane, uint32_t x) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(lane << 2), (int)x);
}
__device__ __forceinline__ float of_lane(uint32_t lane, float x) { return __uint_as_float(of_lane(lane, __float_as_uint(x))); }
template <class T>
__device__ __forceinline__ const T* of_lane(uint32_t lane, const T* x) {
    const uint64_t at = reinterpret_cast<uint64_t>(x);
    return reinterpret_cast<const T*>((uint64_t)of_lane(lane, (uint32_t)(at >> 32)) << 32 | of_lane(lane, (uint32_t)at));
}

// The gate words of two records, and which of their triangles they let a ray through to.
struct __attribute__((aligned(8))) GateWords {
    uint32_t a, b, c, d;
    __device__ __forceinline__ uint32_t open(uint32_t dir, uint32_t bound) const {
        return (gate_open(a, dir, bound) ? 1u : 0u) | (gate_open(b, dir, bound) ? 2u : 0u) |
               (gate_open(c, dir, bound) ? 4u : 0u) | (gate_open(d, dir, bound) ? 8u : 0u);
    }
};

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

// A ray on its way through a walk tree.
struct Walker {
    RayK r;
    Slabs s;
    const WalkNode* nodes;
    const PrimRec* recs;
    uint32_t cur;     // node to visit next (or the next leaf, while `leaf` is taken); kNone: pop the stack
    uint32_t leaf;    // leaf waiting for the wave's leaf phase
    uint32_t ray_id;  // kNone: no ray
    uint32_t hit;     // nearest candidate: record * 2 + (0: A or the quad, 1: B)
    float bt, bu, bv;
    float lim;        // search bound: the window's end, then bt and the slack above it
    float second;     // second nearest distance met
    int sp;
    bool open;        // exact_walk has to answer

    __device__ __forceinline__ bool idle() const { return cur == kNone && leaf == kNone && sp == 0; }
    __device__ __forceinline__ bool walking() const { return (int32_t)cur >= 0 || (cur == kNone && sp > 0); }
    __device__ __forceinline__ bool at_leaf() const { return cur != kNone && (int32_t)cur < 0; }
};

// Takes up ray `my`, or answers it where the scene's box already does.
template <bool ANY, bool MULTI>
__device__ __forceinline__ void start(const TraceArgs& a, uint32_t my, Walker& w, float& slack, uint32_t& gate) {
    load_ray(a.rays, my, w.r);
    w.bt = w.second = FLT_MAX;
    w.lim = w.r.tmax;
    w.bu = w.bv = 0.f;
    w.hit = kNone;
    w.open = false;
    bool known = true;  // the scene id is one of the table's
    const TreeView* tv = &a.tree;
    if (MULTI) {
        const uint32_t sid = a.ray_scene[my];
        known = sid < a.n_trees;
        if (!known) atomicOr(a.error, kFlagBadScene);
        tv = a.trees + (known ? sid : 0u);
        w.nodes = tv->wnodes;
        w.recs = tv->wrecs;
    }
    const bool fits = slabs_setup(w.r, tv->bbox, tv->walk_pad, w.s, slack, gate);
    shear_setup(w.r, w.s);
    // a ray outside the bounds goes to the exact walk, with its root test
    if (known && tv->valid && (!fits || root_test(w.r, w.s, tv->bbox))) {
        w.ray_id = my;
        if (fits) w.cur = 0;
        else w.open = true;
    } else if (!ANY) {
        reinterpret_cast<float4*>(a.out)[my] = make_float4(FLT_MAX, __uint_as_float(kNone), 0.f, 0.f);
    } else if (!a.occ_slot) {
        static_cast<uint8_t*>(a.out)[my] = 0;
    }
}

// Answers the walker's ray: shows that the Fast-BVH walk returns its candidate, or walks that tree.
template <bool ANY, bool MULTI>
__device__ __forceinline__ void settle(const TraceArgs& a, Walker& w, uint2* st) {
    const Slabs& s = w.s;
    RayK& r = w.r;
    Best best{w.bt, w.bu, w.bv, kNone, false};
    if (!w.open && w.hit != kNone) {
        const TreeView& tv = MULTI ? a.trees[a.ray_scene[w.ray_id]] : a.tree;
        const float4* xp = reinterpret_cast<const float4*>(tv.waux + (w.hit >> 1));
        const float4 x0 = xp[0], x1 = xp[1];
        best.any = true;
        if (!ANY) {
            const uint32_t* rw = reinterpret_cast<const uint32_t*>(tv.wrecs + (w.hit >> 1));
            best.prim = rw[18 + (w.hit & 1u)] & PR_ID;
        }
        // the leaf box shrunk by the padding: if even that one is hit, the exact test passes too, with
        // an entry distance no larger than this one
        const bool px = s.rx >= 0.0f, py = s.ry >= 0.0f, pz = s.rz >= 0.0f;
        float entry = fmaxf(fmaxf((px ? x0.x : x0.w) * s.rx + s.bx, (py ? x0.y : x1.x) * s.ry + s.by),
                            fmaxf((pz ? x0.z : x1.y) * s.rz + s.bz, r.tmin));
        const float exit = fminf(fminf((px ? x0.w : x0.x) * s.rx + s.ax, (py ? x1.x : x0.y) * s.ry + s.ay),
                                 fminf((pz ? x1.y : x0.z) * s.rz + s.az, r.tmax));
        // (beyond 1e5 the exact test steps along another line: it clamps the direction)
        const bool clamped = fmaxf(fmaxf(fabsf(s.rx), fabsf(s.ry)), fabsf(s.rz)) > 1e5f;
        const bool inside = entry <= exit && !clamped;
        auto alone = [&](float e) { return ANY || e <= w.bt || (e < w.second && e <= w.lim); };
        if (!(w.second > w.bt) && !ANY) {
            w.open = true;  // a tie
        } else if (!(inside && alone(entry))) {
            load_ray(a.rays, w.ray_id, r);
            ray_setup(r);
            w.open = !box_test(r, x0.x, x0.w, x0.y, x1.x, x0.z, x1.y, entry) || !alone(entry);
        }
    }
    if (w.open) {
        const TreeView& tv = MULTI ? a.trees[a.ray_scene[w.ray_id]] : a.tree;
        load_ray(a.rays, w.ray_id, r);
        exact_walk<ANY>(tv, r, st, best);
    }
    if (!ANY) {
        reinterpret_cast<float4*>(a.out)[w.ray_id] = make_float4(best.t, __uint_as_float(best.prim), best.u, best.v);
    } else if (!a.occ_slot) {
        static_cast<uint8_t*>(a.out)[w.ray_id] = best.any ? 1 : 0;
    } else if (best.any) {  // the shadow ray's contribution is cleared here (w kept)
        const uint32_t slot = a.occ_slot[w.ray_id];
        float* c = reinterpret_cast<float*>(a.occ_rec + 4 * (size_t)(slot >> 1) + 2 + (slot & 1u));
        c[0] = 0.f;
        c[1] = 0.f;
        c[2] = 0.f;
    }
}

// A triangle's or quad's hit in record `ri` (which: A or B).
template <bool ANY, bool MULTI>
__device__ __forceinline__ void found(const TraceArgs& a, Walker& w, float slack, uint32_t ri, float t, float u, float v, uint32_t which) {
    // A tie of two triangles of one Fast-BVH leaf (a mesh with doubled faces has one at every hit): the
    // one that comes first there wins. False: not such a tie.
    auto same_leaf_order = [&]() {
        const TreeView& tv = MULTI ? a.trees[a.ray_scene[w.ray_id]] : a.tree;
        if ((w.recs[ri].id_a & PR_FLAG) || (w.recs[w.hit >> 1].id_a & PR_FLAG)) return false;
        if (ri == w.hit >> 1) {  // the same record again: A before B
            if (which < (w.hit & 1u)) {
                w.hit = 2 * ri + which;
                w.bu = u;
                w.bv = v;
            }
            return true;
        }
        const WalkAux &x = tv.waux[ri], &y = tv.waux[w.hit >> 1];
        const uint32_t px = (x.places >> (16u * which)) & 0xffffu, py = (y.places >> (16u * (w.hit & 1u))) & 0xffffu;
        if (x.leaf != y.leaf || px == 0xffffu || py == 0xffffu) return false;
        if (px < py) {
            w.hit = 2 * ri + which;
            w.bu = u;
            w.bv = v;
        }
        return true;
    };
    if (t < w.bt) {
        w.second = w.bt;
        w.bt = t;
        w.bu = u;
        w.bv = v;
        w.hit = 2 * ri + which;
        w.lim = t + (slack + 4e-7f * t);
    } else if (!ANY && !(t == w.bt && w.hit != kNone && same_leaf_order())) {
        w.second = fminf(w.second, t);
    }
}

// The outcome of record `ri`: t, u, v of the nearer of A and B (`which`; A where they are equal), or
// infinity, and the other one's distance; negative: the record is a quad.
template <bool ANY, bool MULTI>
__device__ __forceinline__ void leaf_outcome(const TraceArgs& a, Walker& w, float slack, uint32_t ri, float t, float u, float v,
                                             float other, uint32_t which) {
    if (other < 0.0f) {
        const TreeView& tv = MULTI ? a.trees[a.ray_scene[w.ray_id]] : a.tree;
        RayK q;
        load_ray(a.rays, w.ray_id, q);
        float qt;
        if ((w.recs[ri].id_a & PR_FLAG) && quad_test(q, tv.quads[__float_as_uint(w.recs[ri].a.p0x)], FLT_MAX, qt))
            found<ANY, MULTI>(a, w, slack, ri, qt, 0.f, 0.f, 0u);
    } else if (t < FLT_INF) {
        found<ANY, MULTI>(a, w, slack, ri, t, u, v, which);
        w.second = fminf(w.second, other);
    }
    if (ANY && w.hit != kNone) {
        w.sp = 0;
        w.cur = w.leaf = kNone;
    }
}

// Tests the triangle at `tp`; true: the record is a quad's (it has a NaN where no triangle of a walk tree
// has one: the builder leaves such triangles out).
__device__ __forceinline__ bool record_tri(RayK& r, const char* tp, float& t, float& u, float& v) {
    r.kz = r.ky == 2 ? 0 : r.ky + 1;
    r.kx = r.kz == 2 ? 0 : r.kz + 1;
    const Float3* vp = reinterpret_cast<const Float3*>(tp);
    const Float3 p0 = vp[0], p1 = vp[1], p2 = vp[2];
    const Tri x{p0.x, p0.y, p0.z, p1.x, p1.y, p1.z, p2.x, p2.y, p2.z};
    float tt, uu, vv;
    if (tri_test(r, x, tt, uu, vv)) {
        t = tt;
        u = uu;
        v = vv;
    }
    return __builtin_isnan(p1.x);
}

// The gates that a wave's rays have come to, and the triangles that these let them through to. Both wait until
// there is one for every lane, or until a ray is to be answered: a lane takes a gate or a triangle of any ray
// of the wave, with the ray fetched from its owner.
struct GateShared {
    uint32_t gate[127];  // first record << 6 | owner
    uint2 tri[127];      // record * 2 + (0: A, 1: B), owner
    uint32_t ray[64];    // each lane's gate_ray()
    float slack[64];     // and its search slack (both are wanted seldom, and registers are short)
};
struct Gates {
    GateShared& sh;
    uint32_t n_gate = 0, n_tri = 0;

    __device__ __forceinline__ explicit Gates(GateShared& s) : sh(s) {}
    __device__ __forceinline__ bool full() const { return n_gate >= 64u; }
    __device__ __forceinline__ bool waiting() const { return (n_gate | n_tri) != 0; }

    // Notes the gate from record `first` on for this lane's ray, where `at`. (Called by the whole wave.)
    __device__ __forceinline__ void put(bool at, uint32_t first, uint32_t lane) {
        const uint64_t m = __ballot(at);
        if (m == 0) return;
        if (at) sh.gate[n_gate + rank_in(m)] = first << 6 | lane;
        n_gate += (uint32_t)__popcll(m);
    }

    // Takes the last of the gates, one to a lane, and tests the triangles behind them by 64; `all`: the last
    // few too. GROUP: lanes that hold one ray.
    template <bool ANY, bool MULTI, uint32_t GROUP>
    __device__ __forceinline__ void pass(const TraceArgs& a, Walker& w, bool all) {
        const uint32_t lane = __lane_id();
        const uint32_t n = min(n_gate, 64u);
        n_gate -= n;
        __builtin_amdgcn_wave_barrier();
        uint32_t count = 0, bound = 0, ray = 0, owner = 0, first = 0;
        const GateWords* gp = nullptr;
        if (lane < n) {
            const uint32_t e = sh.gate[n_gate + lane];
            owner = e & 63u;
            first = e >> 6;
            ray = sh.ray[owner];
            count = 1;
        }
        const uint32_t* words = a.tree.wgates;
        if (MULTI) {
            const uint32_t id = of_lane(owner, w.ray_id);
            if (lane < n) words = a.trees[a.ray_scene[id]].wgates;
        }
        gp = reinterpret_cast<const GateWords*>(words + 2 * (size_t)first);
        uint32_t open = 0, at = 0;
        while (true) {
            uint64_t m = __ballot(open != 0);
            if (m == 0 && __ballot(at < count) != 0) {  // the next eight records' words
                if (at < count) {
                    const GateWords g[4] = {gp[0], gp[1], gp[2], gp[3]};
                    if (at == 0) {
                        count = g[0].a >> 24;
                        bound = gate_bound(ray, g[0].b >> 24);
                    }
#pragma unroll
                    for (uint32_t i = 0; i < 4; i++) open |= g[i].open(ray & 0xffffffu, bound) << (4 * i);
                    open &= (1u << (2u * min(count - at, kGateRecs))) - 1u;
                    gp += kGateRecs / 2;
                }
                at += kGateRecs;
                m = __ballot(open != 0);
            }
            const bool done = m == 0 && __ballot(at < count) == 0;
            if (m != 0) {
                if (open != 0)
                    sh.tri[n_tri + rank_in(m)] =
                        make_uint2(2 * (first + at - kGateRecs) + (uint32_t)__ffs((int)open) - 1u, owner);
                open &= open - 1u;
                n_tri += (uint32_t)__popcll(m);
            }
            if (n_tri >= 64u || (done && all && n_tri != 0)) test<ANY, MULTI, GROUP>(a, w);
            if (done) break;
        }
    }

    // Tests the last of the triangles, one to a lane.
    template <bool ANY, bool MULTI, uint32_t GROUP>
    __device__ __forceinline__ void test(const TraceArgs& a, Walker& w) {
        const uint32_t lane = __lane_id();
        const uint32_t n = min(n_tri, 64u);
        n_tri -= n;
        __builtin_amdgcn_wave_barrier();
        const uint2 e = sh.tri[n_tri + min(lane, n - 1u)];
        const uint32_t owner = e.y;
        RayK r;
        r.okx = of_lane(owner, w.r.okx); r.oky = of_lane(owner, w.r.oky); r.okz = of_lane(owner, w.r.okz);
        r.sx = of_lane(owner, w.r.sx); r.sy = of_lane(owner, w.r.sy); r.sz = of_lane(owner, w.r.sz);
        r.tmin = of_lane(owner, w.r.tmin);
        r.tmax = fminf(of_lane(owner, w.r.tmax), of_lane(owner, w.lim));
        r.ky = (int)of_lane(owner, (uint32_t)w.r.ky);
        const PrimRec* recs = MULTI ? of_lane(owner, w.recs) : w.recs;
        float t = FLT_INF, u = 0.f, v = 0.f;
        if (lane < n) record_tri(r, reinterpret_cast<const char*>(recs + (e.x >> 1)) + (e.x & 1u) * sizeof(Tri), t, u, v);
        // almost never: a hit of an edge-on triangle, to its ray
        for (uint64_t m = __ballot(t < FLT_INF); m != 0; m &= m - 1) {
            const uint32_t l = (uint32_t)__ffsll((unsigned long long)m) - 1u;
            const uint32_t to = (uint32_t)__builtin_amdgcn_readlane((int)owner, (int)l);
            const uint32_t x = (uint32_t)__builtin_amdgcn_readlane((int)e.x, (int)l);
            auto bits = [&](float f) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), (int)l)); };
            const float ht = bits(t), hu = bits(u), hv = bits(v);
            if (lane / GROUP == to / GROUP) {
                found<ANY, MULTI>(a, w, sh.slack[lane], x >> 1, ht, hu, hv, x & 1u);
                if (ANY) {
                    w.sp = 0;
                    w.cur = w.leaf = kNone;
                }
            }
        }
    }
};

// One ray to a lane: batches that fill the chip.
template <bool ANY, bool MULTI, int LDS, int SPILL>
__device__ __forceinline__ void walk_lanes(const TraceArgs& a, uint32_t n_rays, uint2* s_st, GateShared& s_gate,
                                           uint32_t* s_next, uint32_t* s_out) {
    constexpr int CAP = LDS + SPILL;
    uint2 sp_st[SPILL];  // deeper entries; also the stack of exact_walk, whose lane has none of its own left
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = __lane_id();
    const uint32_t refill = a.refill ? a.refill : 16u;
    const uint32_t leaf_batch = a.leaf_batch ? a.leaf_batch : 24u;
    // Handing out the rays. One atomic on the launch's counter takes about 8.5 ns of the whole chip's
    // time (measured: 4.19M rays, 16 at a time, spent 2.2 ms there), so every workgroup has a share of
    // its own that its waves take from through LDS. Of a large batch only three quarters are shares,
    // dealt 64 rays at a time so that all workgroups move through the order together (a contiguous
    // share each has them all over the tree at once: 2.05 instead of 1.87 ms for 4.19M sorted bounce
    // rays); the rest goes out through the counter, in chunks that shrink with what is left, so that
    // the workgroups end together. A batch with less than a full wave of rays for each wave spreads
    // over all of them, on the first `seats` lanes of each.
    const uint32_t waves = gridDim.x * (kBlock / 64);
    const uint32_t seats = min((n_rays + waves - 1) / waves, 64u);
    const bool dealt = n_rays >= kDealtPerWave * waves;
    const uint32_t share = dealt ? (n_rays - n_rays / 4u) / (gridDim.x * 64u) * 64u : (n_rays + gridDim.x - 1) / gridDim.x;
    const uint32_t pooled = min(share * gridDim.x, n_rays);  // first ray that the counter hands out
    if (tid == 0) {
        *s_next = 0;                         // rays of the share taken
        *s_out = pooled >= n_rays ? 1u : 0u;  // whether the counter has run out
    }
    __syncthreads();
    bool sharing = true;            // the share may have rays left
    uint32_t own = 0, own_end = 0;  // this wave's chunk of the rest
    bool more = lane < seats, overflow = false;
    Walker w;
    w.nodes = a.tree.wnodes;
    w.recs = a.tree.wrecs;
    w.cur = w.leaf = w.ray_id = w.hit = kNone;
    w.bt = w.lim = w.second = FLT_MAX;
    w.bu = w.bv = 0.f;
    w.sp = 0;
    w.open = false;
    Gates gates(s_gate);

    while (true) {
        const bool idle = w.idle();
        const uint64_t want = __ballot(idle && (more || w.ray_id != kNone));
        const uint64_t busy = __ballot(!idle);
        if (want == 0 && busy == 0) break;
        const bool answer = want != 0 && (busy == 0 || (uint32_t)__popcll(want) >= refill);
        if (answer) {
            while (gates.waiting()) gates.pass<ANY, MULTI, 1>(a, w, gates.n_gate <= 64u);
            if (idle && w.ray_id != kNone) {
                settle<ANY, MULTI>(a, w, sp_st);
                w.ray_id = kNone;
            }
            const uint64_t take = __ballot(idle && more);
            if (take != 0) {
                const uint32_t cnt = (uint32_t)__popcll(take);
                const uint32_t rank = (uint32_t)__popcll(take & ((1ull << lane) - 1ull));
                uint32_t k = 0;
                bool given = false, out = false;  // a lane without a ray waits for the next refill; out: there is none
                if (sharing) {
                    uint32_t v = 0;
                    if (lane == 0) v = atomicAdd(s_next, cnt);
                    v = __builtin_amdgcn_readfirstlane(v);
                    sharing = v + cnt < share;
                    v += rank;
                    k = dealt ? ((((v >> 6) * gridDim.x + blockIdx.x) << 6) | (v & 63u)) : blockIdx.x * share + v;
                    given = v < share && k < pooled;
                } else {
                    if (own == own_end) {
                        uint32_t done = 0;
                        if (lane == 0) done = __hip_atomic_load(s_out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                        out = __builtin_amdgcn_readfirstlane(done) != 0;
                        if (!out) {
                            const uint32_t rest = n_rays - max(own_end, pooled);
                            const uint32_t chunk = max(min(rest / (2u * waves), 256u), 32u);
                            if (lane == 0) own = atomicAdd(a.counter, chunk);
                            own = pooled + __builtin_amdgcn_readfirstlane(own);
                            own_end = min(own + chunk, n_rays);
                            out = own >= n_rays;
                            if (out && lane == 0)
                                __hip_atomic_store(s_out, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                        }
                    }
                    k = own + rank;
                    given = k < own_end;
                    own = min(own + cnt, own_end);
                }
                if (out) more = false;
                if (idle && more && given) start<ANY, MULTI>(a, a.order ? a.order[k] : k, w, s_gate.slack[lane], s_gate.ray[lane]);
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
            const bool walk = w.walking();
            if (__ballot(walk) == 0 || (uint32_t)__popcll(__ballot(w.leaf != kNone)) >= batch) break;
            const bool pop = walk && w.cur == kNone;
            // Stack accesses are LDS ones unless some lane of the wave is past the entries there: a
            // choice per lane would make every access a generic one.
            if (__ballot(pop && w.sp > LDS) == 0) {
                if (pop) {
                    --w.sp;
                    const uint2 e = s_st[w.sp * kBlock + tid];
                    if (__uint_as_float(e.y) <= w.lim) w.cur = e.x;
                }
            } else if (pop) {
                --w.sp;
                uint2 e;
                if (w.sp < LDS) e = s_st[w.sp * kBlock + tid];
                else e = sp_st[min(w.sp - LDS, SPILL - 1)];
                if (__uint_as_float(e.y) <= w.lim) w.cur = e.x;
            }
            bool gated = false;
            uint32_t first = 0;
            if (walk && (int32_t)w.cur >= 0) {
                const NodeSlabs n(w.nodes, w.cur, w.s);
                uint32_t key[4];
                float near[4];
#pragma unroll
                for (uint32_t j = 0; j < 4; j++) key[j] = n.key(j, 8 * j, w.r, w.lim, near[j]);
                // one bound for the four: a choice by slot would cost more than the visits it saves
                const uint32_t ahead = __float_as_uint(fminf(fminf(near[0], near[1]), fminf(near[2], near[3])));
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
                if (__ballot(w.sp + 3 > LDS) == 0) {
#pragma unroll
                    for (int i = 3; i >= 1; i--) {
                        s_st[w.sp * kBlock + tid] = make_uint2(n.ref(key[i]), ahead);
                        w.sp += key[i] != kNone ? 1 : 0;
                    }
                } else {
#pragma unroll
                    for (int i = 3; i >= 1; i--) {
                        if (key[i] == kNone) continue;
                        const uint2 e = make_uint2(n.ref(key[i]), ahead);
                        if (w.sp < LDS) s_st[w.sp * kBlock + tid] = e;
                        else if (w.sp < CAP) sp_st[w.sp - LDS] = e;
                        // not reached: the host sizes the stack for the tree
                        if (w.sp < CAP) w.sp++;
                        else overflow = true;
                    }
                }
                gated = n.gated;
                first = n.first_record();
                w.cur = key[0] != kNone ? n.ref(key[0]) : kNone;
            }
            gates.put(gated, first, lane);
            if (gates.full()) gates.pass<ANY, MULTI, 1>(a, w, false);
            if (w.at_leaf() && w.leaf == kNone) {
                w.leaf = w.cur;
                w.cur = kNone;
            }
        }
        // ---- leaf phase: the waiting leaves' triangles, one to a lane ----
        // Leaf number i of the wave has its A tested by lane 2i and its B by lane 2i + 1, with the ray
        // fetched from the lane that owns it: twenty leaves keep forty lanes busy for one triangle's
        // time, where their owners would take two. At most 32 leaves a round; others wait.
        const uint64_t holders = __ballot(w.leaf != kNone);
        if (holders == 0) continue;
        const uint32_t rank = (uint32_t)__popcll(holders & ((1ull << lane) - 1ull));
        const bool mine = w.leaf != kNone && rank < 32u;
        // lane 2i learns which lane owns leaf i; lane 2i + 1 has it from its neighbour
        int owner = __builtin_amdgcn_ds_permute((int)((mine ? 2u * rank : 63u) << 2), mine ? (int)lane : -1);
        owner = (int)pair_even((uint32_t)owner);
        const bool tester = (lane >> 1) < (uint32_t)__popcll(holders);
        const int from = owner << 2;
        auto fetch = [&](float x) { return __int_as_float(__builtin_amdgcn_ds_bpermute(from, __float_as_int(x))); };
        RayK r;
        r.okx = fetch(w.r.okx); r.oky = fetch(w.r.oky); r.okz = fetch(w.r.okz);
        r.sx = fetch(w.r.sx); r.sy = fetch(w.r.sy); r.sz = fetch(w.r.sz);
        r.tmin = fetch(w.r.tmin);
        r.tmax = fetch(w.r.tmax);
        r.ky = __builtin_amdgcn_ds_bpermute(from, w.r.ky);
        const uint32_t ri = w.leaf & ~REF_LEAF;
        const char* tp = nullptr;
        if (MULTI) {
            const uint64_t at = reinterpret_cast<uint64_t>(w.recs + ri);
            const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)(uint32_t)at);
            const uint32_t up = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)(uint32_t)(at >> 32));
            tp = reinterpret_cast<const char*>(((uint64_t)up << 32) | lo);
        } else {
            const uint32_t at = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)(ri * (uint32_t)sizeof(PrimRec)));
            tp = reinterpret_cast<const char*>(w.recs) + at;
        }
        float t = FLT_INF, u = 0.f, v = 0.f;
        bool quad = false;
        if (tester) quad = record_tri(r, tp + (lane & 1u) * sizeof(Tri), t, u, v);
        const float to = pair_swap(t), uo = pair_swap(u), vo = pair_swap(v);
        const bool take_b = to < t;  // as lane 2i sees it
        float other = take_b ? t : (to == t ? FLT_INF : to);
        if (quad) other = -1.0f;
        const int back = (int)((2u * min(rank, 31u)) << 2);
        auto result = [&](float x) { return __int_as_float(__builtin_amdgcn_ds_bpermute(back, __float_as_int(x))); };
        const float rt = result(take_b ? to : t), ru = result(take_b ? uo : u), rv = result(take_b ? vo : v);
        const float ro = result(other);
        const bool rb = __builtin_amdgcn_ds_bpermute(back, take_b ? 1 : 0) != 0;
        if (mine) {
            w.leaf = kNone;
            if (w.at_leaf()) {
                w.leaf = w.cur;
                w.cur = kNone;
            }
            leaf_outcome<ANY, MULTI>(a, w, s_gate.slack[lane], ri, rt, ru, rv, ro, rb ? 1u : 0u);
        }
    }
    if (overflow) atomicOr(a.error, kFlagStackOverflow);
}

// One ray to four lanes (a child of its node each, a triangle to every other one): batches too small
// to fill the chip, where the time is that of the longest rays' chains of steps. A step has half
// the instructions of walk_lanes', and a wave's 16 rays wait less for one another.
// All four lanes hold the same walker. The stack has kQuadStack entries in LDS, [entry][ray].
// Against walk_lanes: 1,000 rays in the Cornell room 41 -> 29 us, 64 rays through 50K triangles 132 -> 89,
// 65K 165 -> 131, 100K 182 -> 156; at 32 rays a wave (131K) it takes 182 -> 183, the Cornell room
// 78 -> 94, at 49 (200K) 193 -> 239: four rays' worth of lanes for one stops paying once the chip is full.
constexpr int kQuadStack = 64;
template <bool ANY, bool MULTI, int SPILL>
__device__ __forceinline__ void walk_quads(const TraceArgs& a, uint32_t n_rays, uint2* s_st, GateShared& s_gate,
                                           uint32_t* s_next) {
    uint2 exact_st[SPILL];
    const uint32_t lane = __lane_id();
    const uint32_t sub = lane & 3u;
    const uint32_t waves = gridDim.x * (kBlock / 64);
    const uint32_t seats = min((n_rays + waves - 1) / waves, 16u);
    const uint32_t share = (n_rays + gridDim.x - 1) / gridDim.x;
    if (threadIdx.x == 0) *s_next = 0;
    __syncthreads();
    uint2* st = s_st + (threadIdx.x >> 6) * (kQuadStack * 16) + (lane >> 2);
    bool more = (lane >> 2) < seats, overflow = false;
    Walker w;
    w.nodes = a.tree.wnodes;
    w.recs = a.tree.wrecs;
    w.cur = w.leaf = w.ray_id = w.hit = kNone;
    w.bt = w.lim = w.second = FLT_MAX;
    w.bu = w.bv = 0.f;
    w.sp = 0;
    w.open = false;
    Gates gates(s_gate);
    while (true) {
        const bool idle = w.idle();
        const uint64_t want = __ballot(idle && (more || w.ray_id != kNone));
        const uint64_t busy = __ballot(!idle);
        if (want == 0 && busy == 0) break;
        const bool answer = want != 0 && (busy == 0 || (uint32_t)__popcll(want) >= 16u);
        if (answer) {
            while (gates.waiting()) gates.pass<ANY, MULTI, 4>(a, w, gates.n_gate <= 64u);
            if (idle && w.ray_id != kNone) {
                if (sub == 0) settle<ANY, MULTI>(a, w, exact_st);
                w.ray_id = kNone;
            }
            const uint64_t take = __ballot(idle && more && sub == 0);
            if (take != 0) {
                uint32_t v = 0;
                if (lane == 0) v = atomicAdd(s_next, (uint32_t)__popcll(take));
                v = __builtin_amdgcn_readfirstlane(v) + (uint32_t)__popcll(take & ((1ull << (lane & ~3u)) - 1ull));
                const uint32_t k = blockIdx.x * share + v;
                if (idle && more) {
                    if (v < share && k < n_rays) start<ANY, MULTI>(a, a.order ? a.order[k] : k, w, s_gate.slack[lane], s_gate.ray[lane]);
                    else more = false;
                }
            }
            continue;
        }
        const uint32_t batch = ((uint32_t)__popcll(busy) + 3u) / 4u;
        while (true) {
            const bool walk = w.walking();
            if (__ballot(walk) == 0 || (uint32_t)__popcll(__ballot(w.leaf != kNone)) >= batch) break;
            if (walk && w.cur == kNone) {
                --w.sp;
                const uint2 e = st[w.sp * 16];
                if (__uint_as_float(e.y) <= w.lim) w.cur = e.x;
            }
            bool gated = false;
            uint32_t first = 0;
            if (walk && (int32_t)w.cur >= 0) {
                const NodeSlabs n(w.nodes, w.cur, w.s);
                float near;
                const uint32_t key = n.key(sub, 8 * sub, w.r, w.lim, near);
                const float ahead_2 = fminf(near, quad_rot_f<0xB1>(near));
                const float ahead = fminf(ahead_2, quad_rot_f<0x4E>(ahead_2));
                const uint32_t k1 = quad_rot<0x39>(key), k2 = quad_rot<0x4E>(key), k3 = quad_rot<0x93>(key);
                const uint32_t nearest = min(min(key, k1), min(k2, k3));
                // place of this lane's child: hits farther than it lie below
                const int below = (k1 != kNone && k1 > key ? 1 : 0) + (k2 != kNone && k2 > key ? 1 : 0) +
                                  (k3 != kNone && k3 > key ? 1 : 0);
                const int hits = (key != kNone ? 1 : 0) + (k1 != kNone ? 1 : 0) + (k2 != kNone ? 1 : 0) +
                                 (k3 != kNone ? 1 : 0);
                if (key != kNone && key != nearest) {
                    // always: the host takes this form for trees whose stack fits
                    if (w.sp + below < kQuadStack) st[(w.sp + below) * 16] = make_uint2(n.ref(key), __float_as_uint(ahead));
                    else overflow = true;
                }
                w.sp = min(w.sp + max(hits - 1, 0), kQuadStack);
                gated = n.gated && sub == 0;
                first = n.first_record();
                w.cur = nearest != kNone ? n.ref(nearest) : kNone;
            }
            gates.put(gated, first, lane);
            if (gates.full()) gates.pass<ANY, MULTI, 4>(a, w, false);
            if (w.at_leaf() && w.leaf == kNone) {
                w.leaf = w.cur;
                w.cur = kNone;
            }
        }
        if (w.leaf != kNone) {
            const uint32_t ri = w.leaf & ~REF_LEAF;
            w.leaf = kNone;
            if (w.at_leaf()) {
                w.leaf = w.cur;
                w.cur = kNone;
            }
            float t = FLT_INF, u = 0.f, v = 0.f;
            const bool quad = record_tri(w.r, reinterpret_cast<const char*>(w.recs + ri) + (sub & 1u) * sizeof(Tri), t, u, v);
            const float to = pair_swap(t), uo = pair_swap(u), vo = pair_swap(v);
            // (every lane takes part in the exchange: a lane left out would hand its neighbour a zero)
            const float quad_there = pair_swap(quad ? 1.0f : 0.0f);
            const bool quad_any = quad | (quad_there != 0.0f);
            const bool odd = (sub & 1u) != 0;
            const float ta = odd ? to : t, tb = odd ? t : to;
            const bool take_b = tb < ta;
            const bool own = take_b == odd;  // this lane tested the nearer one
            leaf_outcome<ANY, MULTI>(a, w, s_gate.slack[lane], ri, take_b ? tb : ta, own ? u : uo, own ? v : vo,
                                     quad_any ? -1.0f : take_b ? ta : (ta == tb ? FLT_INF : tb), take_b ? 1u : 0u);
        }
    }
    if (overflow) atomicOr(a.error, kFlagStackOverflow);
}

// 4 waves per SIMD (128 VGPRs): 5 spilled in the rarely taken parts and gained nothing.
template <bool ANY, bool MULTI, int LDS, int SPILL>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4))) void k_walk(TraceArgs a) {
    __shared__ uint2 s_st[LDS * kBlock];  // stacks: (reference, entry distance)
    __shared__ GateShared s_gate[kBlock / 64];
    __shared__ uint32_t s_next, s_out;
    static_assert(LDS < 16 || LDS * kBlock >= kQuadStack * 16 * (kBlock / 64), "the quads' stacks fit");
    const uint32_t n_rays = a.n_dev ? *a.n_dev : a.n;
    const uint32_t stack = MULTI ? a.walk_stack : a.tree.walk_stack;
    if (LDS >= 16 && stack <= (uint32_t)kQuadStack && n_rays <= kQuadsPerWave * gridDim.x * (kBlock / 64))
        walk_quads<ANY, MULTI, SPILL>(a, n_rays, s_st, s_gate[threadIdx.x / 64], &s_next);
    else
        walk_lanes<ANY, MULTI, LDS, SPILL>(a, n_rays, s_st, s_gate[threadIdx.x / 64], &s_next, &s_out);
}

__global__ void k_walk_reset(uint32_t* counter) {
    if (threadIdx.x == 0) *counter = 0;
}

template <bool ANY, bool MULTI, int LDS, int SPILL>
hipError_t launch(const TraceArgs& a, hipStream_t stream, int num_cus) {
    auto kern = k_walk<ANY, MULTI, LDS, SPILL>;
    // asked once: the answer is the kernel's and the architecture's
    static std::atomic<int> resident{0};
    int per_cu = resident.load(std::memory_order_relaxed);
    if (per_cu < 1) {
        hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, kBlock, 0);
        if (e != hipSuccess) return e;
        if (per_cu < 1) per_cu = 1;
        resident.store(per_cu, std::memory_order_relaxed);
    }
    if (a.blocks_per_cu && (int)a.blocks_per_cu < per_cu) per_cu = (int)a.blocks_per_cu;
    // as many waves as run at once, down to one ray each
    const uint64_t want = ((uint64_t)a.n + 3) / 4;
    uint64_t grid = (uint64_t)num_cus * (uint64_t)per_cu;
    if (want < grid) grid = want;
    if (grid < 1) grid = 1;
    // a batch that the workgroups' shares cover never asks the counter (saves a launch, about 5 us)
    if (!a.counter_clear && a.n >= kDealtPerWave * (kBlock / 64) * grid)
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
