// Whether a walk of the walk tree reaches every triangle that could decide a query, with the kernel's own
// arithmetic (walk_step.h, traverse.h) on the CPU: those that the Fast-BVH's triangle test accepts in a leaf
// whose box its slab test accepts. The scenes are those where that test accepts rays far from the triangle:
// flat sheets seen edge-on, needles, triangles at the size of the arithmetic's rounding, and far origins.
#include "traverse.h"
#include "walk_step.h"

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <functional>
#include <random>
#include <string>
#include <thread>
#include <vector>

#include "bvh_build.h"

using namespace sortgpu;

namespace {

using Gen = std::mt19937;
float uni(Gen& g, float a, float b) { return std::uniform_real_distribution<float>(a, b)(g); }
struct V {
    float x, y, z;
};
V point(Gen& g, float a, float b) {
    const float x = uni(g, a, b), y = uni(g, a, b);
    return {x, y, uni(g, a, b)};
}
V add(V a, V b, float s = 1.0f) { return {a.x + s * b.x, a.y + s * b.y, a.z + s * b.z}; }

struct Scene {
    std::vector<float> pos;
    void tri(V a, V b, V c) {
        for (V v : {a, b, c}) pos.insert(pos.end(), {v.x, v.y, v.z});
    }
    V vertex(Gen& g) const {
        const size_t i = 3 * (g() % (pos.size() / 3));
        return {pos[i], pos[i + 1], pos[i + 2]};
    }
};

struct Tree {
    BuiltTree t;
    std::vector<uint32_t> first, count;  // per Fast-BVH leaf: its place in `members`
    std::vector<std::pair<uint32_t, int>> members;  // record, 0: A, 1: B
    std::vector<uint32_t> box_of;        // per leaf: a record with its box
};

bool build(const Scene& s, unsigned width, unsigned leaf, unsigned depth, Tree& out) {
    std::vector<uint32_t> idx(s.pos.size() / 3);
    for (uint32_t i = 0; i < idx.size(); i++) idx[i] = i;
    BuildInput in;
    in.pos = s.pos.data();
    in.nverts = (uint32_t)idx.size();
    in.idx = idx.data();
    in.ntris = in.nverts / 3;
    in.quads = nullptr;
    in.nquads = 0;
    in.width = width;
    in.max_leaf = leaf;
    in.max_depth = depth;
    in.threads = 4;
    std::string err;
    if (!build_tree(in, out.t, err) || !out.t.walk.stack) return false;
    const WalkTree& w = out.t.walk;
    std::vector<std::pair<uint32_t, uint32_t>> at;  // leaf, record
    for (uint32_t r = 0; r + kWalkPadRecs < w.recs.size(); r++) at.push_back({w.aux[r].leaf, r});
    std::sort(at.begin(), at.end());
    for (size_t i = 0; i < at.size(); i++) {
        if (!i || at[i].first != at[i - 1].first) {
            out.first.push_back((uint32_t)out.members.size());
            out.count.push_back(0);
            out.box_of.push_back(at[i].second);
        }
        const PrimRec& p = w.recs[at[i].second];
        for (int k = 0; k < ((p.id_b & PR_ID) == PR_NONE ? 1 : 2); k++) {
            out.members.push_back({at[i].second, k});
            out.count.back()++;
        }
    }
    return true;
}

// The walk with its search bound held at `lim`: marks the triangles it tests; false: it needs more stack than the
// tree announces.
bool walk(const WalkTree& w, const RayK& r, const Slabs& s, uint32_t gate, float lim, std::vector<uint32_t>& mark,
          uint32_t round) {
    std::vector<std::pair<uint32_t, float>> st = {{0u, 0.0f}};
    while (!st.empty()) {
        const auto e = st.back();
        st.pop_back();
        if (!(e.second <= lim)) continue;
        if (e.first & REF_LEAF) {
            mark[2 * (e.first & ~REF_LEAF)] = mark[2 * (e.first & ~REF_LEAF) + 1] = round;
            continue;
        }
        const NodeSlabs n(w.nodes.data(), e.first, s);
        float near[4];
        uint32_t key[4];
        for (uint32_t j = 0; j < 4; j++) key[j] = n.key(j, 8 * j, r, lim, near[j]);
        const float ahead = std::fmin(std::fmin(near[0], near[1]), std::fmin(near[2], near[3]));
        for (uint32_t j = 0; j < 4; j++)
            if (key[j] != kNone) st.push_back({n.ref(key[j]), ahead});
        if (n.gated) {
            const uint32_t first = n.first_record() & ~REF_LEAF;
            const uint32_t* g = &w.gates[2 * (size_t)first];
            const uint32_t count = g[0] >> 24, bound = gate_bound(gate, g[1] >> 24);
            for (uint32_t i = 0; i < 2 * count; i++)
                if (gate_open(g[i], gate & 0xffffffu, bound)) mark[2 * (first + i / 2) + i % 2] = round;
        }
        if (st.size() > w.stack) return false;
    }
    return true;
}

std::atomic<long> g_decided{0}, g_rays{0};

// One ray: 0, or what is wrong.
const char* check_ray(const Tree& tree, RayK r, std::vector<uint32_t>& mark, uint32_t& round) {
    const BuiltTree& t = tree.t;
    const WalkTree& w = t.walk;
    Slabs s;
    uint32_t gate;
    float slack;
    if (!slabs_setup(r, t.bbox, w.pad, s, slack, gate)) return nullptr;  // answered by the Fast-BVH walk
    ray_setup(r);
    if (!(root_slab(r, t.bbox) >= 0.0f)) return nullptr;
    g_rays++;
    std::vector<std::pair<float, uint32_t>> found;  // distance, triangle of a record
    for (size_t l = 0; l < tree.first.size(); l++) {
        const WalkAux& x = w.aux[tree.box_of[l]];
        float entry;
        if (x.leaf != 0 && !box_test(r, x.lo[0], x.hi[0], x.lo[1], x.hi[1], x.lo[2], x.hi[2], entry)) continue;
        for (uint32_t m = 0; m < tree.count[l]; m++) {
            const auto mem = tree.members[tree.first[l] + m];
            const PrimRec& p = w.recs[mem.first];
            float d, u, v;
            if (tri_test(r, mem.second ? p.b : p.a, d, u, v)) found.push_back({d, 2 * mem.first + (uint32_t)mem.second});
        }
    }
    if (found.empty()) return nullptr;
    g_decided++;
    std::sort(found.begin(), found.end());
    RayK k = r;  // the kernel takes its shear constants from the true reciprocals
    shear_setup(k, s);
    if (k.sx != r.sx || k.sy != r.sy || k.sz != r.sz) return "shear constants differ";
    // with the bound at a hit's own distance every hit up to it has to be reached
    for (size_t i : {(size_t)0, found.size() / 2, found.size() - 1}) {
        round++;
        if (!walk(w, k, s, gate, found[i].first, mark, round)) return "stack";
        for (size_t j = 0; j <= i; j++)
            if (mark[found[j].second] != round) return "a deciding triangle is not reached";
    }
    return nullptr;
}

bool check(const char* name, const Scene& s, unsigned width, unsigned leaf, unsigned depth, unsigned rays,
           const std::function<void(Gen&, RayK&)>& make) {
    Tree tree;
    if (!build(s, width, leaf, depth, tree)) {
        std::printf("FAIL %s: no walk tree\n", name);
        return false;
    }
    const unsigned threads = 8;
    std::vector<long> wrong(threads, 0);
    std::vector<const char*> what(threads, nullptr);
    std::vector<std::thread> th;
    for (unsigned i = 0; i < threads; i++)
        th.emplace_back([&, i] {
            Gen g(i + 7u * width);
            std::vector<uint32_t> mark(2 * tree.t.walk.recs.size(), 0);
            uint32_t round = 0;
            for (unsigned k = 0; k < rays / threads; k++) {
                RayK r;
                r.tmin = 0.0f;
                r.tmax = FLT_MAX;
                make(g, r);
                if (const char* bad = check_ray(tree, r, mark, round)) {
                    wrong[i]++;
                    what[i] = bad;
                }
            }
        });
    for (auto& x : th) x.join();
    long sum = 0;
    for (unsigned i = 0; i < threads; i++) sum += wrong[i];
    for (unsigned i = 0; i < threads && sum; i++)
        if (what[i]) {
            std::printf("FAIL %s (width %u, leaf %u, depth %u): %ld of %u rays: %s\n", name, width, leaf, depth, sum, rays, what[i]);
            return false;
        }
    return true;
}

void aim(RayK& r, V o, V d, bool unit) {
    if (unit) {
        const float l = std::sqrt(d.x * d.x + d.y * d.y + d.z * d.z);
        if (l > 0) d = {d.x / l, d.y / l, d.z / l};
    }
    r.ox = o.x; r.oy = o.y; r.oz = o.z;
    r.dx = d.x; r.dy = d.y; r.dz = d.z;
}

// A sheet of n x n squares spanned by a and b from c, and a parallel one `gap` along its normal.
Scene sheets(int n, V c, V a, V b, V gap) {
    Scene s;
    for (int k = 0; k < 2; k++)
        for (int i = 0; i < n; i++)
            for (int j = 0; j < n; j++) {
                auto p = [&](int x, int y) { return add(add(add(c, a, (float)x / n), b, (float)y / n), gap, (float)k); };
                s.tri(p(i, j), p(i + 1, j), p(i + 1, j + 1));
                s.tri(p(i, j), p(i + 1, j + 1), p(i, j + 1));
            }
    return s;
}

// A soup of n triangles in the unit cube; `size(i)` gives the spread of triangle i.
Scene soup(unsigned n, const std::function<V(unsigned)>& size) {
    Scene s;
    Gen g(n);
    for (unsigned i = 0; i < n; i++) {
        const V c = point(g, 0, 1), z = size(i);
        auto p = [&] {
            const V v = point(g, -0.5f, 0.5f);
            return add(c, {v.x * z.x, v.y * z.y, v.z * z.z});
        };
        const V a = p(), b = p();
        s.tri(a, b, p());
    }
    return s;
}

}  // namespace

int main(int argc, char** argv) {
    const unsigned scale = argc > 1 ? (unsigned)std::atoi(argv[1]) : 1u;
    for (unsigned width : {8u, 4u}) {
        const V a{0.9f, 0.31f, -0.17f}, b{-0.23f, 0.77f, 0.41f}, up{0.258f, -0.33f, 0.764f};
        struct Form {
            unsigned leaf, depth;
        };
        for (Form f : {Form{16, 28}, Form{3, 28}, Form{16, 3}})
            for (int n : {2, 4, 16, 48}) {
                if (n == 48 && f.depth == 3) continue;  // a few leaves of hundreds: no walk tree
                const Scene s = sheets(n, {0.1f, 0.05f, 0.2f}, a, b, {up.x * 0.25f, up.y * 0.25f, up.z * 0.25f});
                for (float off : {0.0f, 1e-7f, 1e-6f, 3e-6f, 1e-5f, 1e-4f}) {
                    auto in_plane = [&](Gen& g, RayK& r) {  // between two points of the sheet's plane, `off` beside it
                        auto p = [&] { return add(add(add({0.1f, 0.05f, 0.2f}, a, uni(g, -0.2f, 1.2f)), b, uni(g, -0.2f, 1.2f)), up, uni(g, -off, off)); };
                        const V o = g() % 2 ? p() : s.vertex(g);
                        const V e = g() % 2 ? p() : s.vertex(g);
                        aim(r, o, add(e, o, -1.0f), g() % 2);
                        if (g() % 4 == 0) {
                            r.tmin = uni(g, 0, 0.5f);
                            r.tmax = r.tmin + uni(g, 0, 0.5f);
                        }
                    };
                    if (!check("tilted sheets", s, width, f.leaf, f.depth, 4000 * scale, in_plane)) return 1;
                }
            }
        for (float tiny : {1e-3f, 1e-4f, 1e-5f, 3e-6f, 1e-6f, 1e-7f, 1e-8f})
            for (unsigned every : {2u, 20u}) {
                const Scene s = soup(2000, [&](unsigned i) { const float z = i % every ? 0.2f : tiny; return V{z, z, z}; });
                for (float away : {0.3f, 100.0f}) {
                    auto rays = [&](Gen& g, RayK& r) {  // random rays, and rays at a triangle's vertex
                        const V o = point(g, 0.5f - away, 0.5f + away), v = s.vertex(g);
                        aim(r, o, g() % 2 ? add(v, o, -1.0f) : add(point(g, 0, 1), o, -1.0f), g() % 4 != 0);
                    };
                    if (!check("tiny triangles among others", s, width, 16, 28, 8000 * scale, rays)) return 1;
                }
            }
        for (float thin : {1e-2f, 1e-4f, 1e-6f, 1e-8f}) {  // a needle each way, rays along them
            Scene s = soup(1500, [&](unsigned i) { return i % 10 ? V{0.1f, 0.1f, 0.1f} : V{thin, thin, 0.3f}; });
            const size_t n = s.pos.size();
            for (size_t i = 0; i < n; i += 9) {  // turn them
                const float ang = (float)i;
                for (size_t k = i; k < i + 9; k += 3) {
                    const float x = s.pos[k] - 0.5f, z = s.pos[k + 2] - 0.5f;
                    s.pos[k] = 0.5f + x * std::cos(ang) - z * std::sin(ang);
                    s.pos[k + 2] = 0.5f + x * std::sin(ang) + z * std::cos(ang);
                }
            }
            auto rays = [&](Gen& g, RayK& r) {
                const size_t i = 9 * (g() % (s.pos.size() / 9)) / 90 * 90;
                const V p{s.pos[i], s.pos[i + 1], s.pos[i + 2]}, q{s.pos[i + 3], s.pos[i + 4], s.pos[i + 5]};
                const V d = add(q, p, -1.0f);
                aim(r, add(p, d, uni(g, -3, 3)), d, g() % 2);
                if (g() % 8 == 0) aim(r, point(g, -0.5f, 1.5f), point(g, -1, 1), false);
            };
            if (!check("needles", s, width, 16, 28, 16000 * scale, rays)) return 1;
        }
        {
            const Scene s = soup(4000, [](unsigned) { return V{0.08f, 0.08f, 0.08f}; });
            auto rays = [&](Gen& g, RayK& r) {
                V d = point(g, -1, 1);
                const unsigned kind = g() % 8;
                float* c[3] = {&d.x, &d.y, &d.z};
                if (kind == 1) *c[g() % 3] = uni(g, -1e-5f, 1e-5f);
                if (kind == 2) *c[g() % 3] = *c[g() % 3] = g() % 2 ? 0.0f : uni(g, -1e-5f, 1e-5f);
                if (kind == 3) d = {d.x * 1e-3f, d.y * 1e-3f, d.z * 1e-3f};
                if (kind == 4) d = {d.x * 1e-3f, 1e-6f, d.z * 1e-3f};
                if (kind == 5) d = {d.x * 1e6f, d.y * 1e6f, d.z * 1e6f};
                V o = point(g, -0.5f, 1.5f);
                if (kind == 6) o = add(s.vertex(g), d, -1000.0f);
                if (kind == 7) o = add(s.vertex(g), d, -0.3f);
                aim(r, o, d, kind % 3 == 0);
                if (g() % 4 == 0) {
                    r.tmin = uni(g, 0, 0.5f);
                    r.tmax = r.tmin + uni(g, 0, 0.2f);
                }
            };
            if (!check("soup", s, width, 16, 28, 60000 * scale, rays)) return 1;
            if (!check("soup, large leaves", s, width, 150, 28, 8000 * scale, rays)) return 1;
            for (float size : {1e-7f, 1e9f}) {
                Scene m = s;
                for (float& x : m.pos) x *= size;
                auto sized = [&](Gen& g, RayK& r) {
                    rays(g, r);
                    r.ox *= size; r.oy *= size; r.oz *= size;
                };
                if (!check("sized soup", m, width, 16, 28, 16000 * scale, sized)) return 1;
            }
            Scene lost = s;  // products of its coordinates underflow
            for (float& x : lost.pos) x *= 1e-19f;
            Tree none;
            if (build(lost, width, 16, 28, none)) {
                std::printf("FAIL a walk tree where products underflow\n");
                return 1;
            }
            for (float shift : {30.0f, 1000.0f}) {
                Scene m = s;
                for (float& x : m.pos) x += shift;
                auto moved = [&](Gen& g, RayK& r) {
                    rays(g, r);
                    r.ox += shift; r.oy += shift; r.oz += shift;
                };
                if (!check("shifted soup", m, width, 16, 28, 16000 * scale, moved)) return 1;
            }
        }
        for (unsigned n : {1u, 2u, 3u, 5u, 9u}) {
            const Scene s = soup(n, [](unsigned i) { return i % 3 == 1 ? V{1e-7f, 1e-7f, 1e-7f} : V{1, 1, 1}; });
            auto rays = [&](Gen& g, RayK& r) {
                const V v = s.vertex(g), o = add(g() % 2 ? s.vertex(g) : point(g, -1, 2), point(g, -1e-6f, 1e-6f));
                aim(r, o, add(v, o, -1.0f), g() % 2);
            };
            if (!check("few triangles", s, width, 16, 28, 8000 * scale, rays)) return 1;
        }
    }
    if (argc > 1) std::printf("%ld rays, %ld with a hit\n", g_rays.load(), g_decided.load());
    std::printf("ok\n");
    return 0;
}
