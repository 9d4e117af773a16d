// Builds walk trees of seeded scenes with the library's host builder and checks what the kernel
// relies on: every primitive in exactly one record, every reference in range, each record's
// triangles inside the boxes on the way to it and inside its Fast-BVH leaf's box, and no traversal
// needing more stack than announced.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <string>
#include <vector>

#include "bvh_build.h"

using namespace sortgpu;

static int fail(const char* what, unsigned n) {
    std::printf("FAIL %s (%u triangles)\n", what, n);
    return 1;
}

static int check(unsigned ntris, unsigned nquads, unsigned width, unsigned leaf, unsigned depth, int kind) {
    std::mt19937 g(ntris * 31 + kind);
    std::uniform_real_distribution<float> u(0.f, 1.f);
    std::vector<float> pos;
    std::vector<uint32_t> idx;
    for (unsigned t = 0; t < ntris; t++) {
        const float c[3] = {kind == 1 ? 0.5f : u(g), kind == 2 ? 0.25f : u(g), u(g) * (kind == 3 ? 1e-3f : 1.f)};
        for (int v = 0; v < 3; v++)
            for (int k = 0; k < 3; k++) {
                const float s = kind == 1 ? (v == 0 ? -0.1f : 0.05f) : (kind == 2 && k == 1 ? 0.f : (u(g) - 0.5f) * 0.02f);
                pos.push_back(c[k] + s);
            }
        for (unsigned v = 0; v < 3; v++) idx.push_back(3 * t + v);
    }
    std::vector<QuadIn> quads(nquads);
    for (unsigned q = 0; q < nquads; q++) {
        QuadIn& x = quads[q];
        for (int k = 0; k < 16; k++) x.mat[k] = x.inv[k] = k % 5 == 0 ? 1.f : 0.f;
        x.mat[3] = u(g);
        x.mat[11] = u(g);
        x.inv[3] = -x.mat[3];
        x.inv[11] = -x.mat[11];
        x.size_x = x.size_y = 0.1f;
    }
    BuildInput in;
    in.pos = pos.data();
    in.nverts = (uint32_t)pos.size() / 3;
    in.idx = idx.data();
    in.ntris = ntris;
    in.quads = quads.data();
    in.nquads = nquads;
    in.width = width;
    in.max_leaf = leaf;
    in.max_depth = depth;
    in.threads = 4;
    BuiltTree t;
    std::string err;
    if (!build_tree(in, t, err)) return fail(err.c_str(), ntris);
    const WalkTree& w = t.walk;
    if (!w.stack || w.recs.size() != w.aux.size()) return fail("no walk tree", ntris);
    std::vector<int> seen(ntris + nquads, 0);
    struct At {
        uint32_t node;
        unsigned held;
        double lo[3], hi[3];
    };
    std::vector<At> st = {{0, 0, {-1e30, -1e30, -1e30}, {1e30, 1e30, 1e30}}};
    size_t nodes = 0;
    while (!st.empty()) {
        const At a = st.back();
        st.pop_back();
        nodes++;
        if (a.node >= w.nodes.size()) return fail("node out of range", ntris);
        const WalkNode& n = w.nodes[a.node];
        const unsigned ni = n.counts & 15, nc = n.counts >> 4;
        if (ni > nc || nc < 1 || nc > 4) return fail("counts", ntris);
        if (a.held + nc > w.stack) return fail("stack", ntris);
        const uint8_t *lo[3] = {n.lo_x, n.lo_y, n.lo_z}, *hi[3] = {n.hi_x, n.hi_y, n.hi_z};
        for (unsigned j = 0; j < nc; j++) {
            At c{n.child_base + j, a.held + nc - 1, {}, {}};
            for (int k = 0; k < 3; k++) {
                const double step = std::ldexp(1.0, n.exp[k] - 127);
                c.lo[k] = n.base[k] + lo[k][j] * step;
                c.hi[k] = n.base[k] + hi[k][j] * step;
            }
            if (j < ni) {
                st.push_back(c);
                continue;
            }
            const uint32_t r = n.rec_base + j - ni;
            if (r + kWalkPadRecs >= w.recs.size()) return fail("record out of range", ntris);
            const PrimRec& p = w.recs[r];
            const WalkAux& x = w.aux[r];
            if (!(p.id_b & PR_FLAG)) return fail("record not last", ntris);
            if (p.id_a & PR_FLAG) {
                seen[p.id_a & PR_ID]++;
                continue;
            }
            for (int q = 0; q < 2; q++) {
                const uint32_t id = (q ? p.id_b : p.id_a) & PR_ID;
                if (id == PR_NONE) continue;
                if (id >= ntris) return fail("triangle id", ntris);
                seen[id]++;
                const float* f = q ? &p.b.p0x : &p.a.p0x;
                for (int v = 0; v < 9; v++) {
                    const int k = v % 3;
                    if (f[v] != pos[9 * (size_t)id + v]) return fail("vertex", ntris);
                    if (f[v] < c.lo[k] || f[v] > c.hi[k]) return fail("outside its node's box", ntris);
                    if (f[v] < x.lo[k] || f[v] > x.hi[k]) return fail("outside its leaf's box", ntris);
                }
            }
        }
    }
    if (nodes != w.nodes.size()) return fail("unreached nodes", ntris);
    for (int s : seen)
        if (s != 1) return fail("primitive not in exactly one record", ntris);
    return 0;
}

int main() {
    for (unsigned width : {4u, 8u})
        for (int kind = 0; kind < 4; kind++)
            for (unsigned n : {1u, 2u, 3u, 5u, 16u, 17u, 33u, 700u, 40000u}) {
                if (check(n, n % 3, width, 16, 28, kind)) return 1;
                if (n < 1000 && (check(n, 2, width, 1, 28, kind) || check(n, 0, width, 16, 2, kind))) return 1;
            }
    std::printf("ok\n");
    return 0;
}
