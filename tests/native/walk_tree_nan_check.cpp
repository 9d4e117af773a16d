// Walk trees of scenes in which some vertices have a NaN coordinate: the kernel takes a NaN in a record for
// the mark of a quad, so no triangle's record may hold one, and every record with the mark is a quad in range.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>
#include <string>
#include <vector>

#include "bvh_build.h"

using namespace sortgpu;

static int fail(const char* what, unsigned n) {
    std::printf("FAIL %s (%u triangles)\n", what, n);
    return 1;
}

static int check(unsigned ntris, unsigned nquads, unsigned width, unsigned every) {
    std::mt19937 g(ntris + width);
    std::uniform_real_distribution<float> u(0.f, 1.f);
    std::vector<float> pos(9 * (size_t)ntris);
    std::vector<uint32_t> idx(3 * (size_t)ntris);
    for (float& x : pos) x = u(g);
    for (unsigned i = 0; i < idx.size(); i++) idx[i] = i;
    for (unsigned t = 0; t < ntris; t += every)  // one coordinate each, a different one from triangle to triangle
        pos[9 * (size_t)t + (t / every) % 9] = std::numeric_limits<float>::quiet_NaN();
    std::vector<QuadIn> quads(nquads);
    for (QuadIn& x : quads) {
        for (int k = 0; k < 16; k++) x.mat[k] = x.inv[k] = k % 5 == 0 ? 1.f : 0.f;
        x.size_x = x.size_y = 0.1f;
    }
    BuildInput in;
    in.pos = pos.data();
    in.nverts = 3 * ntris;
    in.idx = idx.data();
    in.ntris = ntris;
    in.quads = quads.data();
    in.nquads = nquads;
    in.width = width;
    in.max_leaf = 16;
    in.max_depth = 28;
    in.threads = 2;
    BuiltTree t;
    std::string err;
    if (!build_tree(in, t, err)) return fail(err.c_str(), ntris);
    const WalkTree& w = t.walk;
    unsigned marked = 0;
    for (const PrimRec& r : w.recs) {
        if (r.id_a & PR_FLAG) {
            uint32_t q;
            std::memcpy(&q, &r.a.p0x, sizeof(q));
            if (!std::isnan(r.a.p1x) || q >= nquads) return fail("quad record", ntris);
            marked++;
            continue;
        }
        const float* f = &r.a.p0x;
        for (int v = 0; v < 18; v++)
            if (std::isnan(f[v])) return fail("a triangle's record holds a NaN", ntris);
    }
    if (w.recs.empty()) return fail("no walk tree", ntris);
    return marked == nquads ? 0 : fail("marked records", ntris);
}

int main() {
    for (unsigned width : {4u, 8u})
        for (unsigned n : {9u, 40u, 1000u, 20000u})
            for (unsigned every : {2u, 3u, 50u})
                if (check(n, n % 3, width, every)) return 1;
    std::printf("ok\n");
    return 0;
}
