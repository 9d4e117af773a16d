// Walk-tree builder. See walk_tree.h.
#include "walk_tree.h"

#include <algorithm>
#include <atomic>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <limits>
#include <memory>
#include <new>
#include <thread>

#include "bvh_build.h"

namespace sortgpu {
namespace {

struct Bin {  // binary node; leaf: l = ~first (place in ord), r = primitive count
    float mn[3], mx[3];
    int32_t l, r;
    bool leaf() const { return l < 0; }
    float area() const {
        const float x = mx[0] - mn[0], y = mx[1] - mn[1], z = mx[2] - mn[2];
        return x * y + y * z + z * x;
    }
};

struct Item {  // something to arrange in a binary tree
    float mn[3], mx[3], c[3];
    uint32_t ref;
    uint32_t weight;  // leaf records below it
};

float box_area(const float* mn, const float* mx) {
    const float x = mx[0] - mn[0], y = mx[1] - mn[1], z = mx[2] - mn[2];
    return x * y + y * z + z * x;
}
void empty_box(float* mn, float* mx) {
    for (int k = 0; k < 3; k++) {
        mn[k] = FLT_MAX;
        mx[k] = -FLT_MAX;
    }
}
void grow(float* mn, float* mx, const float* bmn, const float* bmx) {
    for (int k = 0; k < 3; k++) {
        mn[k] = std::min(mn[k], bmn[k]);
        mx[k] = std::max(mx[k], bmx[k]);
    }
}

// Runs f(i) for i in [0, n) on up to `threads` threads, `grain` at a time.
template <class F>
void parallel_for(uint32_t n, uint32_t grain, unsigned threads, F f) {
    const unsigned want = (unsigned)std::min<uint64_t>(threads, ((uint64_t)n + grain - 1) / grain);
    if (want <= 1) {
        for (uint32_t i = 0; i < n; i++) f(i);
        return;
    }
    std::atomic<uint32_t> next{0};
    std::atomic<bool> short_of_memory{false};  // an exception may not leave a thread
    auto work = [&] {
        try {
            while (!short_of_memory) {
                const uint32_t a = next.fetch_add(grain);
                if (a >= n) return;
                const uint32_t b = std::min(n, a + grain);
                for (uint32_t i = a; i < b; i++) f(i);
            }
        } catch (const std::bad_alloc&) {
            short_of_memory = true;
        }
    };
    std::vector<std::thread> th;
    th.reserve(want);
    for (unsigned w = 1; w < want; w++) {
        try {
            th.emplace_back(work);
        } catch (const std::exception&) {
            break;  // no more threads to be had: those there are do the work
        }
    }
    work();
    for (auto& t : th) t.join();
    if (short_of_memory) throw std::bad_alloc();
}

uint32_t float_bits(float f) {
    uint32_t u;
    std::memcpy(&u, &f, sizeof(u));
    return u;
}

struct Builder {
    const BuildInput& in;
    const std::vector<BuildPrim>& P;
    const std::vector<SrcNode>& S;
    std::unique_ptr<Bin[]> bins;       // left uninitialised: every node is written before it is read
    RawVec<uint32_t> ord;            // primitive places, grouped as the walk records take them
    RawVec<uint32_t> place_leaf;     // Fast-BVH leaf (SrcNode index) of each primitive place
    std::vector<uint32_t> root;      // binary root of each SrcNode
    RawVec<float> sbox;              // 6 per SrcNode leaf: its box, as the Fast-BVH has it
    RawVec<float> wbox;              // 6 per SrcNode: the box of what lies below it in this tree
    const float* bbox;               // the scene's box, and its largest extent
    float extent;

    Builder(const BuildInput& i, const std::vector<BuildPrim>& p, const std::vector<SrcNode>& s, const float* bb, float ext)
        : in(i), P(p), S(s), bbox(bb), extent(ext) {}

    // Arranges it[0..n) as a binary tree: bin nodes from bins[at], the root first. `unit`: the split
    // falls on whole groups of so many items, and a group is a leaf of the primitives it holds
    // (unit > 0, items are primitives placed at ord[first..]) or the item's own subtree (unit = 0).
    uint32_t arrange(Item* it, uint32_t n, uint32_t first, uint32_t unit, uint32_t& at) {
        const uint32_t id = at++;
        float mn[3], mx[3];
        empty_box(mn, mx);
        for (uint32_t i = 0; i < n; i++) grow(mn, mx, it[i].mn, it[i].mx);
        Bin& b = bins[id];
        std::memcpy(b.mn, mn, sizeof(mn));
        std::memcpy(b.mx, mx, sizeof(mx));
        if (unit && n <= unit) {
            for (uint32_t i = 0; i < n; i++) ord[first + i] = it[i].ref;
            b.l = ~(int32_t)first;
            b.r = (int32_t)n;
            return id;
        }
        const uint32_t step = unit ? unit : 1u;
        uint32_t cut = (n / 2 + step - 1) / step * step;
        if (n <= 32) {
            // surface-area sweep on each axis; ties take the more even split, so that equal boxes
            // (all costs alike) make a balanced tree and not a chain
            float best = FLT_MAX, suffix[33];
            uint32_t best_skew = 0;
            uint8_t perm[32], best_perm[32];
            bool found = false;
            for (int ax = 0; ax < 3; ax++) {
                for (uint32_t i = 0; i < n; i++) {  // insertion sort by centroid
                    uint32_t j = i;
                    const float c = it[i].c[ax];
                    while (j > 0 && it[perm[j - 1]].c[ax] > c) {
                        perm[j] = perm[j - 1];
                        j--;
                    }
                    perm[j] = (uint8_t)i;
                }
                empty_box(mn, mx);
                uint32_t wr[33];
                wr[n] = 0;
                for (uint32_t i = n - 1; i >= 1; i--) {
                    grow(mn, mx, it[perm[i]].mn, it[perm[i]].mx);
                    suffix[i] = box_area(mn, mx);
                    wr[i] = wr[i + 1] + it[perm[i]].weight;
                }
                empty_box(mn, mx);
                uint32_t wl = 0;
                for (uint32_t i = 1; i < n; i++) {
                    grow(mn, mx, it[perm[i - 1]].mn, it[perm[i - 1]].mx);
                    wl += it[perm[i - 1]].weight;
                    if (i % step) continue;
                    const float kl = unit ? (float)((i + unit - 1) / unit) : (float)wl;
                    const float kr = unit ? (float)((n - i + unit - 1) / unit) : (float)wr[i];
                    const float cost = box_area(mn, mx) * kl + suffix[i] * kr;
                    const uint32_t skew = i > n - i ? 2 * i - n : n - 2 * i;
                    if (cost < best || (cost == best && skew < best_skew)) {
                        best = cost;
                        best_skew = skew;
                        cut = i;
                        std::memcpy(best_perm, perm, n);
                        found = true;
                    }
                }
            }
            if (found) {
                Item tmp[32];
                for (uint32_t i = 0; i < n; i++) tmp[i] = it[best_perm[i]];
                std::copy(tmp, tmp + n, it);
            }
        } else {
            // a leaf the depth limit or equal centroids left large: median of the widest axis
            float cm[3], cx[3];
            empty_box(cm, cx);
            for (uint32_t i = 0; i < n; i++) grow(cm, cx, it[i].c, it[i].c);
            int ax = 0;
            for (int k = 1; k < 3; k++)
                if (cx[k] - cm[k] > cx[ax] - cm[ax]) ax = k;
            std::nth_element(it, it + cut, it + n, [ax](const Item& a, const Item& c) { return a.c[ax] < c.c[ax]; });
        }
        uint32_t l, r;
        if (!unit && cut == 1) l = it[0].ref;
        else l = arrange(it, cut, first, unit, at);
        if (!unit && n - cut == 1) r = it[cut].ref;
        else r = arrange(it + cut, n - cut, first + cut, unit, at);
        bins[id].l = (int32_t)l;
        bins[id].r = (int32_t)r;
        return id;
    }

    // Binary tree over one Fast-BVH leaf: triangles two to a leaf, then the quads one to a leaf. A triangle
    // stands with its box widened by kWalkWiden of its longest edge (walk.hip), a quad with its Fast-BVH
    // leaf's box: its own corners come from another matrix (light to world) than its test (world to light).
    void leaf_tree(uint32_t s, uint32_t at, std::vector<Item>& it) {
        const SrcNode& n = S[s];
        it.clear();
        uint32_t tris = 0;
        for (int pass = 0; pass < 2; pass++)
            for (uint32_t i = n.off; i < n.off + n.cnt; i++) {
                if ((P[i].id >= in.ntris) != (pass == 1)) continue;
                Item x;
                std::memcpy(x.mn, pass ? &sbox[6 * (size_t)s] : P[i].mn, sizeof(x.mn));
                std::memcpy(x.mx, pass ? &sbox[6 * (size_t)s + 3] : P[i].mx, sizeof(x.mx));
                if (!pass) {  // (the box's diagonal is no shorter than the longest edge)
                    const float e[3] = {x.mx[0] - x.mn[0], x.mx[1] - x.mn[1], x.mx[2] - x.mn[2]};
                    const float by = kWalkWiden * 1.001f * std::sqrt(e[0] * e[0] + e[1] * e[1] + e[2] * e[2]);
                    for (int k = 0; k < 3; k++) {
                        x.mn[k] -= by;
                        x.mx[k] += by;
                    }
                }
                std::memcpy(x.c, P[i].c, sizeof(x.c));
                x.ref = i;
                x.weight = 1;
                it.push_back(x);
                tris += pass == 0 ? 1u : 0u;
            }
        const uint32_t nq = n.cnt - tris;
        if (tris && nq) {  // a node over both parts
            const uint32_t id = at++;
            const uint32_t l = arrange(it.data(), tris, n.off, 2, at);
            const uint32_t r = arrange(it.data() + tris, nq, n.off + tris, 1, at);
            for (int k = 0; k < 3; k++) {
                bins[id].mn[k] = std::min(bins[l].mn[k], bins[r].mn[k]);
                bins[id].mx[k] = std::max(bins[l].mx[k], bins[r].mx[k]);
            }
            bins[id].l = (int32_t)l;
            bins[id].r = (int32_t)r;
        } else {
            arrange(it.data(), n.cnt, n.off, tris ? 2u : 1u, at);
        }
    }

    void inner_tree(uint32_t s, uint32_t at) {
        const SrcNode& n = S[s];
        Item it[8];
        for (uint32_t j = 0; j < n.nchild; j++) {
            const uint32_t c = n.first + j;
            std::memcpy(it[j].mn, &wbox[6 * (size_t)c], 12);
            std::memcpy(it[j].mx, &wbox[6 * (size_t)c + 3], 12);
            for (int k = 0; k < 3; k++) it[j].c[k] = (it[j].mn[k] + it[j].mx[k]) * 0.5f;
            it[j].ref = root[c];
            it[j].weight = (S[c].cnt + 1) / 2;
        }
        arrange(it, n.nchild, 0, 0, at);
    }

    // Whether binary node `b` lies in a Fast-BVH leaf (its root or below), and whether it is the root of one
    // that takes more than one record.
    bool in_leaf(uint32_t b) const { return b < 2 * (uint32_t)P.size(); }
    bool gated(uint32_t b) const {
        return in_leaf(b) && !bins[b].leaf() && 2 * S[place_leaf[b / 2]].off == b;
    }

    // The children of the wide node over binary node `b`. A gated node below it stays whole.
    uint32_t fold(uint32_t b, uint32_t out[4]) const {
        uint32_t n = 1;
        out[0] = b;
        while (n < 4) {
            int best = -1;
            float ba = -1.0f;
            for (uint32_t i = 0; i < n; i++) {
                const Bin& x = bins[out[i]];
                if (x.leaf() || (out[i] != b && gated(out[i]))) continue;
                const float a = x.area();
                if (a > ba) {
                    ba = a;
                    best = (int)i;
                }
            }
            if (best < 0) break;
            const Bin& x = bins[out[best]];
            out[best] = (uint32_t)x.l;
            out[n++] = (uint32_t)x.r;
        }
        uint32_t ni = 0, nl = 0, leaves[4];  // inner children first
        for (uint32_t i = 0; i < n; i++) {
            if (bins[out[i]].leaf()) leaves[nl++] = out[i];
            else out[ni++] = out[i];
        }
        for (uint32_t i = 0; i < nl; i++) out[ni + i] = leaves[i];
        return n;
    }

    void put_tri(Tri& t, uint32_t id) const {
        const uint32_t* v = in.idx + 3 * (size_t)id;
        const float* a = in.pos + 3 * (size_t)v[0];
        const float* b = in.pos + 3 * (size_t)v[1];
        const float* c = in.pos + 3 * (size_t)v[2];
        // A triangle with a NaN coordinate passes no test; its record holds three equal corners, which pass
        // none either. (Its box bounds the other coordinates, so it reaches this tree; an infinite one does not.)
        for (int k = 0; k < 3; k++)
            if (!std::isfinite(a[k]) || !std::isfinite(b[k]) || !std::isfinite(c[k])) return;
        t.p0x = a[0]; t.p0y = a[1]; t.p0z = a[2];
        t.p1x = b[0]; t.p1y = b[1]; t.p1z = b[2];
        t.p2x = c[0]; t.p2y = c[1]; t.p2z = c[2];
    }

    // The gate word of triangle `id` (layout.h): its normal in 127ths, and how near to its plane's direction a
    // ray has to run to be let through, in 1,024ths; a triangle so narrow that this says little lets every ray
    // through (a normal of zeros).
    uint32_t gate_word(uint32_t id, uint32_t leaf) const {
        const float* b = &sbox[6 * (size_t)leaf];
        double across = 0.0;  // the leaf box's diagonal, squared
        for (int k = 0; k < 3; k++) across += ((double)b[3 + k] - b[k]) * ((double)b[3 + k] - b[k]);
        const uint32_t* v = in.idx + 3 * (size_t)id;
        double e[3][3], len[3];  // the edges, and their lengths squared
        for (int i = 0; i < 3; i++) {
            len[i] = 0.0;
            for (int k = 0; k < 3; k++) {
                e[i][k] = (double)in.pos[3 * (size_t)v[(i + 1) % 3] + k] - (double)in.pos[3 * (size_t)v[i] + k];
                len[i] += e[i][k] * e[i][k];
            }
        }
        if (len[0] == 0.0 || len[1] == 0.0 || len[2] == 0.0) return kGateShut;  // two equal corners: never hit
        double n[3];
        for (int k = 0; k < 3; k++) n[k] = e[0][(k + 1) % 3] * e[1][(k + 2) % 3] - e[0][(k + 2) % 3] * e[1][(k + 1) % 3];
        const double area = std::sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);  // twice the triangle's
        const double longest = std::sqrt(std::max(len[0], std::max(len[1], len[2])));
        const double height = area / longest;
        const double s = std::max(kGateReach * extent + kGateLeaf * std::sqrt(across), kGateShape * longest) / height;
        if (!(s <= 1.0 / 16.0)) return 0;
        uint32_t word = (uint32_t)std::ceil(s * 1024.0) << 24;
        for (int k = 0; k < 3; k++) word |= ((uint32_t)(int)std::lrint(127.0 * n[k] / area) & 0xffu) << (8 * k);
        return word;
    }

    // Fills record `r`, its `x` and its two gate words from the leaf `b`.
    void record(const Bin& b, PrimRec& r, WalkAux& x, uint32_t* gate) const {
        std::memset(&r, 0, sizeof(r));
        uint32_t place[2] = {ord[~b.l], b.r > 1 ? ord[~b.l + 1] : 0u};
        if (b.r > 1 && place[1] < place[0]) std::swap(place[0], place[1]);  // A before B in build order
        const uint32_t leaf = place_leaf[place[0]];
        const uint32_t id = P[place[0]].id;
        r.id_b = PR_NONE | PR_FLAG;
        if (id >= in.ntris) {
            const uint32_t q = id - in.ntris;
            std::memcpy(&r.a.p0x, &q, sizeof(q));
            r.a.p1x = std::numeric_limits<float>::quiet_NaN();  // never hit as a triangle
            r.id_a = id | PR_FLAG;
            gate[0] = gate[1] = kGateShut;
        } else {
            put_tri(r.a, id);
            r.id_a = id;
            gate[0] = gate[1] = gate_word(id, leaf);
            if (b.r > 1) {
                gate[1] = gate_word(P[place[1]].id, leaf);
                put_tri(r.b, P[place[1]].id);
                r.id_b = P[place[1]].id | PR_FLAG;
            }
        }
        std::memcpy(x.lo, &sbox[6 * (size_t)leaf], 12);
        std::memcpy(x.hi, &sbox[6 * (size_t)leaf + 3], 12);
        if (leaf == 0) {  // the root is a leaf: no node bounds it but the scene box
            for (int k = 0; k < 3; k++) {
                x.lo[k] = -FLT_MAX;
                x.hi[k] = FLT_MAX;
            }
        }
        x.leaf = leaf;
        const uint32_t pa = std::min(place[0] - S[leaf].off, 0xffffu);
        const uint32_t pb = b.r > 1 ? std::min(place[1] - S[leaf].off, 0xffffu) : 0xffffu;
        x.places = pa | (pb << 16);
    }

    struct Part {
        RawVec<WalkNode> nodes;
        RawVec<PrimRec> recs;
        RawVec<WalkAux> aux;
        RawVec<uint32_t> gates;
        uint32_t stack = 0;
    };
    struct Todo {
        uint32_t bin, slot, held;  // held: stack entries below this node on the way to it
    };

    uint32_t records_below(uint32_t b) const {
        return bins[b].leaf() ? 1u : records_below((uint32_t)bins[b].l) + records_below((uint32_t)bins[b].r);
    }

    // Fills the wide node of `t` in `p`; its inner children are appended to p.nodes and to `more`.
    void wide(const Todo& t, Part& p, std::vector<Todo>& more) const {
        uint32_t c[4];
        const uint32_t n = fold(t.bin, c);
        WalkNode w;
        std::memset(&w, 0, sizeof(w));
        const Bin& b = bins[t.bin];
        uint32_t ni = 0;
        while (ni < n && !bins[c[ni]].leaf()) ni++;
        w.counts = (uint8_t)(ni | (n << 4));
        w.child_base = (uint32_t)p.nodes.size();
        w.rec_base = (uint32_t)p.recs.size();
        uint8_t* lo[3] = {w.lo_x, w.lo_y, w.lo_z};
        uint8_t* hi[3] = {w.hi_x, w.hi_y, w.hi_z};
        const bool gate = gated(t.bin);
        for (int k = 0; k < 3; k++) {
            w.base[k] = b.mn[k];
            // the last bit of base[0] says whether the node has a gate
            while (k == 0 && (float_bits(w.base[0]) & 1u) != (gate ? 1u : 0u)) w.base[0] = std::nextafter(w.base[0], -FLT_MAX);
            // smallest power-of-two step with which 255 of them reach the far plane
            const double ext = (double)b.mx[k] - (double)w.base[k];
            int e = 1;
            if (ext > 0.0) {
                (void)std::frexp(ext / 255.0, &e);  // ext / 255 = m * 2^e, m in [0.5, 1)
                e = std::max(1, std::min(254, e + 127));
                if (e > 1 && std::ceil(std::ldexp(ext, 127 - (e - 1))) <= 255.0) e--;
            }
            w.exp[k] = (uint8_t)e;
            for (uint32_t j = 0; j < 4; j++) {
                if (j >= n) {  // unused slot
                    lo[k][j] = hi[k][j] = 255;
                    continue;
                }
                const Bin& x = bins[c[j]];
                // exact in double: a difference of floats scaled by a power of two
                lo[k][j] = (uint8_t)std::floor(std::ldexp((double)x.mn[k] - (double)w.base[k], 127 - e));
                hi[k][j] = (uint8_t)std::ceil(std::ldexp((double)x.mx[k] - (double)w.base[k], 127 - e));
            }
        }
        const uint32_t held = t.held + n;
        // a gate counts its records in a byte
        p.stack = std::max(p.stack, gate && records_below(t.bin) > 255u ? kWalkMaxStack + 1 : held);
        for (uint32_t j = 0; j < n; j++) {
            if (j < ni) {
                more.push_back({c[j], (uint32_t)p.nodes.size(), held - 1});
                p.nodes.emplace_back();
            } else {
                p.recs.emplace_back();
                p.aux.emplace_back();
                p.gates.resize(p.gates.size() + 2);
                record(bins[c[j]], p.recs.back(), p.aux.back(), &p.gates[p.gates.size() - 2]);
            }
        }
        p.nodes[t.slot] = w;
    }

    // Fills every wide node from `t` down, depth first: the records of a gated node follow one another.
    void subtree(const Todo& t, Part& p) const {
        std::vector<Todo> st = {t};
        while (!st.empty()) {
            const Todo x = st.back();
            st.pop_back();
            const size_t first = p.recs.size();
            if (gated(x.bin)) {
                std::vector<Todo> in_leaf;
                wide(x, p, in_leaf);
                while (!in_leaf.empty()) {
                    const Todo y = in_leaf.back();
                    in_leaf.pop_back();
                    wide(y, p, in_leaf);
                }
                // the first two words carry what the whole gate needs: its records and its widest reach
                uint32_t s = 0;
                for (size_t i = 2 * first; i < p.gates.size(); i++) s = std::max(s, p.gates[i] >> 24);
                uint32_t* g = &p.gates[2 * first];
                g[0] = (g[0] & 0xffffffu) | (uint32_t)(p.recs.size() - first) << 24;
                g[1] = (g[1] & 0xffffffu) | s << 24;
            } else {
                wide(x, p, st);
            }
        }
    }

    void run(unsigned threads, WalkTree& out) {
        const uint32_t n = (uint32_t)P.size(), ns = (uint32_t)S.size();
        sbox.resize(6 * (size_t)ns);
        wbox.resize(6 * (size_t)ns);
        root.resize(ns);
        ord.resize(n);
        place_leaf.resize(n);
        // binary nodes: a leaf of c primitives takes fewer than 2 c, from 2 * off; an inner node of
        // at most 8 children takes at most 7 (and 1 where it has a single child), after them
        std::vector<uint32_t> leaves, inner;
        for (uint32_t s = 0; s < ns; s++) (S[s].nchild ? inner : leaves).push_back(s);
        bins.reset(new Bin[2 * (size_t)n + 8 * inner.size()]);
        for (uint32_t s : leaves) root[s] = 2 * S[s].off;
        for (uint32_t i = 0; i < inner.size(); i++) root[inner[i]] = 2 * n + 8 * i;
        parallel_for((uint32_t)leaves.size(), 64, threads, [&](uint32_t i) {
            const SrcNode& l = S[leaves[i]];
            float* b = &sbox[6 * (size_t)leaves[i]];
            empty_box(b, b + 3);
            for (uint32_t k = l.off; k < l.off + l.cnt; k++) {
                grow(b, b + 3, P[k].mn, P[k].mx);
                place_leaf[k] = leaves[i];
            }
            static thread_local std::vector<Item> it;
            leaf_tree(leaves[i], root[leaves[i]], it);
            const Bin& r = bins[root[leaves[i]]];
            float* w = &wbox[6 * (size_t)leaves[i]];
            std::memcpy(w, r.mn, 12);
            std::memcpy(w + 3, r.mx, 12);
        });
        for (uint32_t i = (uint32_t)inner.size(); i-- > 0;) {  // children follow their parents
            const SrcNode& s = S[inner[i]];
            float* b = &wbox[6 * (size_t)inner[i]];
            empty_box(b, b + 3);
            for (uint32_t j = 0; j < s.nchild; j++) grow(b, b + 3, &wbox[6 * (size_t)(s.first + j)], &wbox[6 * (size_t)(s.first + j) + 3]);
        }
        parallel_for((uint32_t)inner.size(), 256, threads, [&](uint32_t i) { inner_tree(inner[i], root[inner[i]]); });

        // a tree of one record: nothing bounds it but the scene's box
        if (S[0].nchild == 0 && bins[root[0]].leaf()) {
            std::memcpy(bins[root[0]].mn, bbox, 12);
            std::memcpy(bins[root[0]].mx, bbox + 3, 12);
        }

        // fold: the upper nodes one after another, then one part per subtree
        Part top;
        top.nodes.emplace_back();
        std::vector<Todo> queue = {{root[0], 0, 0}};
        size_t head = 0;
        const size_t parts_wanted = n < 16384 ? SIZE_MAX : 512;
        while (head < queue.size() && queue.size() - head < parts_wanted) {
            const Todo t = queue[head++];
            if (gated(t.bin)) subtree(t, top);
            else wide(t, top, queue);
        }
        const uint32_t np = (uint32_t)(queue.size() - head);
        std::vector<Part> parts(np);
        parallel_for(np, 1, threads, [&](uint32_t i) {
            parts[i].nodes.reserve(n / np);
            parts[i].recs.reserve(n / np);
            parts[i].aux.reserve(n / np);
            parts[i].gates.reserve(2 * (n / np));
            parts[i].nodes.emplace_back();
            subtree({queue[head + i].bin, 0, queue[head + i].held}, parts[i]);
        });
        // a part's node 0 takes the slot its parent kept; the others follow the nodes before them
        std::vector<uint64_t> nbase(np + 1), rbase(np + 1);
        nbase[0] = top.nodes.size();
        rbase[0] = top.recs.size();
        uint32_t stack = top.stack;
        for (uint32_t i = 0; i < np; i++) {
            nbase[i + 1] = nbase[i] + parts[i].nodes.size() - 1;
            rbase[i + 1] = rbase[i] + parts[i].recs.size();
            stack = std::max(stack, parts[i].stack);
        }
        // the kernel's offsets into both arrays are 32-bit bytes, and a record index shares its
        // word with the leaf bit
        if (stack > kWalkMaxStack || nbase[np] * sizeof(WalkNode) > UINT32_MAX || (rbase[np] + kWalkPadRecs) * sizeof(PrimRec) > UINT32_MAX)
            return;
        out.nodes.resize(nbase[np]);
        out.recs.resize(rbase[np] + kWalkPadRecs);
        out.aux.resize(rbase[np] + kWalkPadRecs);
        out.gates.resize(2 * rbase[np] + kGatePad);
        PrimRec none;  // a triangle of three equal corners is never hit
        std::memset(&none, 0, sizeof(none));
        none.id_b = PR_NONE | PR_FLAG;
        std::fill(out.recs.begin() + rbase[np], out.recs.end(), none);
        std::fill(out.aux.begin() + rbase[np], out.aux.end(), WalkAux{});
        std::copy(top.nodes.begin(), top.nodes.end(), out.nodes.begin());
        std::copy(top.recs.begin(), top.recs.end(), out.recs.begin());
        std::copy(top.aux.begin(), top.aux.end(), out.aux.begin());
        std::fill(out.gates.end() - kGatePad, out.gates.end(), 0u);
        std::copy(top.gates.begin(), top.gates.end(), out.gates.begin());
        parallel_for(np, 1, threads, [&](uint32_t i) {
            const Part& p = parts[i];
            for (size_t k = 0; k < p.nodes.size(); k++) {
                WalkNode w = p.nodes[k];
                w.child_base += (uint32_t)nbase[i] - 1;
                w.rec_base += (uint32_t)rbase[i];
                out.nodes[k ? nbase[i] + k - 1 : queue[head + i].slot] = w;
            }
            std::copy(p.recs.begin(), p.recs.end(), out.recs.begin() + rbase[i]);
            std::copy(p.aux.begin(), p.aux.end(), out.aux.begin() + rbase[i]);
            std::copy(p.gates.begin(), p.gates.end(), out.gates.begin() + 2 * rbase[i]);
        });
        out.stack = stack;
    }
};

}  // namespace

void build_walk_tree(const BuildInput& in, const std::vector<BuildPrim>& prims, const std::vector<SrcNode>& src,
                     const float bbox[6], unsigned threads, WalkTree& out) {
    out = WalkTree();
    if (prims.empty() || src.empty()) return;
    float far = 0.0f, ext = 0.0f;
    for (int k = 0; k < 3; k++) {
        if (!std::isfinite(bbox[k]) || !std::isfinite(bbox[3 + k])) return;
        far = std::max(far, std::max(std::fabs(bbox[k]), std::fabs(bbox[3 + k])));
        ext = std::max(ext, bbox[3 + k] - bbox[k]);
    }
    for (const BuildPrim& p : prims)  // an axis on which every coordinate is NaN has a box that bounds nothing
        for (int k = 0; k < 3; k++)
            if (!(p.mn[k] <= p.mx[k]) || !(p.mn[k] >= bbox[k] && p.mx[k] <= bbox[3 + k])) return;
    if (far > 1e12f || far < 1e-8f || far > 4096.0f * ext) return;
    if (prims.size() / 2 * sizeof(PrimRec) > UINT32_MAX) return;
    // A quad is tested in its own space: what the walk sees of its rounding and of the disagreement of its
    // matrices, as a part of the largest coordinate.
    double off = 0.0;
    for (uint32_t q = 0; q < in.nquads; q++) {
        const float *m = in.quads[q].mat, *v = in.quads[q].inv;
        for (int k = 0; k < 4; k++)
            if (m[12 + k] != (k == 3 ? 1.0f : 0.0f) || v[12 + k] != (k == 3 ? 1.0f : 0.0f)) return;
        for (int k = 0; k < 3; k++) {
            double wrong = 0.0, shift = m[4 * k + 3], round = 0.0;
            for (int j = 0; j < 3; j++) {
                double e = k == j ? -1.0 : 0.0, row = 0.0;
                for (int i = 0; i < 3; i++) {
                    e += (double)m[4 * k + i] * v[4 * i + j];
                    row += 16.0 * std::fabs((double)v[4 * j + i]);
                }
                wrong += std::fabs(e);
                shift += (double)m[4 * k + j] * v[4 * j + 3];
                round += std::fabs((double)m[4 * k + j]) * (row + 4.0 * std::fabs((double)v[4 * j + 3]) / far);
            }
            const double axis = wrong + std::fabs(shift) / far + round * kUnit;
            if (!(axis <= 1.0 / 4096)) return;
            off = std::max(off, axis);
        }
    }
    try {
        Builder b(in, prims, src, bbox, ext);
        b.run(prims.size() < 16384 ? 1u : threads, out);
    } catch (const std::bad_alloc&) {  // queries go without
        out.stack = 0;
    }
    if (!out.stack) out = WalkTree();
    out.pad = std::max(kPadUnits * kUnit, (float)off * 1.0001f + kPadOther * kUnit);
}

}  // namespace sortgpu
