// Host builder of the walk tree (layout.h WalkNode), derived from the finished Fast-BVH.
//
// The Fast-BVH decides what a query returns: which leaves a ray may take hits from and which of two
// equal hits wins. The walk tree only finds candidates, so its shape is free. It keeps the
// Fast-BVH's upper splits (each node's children arranged as a binary tree by surface area), goes
// on splitting inside its leaves down to two triangles, and folds the binary tree into 4-wide nodes,
// opening the largest child first; the root of a Fast-BVH leaf's part stays a node of its own, with a gate.
#pragma once
#include <stdint.h>
#include <memory>
#include <vector>

#include "layout.h"

namespace sortgpu {

// One primitive as the Fast-BVH build leaves it (in its primitive order).
struct BuildPrim {
    float mn[3];
    float mx[3];
    float c[3];  // centroid
    uint32_t id;
};

// A Fast-BVH node: primitives [off, off + cnt); children are src[first .. first + nchild), after
// their parent; a leaf has none.
struct SrcNode {
    uint32_t off, cnt, first, nchild;
};

// Vectors whose resize() leaves new elements unset: the builder's threads fill them, and touching
// 70 MB for a million triangles on one thread first would cost as much as the rest of the build.
template <class T> struct Unset : std::allocator<T> {
    template <class U> struct rebind { using other = Unset<U>; };
    template <class U> void construct(U* p) noexcept { ::new (static_cast<void*>(p)) U; }
    template <class U, class... A> void construct(U* p, A&&... a) { ::new (static_cast<void*>(p)) U(std::forward<A>(a)...); }
};
template <class T> using RawVec = std::vector<T, Unset<T>>;

struct WalkTree {
    RawVec<WalkNode> nodes;
    RawVec<PrimRec> recs;
    RawVec<WalkAux> aux;
    RawVec<uint32_t> gates;  // two words a record, and kGatePad more
    uint32_t stack = 0;  // most stack entries a traversal holds (0: no walk tree)
    float pad = 0.0f;    // padding of its boxes, as a part of the largest coordinate in play
};

struct BuildInput;

// Deepest walk-tree traversal stack the kernels hold (walk.hip).
constexpr uint32_t kWalkMaxStack = 8 + 256;

// Bounds that walk.hip's header derives, in units of 2^-24 of the largest coordinate in play: the padding of a
// ray's slabs where no quad asks for more, and what it has to cover besides a quad's own error. The reach of a
// triangle's gate over its height: of the scene's extent and its leaf box's diagonal, or of its longest edge.
constexpr float kUnit = 1.0f / (1 << 24);
constexpr float kPadUnits = 32.0f, kPadOther = 17.0f;
constexpr double kGateReach = 52.0 * kUnit, kGateLeaf = 18.0 * kUnit, kGateShape = 40.0 / kWalkWiden * kUnit;

// Leaves `out` empty when the tree cannot have a walk tree: boxes not finite, past 1e12 or below 1e-8 (the
// kernel's error bounds need products that neither overflow nor underflow), far smaller than their distance from the origin
// (its padding would swallow them), a quad whose two matrices are not each other's inverse, records past 4 GiB,
// or a deeper stack than kWalkMaxStack, or no host memory for it.
void build_walk_tree(const BuildInput& in, const std::vector<BuildPrim>& prims, const std::vector<SrcNode>& src,
                     const float bbox[6], unsigned threads, WalkTree& out);

}  // namespace sortgpu
