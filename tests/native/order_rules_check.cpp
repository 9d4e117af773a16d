// Which batches are traced in traversal order by default: both sides of each line, for trees with a walk tree
// and without.
#include <cstdio>

#include "api_internal.h"

hipError_t hipMemPoolDestroy(hipMemPool_t) { return hipSuccess; }  // (of a context; there is none here)

using namespace sortgpu;

int main() {
    struct {
        uint32_t rays;
        size_t bytes;
        bool pays;
    } cases[] = {
        {kReorderMinRays - 1, 0, false},
        {kReorderMinRays, 0, true},
        {0x7fffffffu, 0, true},
        {kReorderMinRays, 1, false},
        {kReorderMinWalkRays - 1, kReorderMinWalkBytes, false},
        {kReorderMinWalkRays, kReorderMinWalkBytes - 1, false},
        {kReorderMinWalkRays, kReorderMinWalkBytes, true},
        {0x7fffffffu, kReorderMinWalkBytes - 1, false},
        {0x7fffffffu, (size_t)1 << 32, true},
        {0, 0, false},
    };
    for (const auto& c : cases)
        if (reorder_pays(c.rays, c.bytes) != c.pays) {
            std::printf("FAIL %u rays, %zu bytes\n", c.rays, c.bytes);
            return 1;
        }
    BuiltTree t;
    if (walk_bytes(t) != 0) return 1;
    t.walk.nodes.resize(3);
    t.walk.recs.resize(2);
    if (walk_bytes(t) != 3 * sizeof(WalkNode) + 2 * sizeof(PrimRec)) return 1;
    std::printf("ok\n");
    return 0;
}
