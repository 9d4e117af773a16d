// What the device headers of the traversal take from the HIP runtime, for a build by the host compiler: the
// checks run the kernels' own arithmetic on the CPU.
#pragma once
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <cstring>

#define __device__
#define __forceinline__ inline

struct float4 {
    float x, y, z, w;
};
struct uint4 {
    uint32_t x, y, z, w;
};
inline uint32_t __float_as_uint(float f) {
    uint32_t u;
    std::memcpy(&u, &f, sizeof(u));
    return u;
}
inline float __uint_as_float(uint32_t u) {
    float f;
    std::memcpy(&f, &u, sizeof(f));
    return f;
}
inline int __popc(uint32_t x) { return __builtin_popcount(x); }
inline int __builtin_amdgcn_sdot4(int a, int b, int c, bool) {
    for (int k = 0; k < 32; k += 8) c += (int)(int8_t)(a >> k) * (int)(int8_t)(b >> k);
    return c;
}
