// Arithmetic of a step through the walk tree (walk.hip, whose header says why its candidates are complete):
// a ray's padded slabs, the boxes of a node's children, the gate of a Fast-BVH leaf, and the Fast-BVH's own
// test of one box.
#pragma once
#include "traverse.h"

#pragma clang fp contract(off)

namespace sortgpu {

constexpr uint32_t kNone = 0xffffffffu;

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

// What a ray shows to the gates: its direction in 127ths in three bytes, and in the fourth how many times the
// reaches, which are given for the scene's extent `ext`, are doubled for a vertex `away` from the origin.
__device__ __forceinline__ uint32_t gate_ray(const RayK& r, float away, float ext) {
    const float unit = 127.0f / sqrtf(r.dx * r.dx + r.dy * r.dy + r.dz * r.dz);
    const int qx = (int)rintf(r.dx * unit), qy = (int)rintf(r.dy * unit), qz = (int)rintf(r.dz * unit);
    uint32_t twice = 0;  // (an origin lies at most 4,096 sizes of the scene out)
    for (float f = ext; f < away && twice < 15u; f += f) twice++;
    return ((uint32_t)qx & 0xffu) | ((uint32_t)qy & 0xffu) << 8 | ((uint32_t)qz & 0xffu) << 16 | twice << 24;
}
// Bound on the product of a ray's and a normal's 127ths, for a reach of `s` 1,024ths: 127 * 127 / 1,024 each,
// and what both lost to rounding, half a 127th of each component times the other vector's (127 sqrt(3) + 1).
__device__ __forceinline__ uint32_t gate_bound(uint32_t ray, uint32_t s) { return 224u + ((16u * s) << (ray >> 24)); }
// Whether a gate word lets the ray through: its direction lies within the bound of the triangle's plane.
__device__ __forceinline__ bool gate_open(uint32_t word, uint32_t dir, uint32_t bound) {
    return (uint32_t)__builtin_amdgcn_sdot4((int)word, (int)dir, (int)bound, false) <= 2u * bound;
}

// Whether the error bounds of the walk hold for this ray; fills `s`, the search slack and `gate`. `kpad`: the
// tree's padding as a part of the largest coordinate in play.
__device__ __forceinline__ bool slabs_setup(const RayK& r, const float* bb, float kpad, Slabs& s, float& slack,
                                            uint32_t& gate) {
    const float mo = fmaxf(fmaxf(fabsf(r.ox), fabsf(r.oy)), fabsf(r.oz));
    const float md = fmaxf(fmaxf(fabsf(r.dx), fabsf(r.dy)), fabsf(r.dz));
    const float o[3] = {r.ox, r.oy, r.oz};
    float mb = 0.0f, ext = 0.0f, away = 0.0f;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        mb = fmaxf(mb, fmaxf(fabsf(bb[k]), fabsf(bb[3 + k])));
        ext = fmaxf(ext, bb[3 + k] - bb[k]);
        away = fmaxf(away, fmaxf(o[k] - bb[k], bb[3 + k] - o[k]));
    }
    const float far = mo + mb;
    const float pad = kpad * far;
    s.rx = recip(r.dx);
    s.ry = recip(r.dy);
    s.rz = recip(r.dz);
    // The Fast-BVH steps through its boxes along a direction of no component below 1e-5: by the end of the
    // scene, far / md along the ray, it has left the ray by up to 1e-5 of that on such an axis.
    const float stray = 1.1e-5f * (far / md);
    const bool cx = fabsf(r.dx) < 0.00001f, cy = fabsf(r.dy) < 0.00001f, cz = fabsf(r.dz) < 0.00001f;
    const float ox = -r.ox * s.rx, oy = -r.oy * s.ry, oz = -r.oz * s.rz;
    const float px = (cx ? pad + stray : pad) * fabsf(s.rx), py = (cy ? pad + stray : pad) * fabsf(s.ry),
                pz = (cz ? pad + stray : pad) * fabsf(s.rz);
    s.ax = ox - px;
    s.ay = oy - py;
    s.az = oz - pz;
    s.bx = ox + px;
    s.by = oy + py;
    s.bz = oz + pz;
    slack = 2.0f * pad * fminf(fminf(fabsf(s.rx), fabsf(s.ry)), fabsf(s.rz));
    gate = gate_ray(r, away, ext);
    // comparisons with a NaN are false; fmaxf drops one, so every component is tested
    return __builtin_isfinite(r.ox) & __builtin_isfinite(r.oy) & __builtin_isfinite(r.oz) &
           __builtin_isfinite(r.dx) & __builtin_isfinite(r.dy) & __builtin_isfinite(r.dz) & (r.tmin >= 0.0f) &
           !__builtin_isnan(r.tmax) & (mo <= 1e12f) & (mo <= 4096.0f * ext) & (md <= 1e12f) &
           (md >= ((cx | cy | cz) ? 1e-3f : 1e-5f));
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

// A node record with the ray's near and far planes picked out, and where its children lie.
struct NodeSlabs {
    float gx, gy, gz, nx, ny, nz, fx, fy, fz;
    uint32_t wnx, wfx, wny, wfy, wnz, wfz;
    uint32_t ni, child_at, leaf_at;
    bool gated;

    __device__ __forceinline__ NodeSlabs(const WalkNode* nodes, uint32_t i, const Slabs& s) {
        const uint4* np = reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(nodes) + (((i << 1) + i) << 4));
        const uint4 q0 = np[0], q1 = np[1], q2 = np[2];
        const uint32_t meta = q0.w;
        gated = (q0.x & 1u) != 0;
        ni = (meta >> 24) & 15u;
        gx = __uint_as_float((meta & 0xffu) << 23) * s.rx;
        gy = __uint_as_float(((meta >> 8) & 0xffu) << 23) * s.ry;
        gz = __uint_as_float(((meta >> 16) & 0xffu) << 23) * s.rz;
        const float bx = __uint_as_float(q0.x) * s.rx, by = __uint_as_float(q0.y) * s.ry, bz = __uint_as_float(q0.z) * s.rz;
        nx = bx + s.ax;
        ny = by + s.ay;
        nz = bz + s.az;
        fx = bx + s.bx;
        fy = by + s.by;
        fz = bz + s.bz;
        const bool px = s.rx >= 0.0f, py = s.ry >= 0.0f, pz = s.rz >= 0.0f;
        wnx = px ? q1.z : q1.w;
        wfx = px ? q1.w : q1.z;
        wny = py ? q2.x : q2.y;
        wfy = py ? q2.y : q2.x;
        wnz = pz ? q2.z : q2.w;
        wfz = pz ? q2.w : q2.z;
        child_at = q1.x;
        leaf_at = (q1.y | REF_LEAF) - ni;
    }
    // Sort key of slot j: kNone where the ray misses its box in its window or what it holds lies past `lim`,
    // else the entry distance (not negative, so that its bits order as it does) with the slot in the last two
    // bits. `near`: no hit in the box is nearer. `shift`: 8 j.
    __device__ __forceinline__ uint32_t key(uint32_t j, uint32_t shift, const RayK& r, float lim, float& near) const {
        auto q = [&](uint32_t x) { return (float)((x >> shift) & 0xffu); };
        const float x = __builtin_fmaf(q(wnx), gx, nx), y = __builtin_fmaf(q(wny), gy, ny), z = __builtin_fmaf(q(wnz), gz, nz);
        const float t0 = fmaxf(fmaxf(x, y), fmaxf(z, r.tmin));
        const float t1 = fminf(fminf(__builtin_fmaf(q(wfx), gx, fx), __builtin_fmaf(q(wfy), gy, fy)),
                               fminf(__builtin_fmaf(q(wfz), gz, fz), r.tmax));
        near = sel3(x, y, z, r.ky);
        return (t0 <= t1) & (near <= lim) ? ((__float_as_uint(t0) & ~3u) | j) : kNone;
    }
    __device__ __forceinline__ uint32_t ref(uint32_t key) const {
        const uint32_t j = key & 3u;
        return (j < ni ? child_at : leaf_at) + j;
    }
    // Reference of the first record below a gated node.
    __device__ __forceinline__ uint32_t first_record() const { return leaf_at + ni; }
};

}  // namespace sortgpu
