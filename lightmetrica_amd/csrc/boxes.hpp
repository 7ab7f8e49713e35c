// Ray / box arithmetic of the BVH traversal and the packing of its nodes, for the kernels and for the
// host-side check (tests/native/packed_check.cpp).
#pragma once

#include <cmath>

#include "bvh_build.h"

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define LMGPU_HD __host__ __device__ __forceinline__
#define LMGPU_UNROLL _Pragma("unroll")
#else
#define LMGPU_HD inline
#define LMGPU_UNROLL
#endif

namespace lmgpu {

// u = 2^-24, gamma(n) = n u / (1 - n u).  A box whose planes are at hand is met with 1 + 2 gamma(4).
constexpr float kBoxRobustExact = 1.0f + 2.0f * 2.4e-7f;
// What a hit's leaf may lie behind the hit by without being taken for another order (hit_order), 64u
// of the distance: of rays that meet a triangle in an axis-parallel plane the FP32 distance lies before
// the plane by more than 4u for 1 in 300, by more than 64u for 1 in 12,000.
constexpr float kOrderScale = 1.0f - 64.0f * 5.9604645e-8f;
// A box is left out for a hit that comes before it if it lies behind that hit by more than this: 1 +
// 72u, so that no hit that comes first in the order is (1 / kOrderScale is 1 + 64.0002u, and the
// products round).
constexpr float kOrderPrune = 1.0f + 72.0f * 5.9604645e-8f;
// Packed boxes: 1 + 80u.  Against the built box's distances each of the two is off by 3 more roundings,
// the node's offset fma(origin, inv, offset), the step's product and the plane's own FMA, beyond what
// the planes' margin covers: whatever the built box accepts the packed one accepts, and what
// kOrderPrune keeps it keeps.
constexpr float kBoxRobust = 1.0f + 80.0f * 5.9604645e-8f;
// t moved up by k's excess over 1 of itself: t * k, also behind the origin, where a product would
// move it down.
LMGPU_HD float widened(float t, float k) { return fmaf(fabsf(t), k - 1.0f, t); }

// Per-ray constants of the slab test.  A plane at coordinate x is reached at
// t = fma(x, inv, offset).  The offset fma(-o, inv, -+e) is -o * inv -+ e rounded once, so
// fma(x, inv, offset) equals (x - o) * inv -+ e up to one rounding of the result and an
// absolute error of about u |o * inv| (the offset's rounding); e = 4u |p| = 2^-22 |p|, with
// p = o * inv, exceeds it, so moving the plane that is entered first (lo when inv >= 0)
// earlier by e and the plane that is left last later by e leaves the entry and exit distances
// with relative errors only, which kBoxRobust covers.  Coordinates are assumed below 1e8 in
// magnitude so that o * inv stays finite for the clamped reciprocal (<= 1e30).
// Per axis the ray knows which plane it enters first (lo when inv >= 0), so a select per axis
// and node takes the near and far planes of all four children and no min / max orders them.
struct Slab {
    float ix, iy, iz;
    float nx, fx, ny, fy, nz, fz;  // offsets of the near and far planes per axis
};

LMGPU_HD void slab_axis(float o, float inv, float& near_off, float& far_off) {
    const float e = fabsf(o * inv) * 2.384185791015625e-7f;  // 2^-22 |p|
    const float lo = fmaf(-o, inv, inv >= 0.f ? -e : e);       // lo plane, moved away from the box's inside
    const float hi = fmaf(-o, inv, inv >= 0.f ? e : -e);
    near_off = inv >= 0.f ? lo : hi;
    far_off = inv >= 0.f ? hi : lo;
}

// From the origin and the reciprocals of the direction, within 1 ulp (safe_rcp).
LMGPU_HD Slab make_slab(float ox, float oy, float oz, float ix, float iy, float iz) {
    Slab s;
    s.ix = ix;
    s.iy = iy;
    s.iz = iz;
    slab_axis(ox, ix, s.nx, s.fx);
    slab_axis(oy, iy, s.ny, s.fy);
    slab_axis(oz, iz, s.nz, s.fz);
    return s;
}

// Where a ray enters and leaves a box within [tmin, tmax]; it meets the box if
// tn <= widened(tf, kBoxRobustExact).  Monotone in every plane: a box that contains this one is met too.
LMGPU_HD void box_span(const Slab& s, float lx, float hx, float ly, float hy, float lz, float hz, float tmin, float tmax,
                       float& tn, float& tf) {
    tn = fmaxf(fmaxf(fmaf(s.ix >= 0.f ? lx : hx, s.ix, s.nx), fmaf(s.iy >= 0.f ? ly : hy, s.iy, s.ny)),
               fmaxf(fmaf(s.iz >= 0.f ? lz : hz, s.iz, s.nz), tmin));
    tf = fminf(fminf(fmaf(s.ix >= 0.f ? hx : lx, s.ix, s.fx), fmaf(s.iy >= 0.f ? hy : ly, s.iy, s.fy)),
               fminf(fmaf(s.iz >= 0.f ? hz : lz, s.iz, s.fz), tmax));
}

// One axis of a packed node along a ray: the planes are origin + q * step, reached at
// fma(q, step * inv, fma(origin, inv, offset)).
struct PackedAxis {
    float a, near_off, far_off;
    uint32_t near, far;  // the children's planes, a byte each
};
LMGPU_HD PackedAxis packed_axis(float origin, float step, uint32_t lo, uint32_t hi, float inv, float near_off,
                                float far_off) {
    return PackedAxis{step * inv, fmaf(origin, inv, near_off), fmaf(origin, inv, far_off), inv >= 0.f ? lo : hi,
                      inv >= 0.f ? hi : lo};
}
// Child i's span within [tmin, tmax]; the ray may meet the child if
// tn <= widened(tf, kBoxRobust).
LMGPU_HD void packed_span(const PackedAxis& x, const PackedAxis& y, const PackedAxis& z, int i, float tmin, float tmax,
                          float& tn, float& tf) {
    auto at = [i](uint32_t q, float a, float off) { return fmaf(float((q >> (8 * i)) & 0xffu), a, off); };
    tn = fmaxf(fmaxf(at(x.near, x.a, x.near_off), at(y.near, y.a, y.near_off)), fmaxf(at(z.near, z.a, z.near_off), tmin));
    tf = fminf(fminf(at(x.far, x.a, x.far_off), at(y.far, y.a, y.far_off)), fminf(at(z.far, z.a, z.far_off), tmax));
}

// A node of the built tree in the form the kernels read.  Along each axis the children's planes
// are 8-bit steps of ext / 254.9 from the lowest plane, lo planes rounded down and hi planes up
// and moved out by at least kPlaneMargin steps more, which exceeds what evaluating
// origin + q * scale along a ray can lose against the extent (3 roundings of 255 steps).
// Step 0 is the lowest plane itself.  An empty slot's box is inverted (255, 0) and its child
// word a one-record leaf: where rounding or NaN lets a ray in, the record's own test decides.
constexpr double kPlaneMargin = 1.0 / 512;
LMGPU_HD NodeQ pack_node(const Node4& n) {
    NodeQ q;
    const float* lo[3] = {n.lo_x, n.lo_y, n.lo_z};
    const float* hi[3] = {n.hi_x, n.hi_y, n.hi_z};
    LMGPU_UNROLL
    for (int a = 0; a < 3; a++) {
        float l = INFINITY, h = -INFINITY;
        LMGPU_UNROLL
        for (int i = 0; i < 4; i++) {
            if (n.child[i] == kEmptyChild) continue;
            l = fminf(l, lo[a][i]);
            h = fmaxf(h, hi[a][i]);
        }
        const double ext = double(h) - double(l);
        const float step = ext > 0.0 ? fmaxf(float(ext * (1.0 / 254.9)), 1.17549435e-38f) : 0.f;
        uint32_t ql = 0u, qh = 0u;
        LMGPU_UNROLL
        for (int i = 0; i < 4; i++) {
            uint32_t b0 = 255u, b1 = 0u;
            if (n.child[i] != kEmptyChild) {
                b0 = 0u;
                if (step > 0.f) {
                    const double s0 = (double(lo[a][i]) - double(l)) / double(step) - kPlaneMargin;
                    const double s1 = (double(hi[a][i]) - double(l)) / double(step) + kPlaneMargin;
                    b0 = uint32_t(fmax(floor(s0), 0.0));
                    b1 = uint32_t(fmin(ceil(s1), 255.0));
                }
            }
            ql |= b0 << (8 * i);
            qh |= b1 << (8 * i);
        }
        q.origin[a] = l;
        q.step[a] = step;
        q.planes[a][0] = ql;
        q.planes[a][1] = qh;
    }
    LMGPU_UNROLL
    for (int i = 0; i < 4; i++) q.child[i] = n.child[i] == kEmptyChild ? kLeafBit : n.child[i];
    return q;
}

}  // namespace lmgpu
