// Closest-hit and any-hit traversal of the 4-wide BVH (bvh_build.h) on gfx950.
//
// Replaces QBVHScene::IntersectTriangles (src/liblightmetrica/scene.qbvh.cpp:837-960):
//   * one ray per lane, 64-lane wavefronts; every step of a wave is either one node visit or
//     one leaf step (two triangles), whichever more of its lanes wait for, so that a step
//     runs with 26 to 43 lanes instead of the 14 of separate node and leaf loops;
//   * a node is 64 bytes (NodeQ: 8-bit planes of four children), fetched as four 16-byte
//     loads; a leaf of two or more triangles starts on a 128-byte line (LeafTri, two a line)
//     and its triangles are fetched two at a time: what bounds a large batch is the lines
//     fetched beyond L1 and L2;
//   * children hit by the ray are sorted by entry distance; the nearest is descended
//     into and the others are pushed, farthest first (closest and any hit);
//   * the traversal stack lives in LDS, [level][lane] so the 64 lanes of a wave hit
//     distinct banks, and spills to per-lane private memory beyond StackLevels::kLds levels;
//     closest-hit entries carry their box's entry distance, and pops skip the boxes that
//     lie beyond the nearest hit found since they were pushed;
//   * boxes are tested with the reciprocal-direction slab test in fused form, one FMA
//     per plane (step * (scale * inv) + (origin * inv + offset)); the per-ray offsets -o * inv
//     are widened by the rounding that form adds, packed planes are moved out by more than
//     theirs, and the exit distance is moved up by 2 gamma(4) of itself (packed boxes: 80u), so
//     rounding never culls a box the ray touches (Ize, "Robust BVH Ray Traversal", JCGT 2013, with
//     the absolute error of the fused form and the 1-ulp hardware reciprocal accounted for);
//   * triangles use the watertight test of Woop, Benthin and Wald (JCGT 2013), with
//     the FP64 fallback for edge functions that evaluate to exactly zero.
// Measured on 16M incoherent rays against 1M triangles (closest hit with the FP64 pass):
// 3.98 ms with separate node and leaf loops over 128-byte nodes and unaligned leaves, 3.11 ms
// so; 4M any-hit segments 1.75 -> 1.29 ms; the extension rays of a 96k-triangle room (8.4M
// paths, 8 segments, twice) 15.2 -> 10.3 ms.  With 128-byte nodes in the same loop: 3.35, 1.65 and
// 13.8 ms.  Of that 0.05, 0 and 0.1 ms go into checking each ray's last hit against the built boxes
// (sound_hit); checked as each hit is met it took 0.13, 0.04 and 0.5 ms.
// Acceptance follows the reference's QBVH: t strictly inside (tmin, tmax), the first
// triangle found wins an exact tie (scene.qbvh.cpp:124-133).
#pragma once

#include "boxes.hpp"
#include "bvh_build.h"
#include "device_math.hpp"

namespace lmgpu {

constexpr int kTraceBlock = 256;
constexpr int kStackTotal = 96;  // supports 4-wide trees of depth <= 32

struct RayIn {
    float ox, oy, oz, dx, dy, dz, tmin, tmax;
};

// The descents of the BVH report a hit by its record alone (`rec`), which hit_at turns into the rest.
struct HitOut {
    float t;
    uint32_t rec;  // leaf-order triangle record of the winner
    uint32_t prim; // scene-order triangle index, 0xffffffff = miss
    float b0, b1;  // FP32 barycentric weights of v1 and v2 (closest hit)
    float det;     // what b0 and b1 still have to be divided by (hit_weights)
};

struct TraceCounters {
    uint32_t nodes;
    uint32_t tris;
};

// Per-ray constants of the watertight test.
struct Shear {
    int kx, ky, kz;
    float Sx, Sy, Sz;
    float ox, oy, oz;  // origin permuted into (kx, ky, kz)
};

__device__ __forceinline__ float pick3(float a, float b, float c, int k) { return k == 0 ? a : (k == 1 ? b : c); }

__device__ __forceinline__ Shear make_shear(const RayIn& r) {
    Shear s;
    const float ax = fabsf(r.dx), ay = fabsf(r.dy), az = fabsf(r.dz);
    s.kz = (ax > ay) ? (ax > az ? 0 : 2) : (ay > az ? 1 : 2);
    s.kx = s.kz == 2 ? 0 : s.kz + 1;
    s.ky = s.kx == 2 ? 0 : s.kx + 1;
    const float dkz = pick3(r.dx, r.dy, r.dz, s.kz);
    if (dkz < 0.f) {  // keep the winding of the projected triangle
        int t = s.kx;
        s.kx = s.ky;
        s.ky = t;
    }
    // The shear only has to be the same for every triangle of the ray, so the hardware
    // reciprocal (1 ulp) serves.
    const float inv = __builtin_amdgcn_rcpf(dkz);
    s.Sx = pick3(r.dx, r.dy, r.dz, s.kx) * inv;
    s.Sy = pick3(r.dx, r.dy, r.dz, s.ky) * inv;
    s.Sz = inv;
    s.ox = pick3(r.ox, r.oy, r.oz, s.kx);
    s.oy = pick3(r.ox, r.oy, r.oz, s.ky);
    s.oz = pick3(r.ox, r.oy, r.oz, s.kz);
    return s;
}

__device__ __forceinline__ bool watertight_tail(float ax, float ay, float bx, float by, float cx, float cy, float za,
                                                float zb, float zc, float tmin, float tmax, float& t, float& U,
                                                float& V, float& W, float& det);

// The shear of the BVH traversal, whose vertices differ from lane to lane: the axes are
// permuted cyclically (kz the largest direction component) and two selects per component
// apply the permutation.  make_shear also swaps kx and ky when the ray points down kz; the
// swap negates U, V, W and det exactly and leaves t and the barycentric weights as they are,
// so it is left out here.
struct ShearCyclic {
    uint32_t kz;
    float Sx, Sy, Sz;
    float ox, oy, oz;  // origin permuted into (kx, ky, kz)
};

__device__ __forceinline__ void permute(uint32_t kz, float x, float y, float z, float& px, float& py, float& pz) {
    const bool k2 = kz == 2u, k1 = kz == 1u;
    px = k2 ? x : (k1 ? z : y);
    py = k2 ? y : (k1 ? x : z);
    pz = k2 ? z : (k1 ? y : x);
}

__device__ __forceinline__ ShearCyclic make_shear_cyclic(const RayIn& r) {
    ShearCyclic s;
    const float ax = fabsf(r.dx), ay = fabsf(r.dy), az = fabsf(r.dz);
    s.kz = (ax > ay) ? (ax > az ? 0u : 2u) : (ay > az ? 1u : 2u);
    float dx, dy, dz;
    permute(s.kz, r.dx, r.dy, r.dz, dx, dy, dz);
    permute(s.kz, r.ox, r.oy, r.oz, s.ox, s.oy, s.oz);
    s.Sz = __builtin_amdgcn_rcpf(dz);
    s.Sx = dx * s.Sz;
    s.Sy = dy * s.Sz;
    return s;
}

// Watertight ray/triangle test.  Returns true with t in (tmin, tmax] (a hit has t < tmax: the
// caller sees a tie with the hit it has);
// U, V, W are the scaled barycentric weights of v0, v1, v2 and det = U + V + W.
__device__ __forceinline__ bool watertight(const ShearCyclic& s, float4 v0, float4 v1, float4 v2, float tmin,
                                           float tmax, float& t, float& U, float& V, float& W, float& det) {
#pragma clang fp contract(off)
    float Ax, Ay, Az, Bx, By, Bz, Cx, Cy, Cz;
    permute(s.kz, v0.x, v0.y, v0.z, Ax, Ay, Az);
    permute(s.kz, v1.x, v1.y, v1.z, Bx, By, Bz);
    permute(s.kz, v2.x, v2.y, v2.z, Cx, Cy, Cz);
    Ax -= s.ox; Ay -= s.oy; Az -= s.oz;
    Bx -= s.ox; By -= s.oy; Bz -= s.oz;
    Cx -= s.ox; Cy -= s.oy; Cz -= s.oz;
    const float ax = Ax - s.Sx * Az, ay = Ay - s.Sy * Az;
    const float bx = Bx - s.Sx * Bz, by = By - s.Sy * Bz;
    const float cx = Cx - s.Sx * Cz, cy = Cy - s.Sy * Cz;
    return watertight_tail(ax, ay, bx, by, cx, cy, s.Sz * Az, s.Sz * Bz, s.Sz * Cz, tmin, tmax, t, U, V, W, det);
}

// The shear of make_shear as three world-frame rows, for triangles whose vertices are the
// same in every lane (trace_brute), where selecting a vertex's permuted components costs
// more than the shear: with A = v - o, x' = A . (e_kx - Sx e_kz), y' = A . (e_ky - Sy e_kz)
// and z = A . e_kz (exact), by fused multiply-adds.  Every triangle sees a vertex through
// the same arithmetic, so shared edges stay closed.
struct ShearRows {
    float rx[3], ry[3], rz[3];
    float o[3];
    float Sz;
};

__device__ __forceinline__ ShearRows make_shear_rows(const RayIn& r, const Shear& s) {
    ShearRows w;
    for (int k = 0; k < 3; k++) {
        w.rx[k] = (k == s.kx ? 1.f : 0.f) - (k == s.kz ? s.Sx : 0.f);
        w.ry[k] = (k == s.ky ? 1.f : 0.f) - (k == s.kz ? s.Sy : 0.f);
        w.rz[k] = k == s.kz ? 1.f : 0.f;
    }
    w.o[0] = r.ox;
    w.o[1] = r.oy;
    w.o[2] = r.oz;
    w.Sz = s.Sz;
    return w;
}

__device__ __forceinline__ bool watertight_rows(const ShearRows& s, float4 v0, float4 v1, float4 v2, float tmin,
                                                float tmax, float& t, float& U, float& V, float& W, float& det) {
    auto row = [](const float r[3], float x, float y, float z) { return fmaf(z, r[2], fmaf(y, r[1], x * r[0])); };
    const float Ax = v0.x - s.o[0], Ay = v0.y - s.o[1], Az = v0.z - s.o[2];
    const float Bx = v1.x - s.o[0], By = v1.y - s.o[1], Bz = v1.z - s.o[2];
    const float Cx = v2.x - s.o[0], Cy = v2.y - s.o[1], Cz = v2.z - s.o[2];
    const float ax = row(s.rx, Ax, Ay, Az), ay = row(s.ry, Ax, Ay, Az);
    const float bx = row(s.rx, Bx, By, Bz), by = row(s.ry, Bx, By, Bz);
    const float cx = row(s.rx, Cx, Cy, Cz), cy = row(s.ry, Cx, Cy, Cz);
    const float za = row(s.rz, Ax, Ay, Az), zb = row(s.rz, Bx, By, Bz), zc = row(s.rz, Cx, Cy, Cz);
    return watertight_tail(ax, ay, bx, by, cx, cy, s.Sz * za, s.Sz * zb, s.Sz * zc, tmin, tmax, t, U, V, W, det);
}

// Watertight test after the shear: (ax, ay) ... the sheared 2D vertices, za ... their
// scaled distances along the ray.
__device__ __forceinline__ bool watertight_tail(float ax, float ay, float bx, float by, float cx, float cy, float za,
                                                float zb, float zc, float tmin, float tmax, float& t, float& U,
                                                float& V, float& W, float& det) {
#pragma clang fp contract(off)
    U = cx * by - cy * bx;
    V = ax * cy - ay * cx;
    W = bx * ay - by * ax;
    if (fminf(fminf(fabsf(U), fabsf(V)), fabsf(W)) == 0.f) {
        // Exact products in FP64 decide the sign on the edge (Woop et al., section 3.3).
        U = float(double(cx) * double(by) - double(cy) * double(bx));
        V = float(double(ax) * double(cy) - double(ay) * double(cx));
        W = float(double(bx) * double(ay) - double(by) * double(ax));
    }
    if (fminf(fminf(U, V), W) < 0.f && fmaxf(fmaxf(U, V), W) > 0.f) return false;
    det = U + V + W;
    if (det == 0.f) return false;
    const float T = U * za + V * zb + W * zc;
    t = T * __builtin_amdgcn_rcpf(det);  // within 3 ulp of T / det
    return t > tmin && t <= tmax;
}

// The winner re-evaluated in FP64 (Moeller-Trumbore form): t and the weights of v1, v2.  Reads
// only the ray's origin and direction; leaves t, b0, b1 as they are (and returns false) when
// the FP64 determinant is 0.  Fused operations are spelled out: left to the compiler they differed
// from kernel to kernel, and the last bit of one result in 2000 with them.
__device__ __forceinline__ bool refine_fp64(const RayIn& r, float4 v0, float4 v1, float4 v2, float& t, float& b0,
                                            float& b1) {
#pragma clang fp contract(off)
    struct D3 {
        double x, y, z;
    };
    auto cross = [](const D3& a, const D3& b) {
        return D3{fma(a.y, b.z, -(a.z * b.y)), fma(a.z, b.x, -(a.x * b.z)), fma(a.x, b.y, -(a.y * b.x))};
    };
    auto dot = [](const D3& a, const D3& b) { return fma(a.z, b.z, fma(a.x, b.x, a.y * b.y)); };
    const D3 d{r.dx, r.dy, r.dz}, p0{v0.x, v0.y, v0.z};
    const D3 e1{double(v1.x) - p0.x, double(v1.y) - p0.y, double(v1.z) - p0.z};
    const D3 e2{double(v2.x) - p0.x, double(v2.y) - p0.y, double(v2.z) - p0.z};
    const D3 s1 = cross(d, e2);
    const double div = dot(s1, e1);
    if (div == 0.0) return false;
    const double inv = 1.0 / div;
    const D3 q{r.ox - p0.x, r.oy - p0.y, r.oz - p0.z};
    const D3 s2 = cross(q, e1);
    t = float(dot(e2, s2) * inv);
    b0 = float(dot(q, s1) * inv);
    b1 = float(dot(d, s2) * inv);
    return true;
}

// Hardware reciprocal (v_rcp_f32, within 1 ulp) of a direction component kept away from 0.
__device__ __forceinline__ float safe_rcp(float d) {
    return __builtin_amdgcn_rcpf(fabsf(d) > 1e-30f ? d : copysignf(1e-30f, d));
}

__device__ __forceinline__ Slab make_slab(const RayIn& r) {
    return make_slab(r.ox, r.oy, r.oz, safe_rcp(r.dx), safe_rcp(r.dy), safe_rcp(r.dz));
}

// Orders two (key, reference) pairs, nearer first.  A pair is one 64-bit value, the key in the
// upper half: read as doubles such values order by key (floats order like the upper halves of
// doubles, and the lower half only decides between equal keys), so the exchange is one
// minimum and one maximum instead of a compare and four selects.
__device__ __forceinline__ void cswap(double& a, double& b) {
    double lo, hi;
    asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
    asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
    a = lo;
    b = hi;
}

__device__ __forceinline__ double pack_entry(float key, uint32_t ref) {
    return __hiloint2double(int(__float_as_uint(key)), int(ref));
}
__device__ __forceinline__ uint32_t entry_ref(double e) { return uint32_t(__double2loint(e)); }
__device__ __forceinline__ float entry_key(double e) { return __uint_as_float(uint32_t(__double2hiint(e))); }

constexpr uint32_t kDone = 0xffffffffu;  // nothing left to visit
constexpr uint32_t kPop = 0xfffffffeu;   // the next reference is on the stack (no leaf of 16 records starts at 2^27 - 2)
__device__ __forceinline__ bool is_inner(uint32_t ref) { return int(ref) >= 0; }
__device__ __forceinline__ bool is_leaf(uint32_t ref) { return ref >= kLeafBit && ref < kPop; }

// Node words are fetched through a buffer resource over the node array: the
// constant part of each fetch's offset goes into the instruction's offset field, so a fetch
// costs one 32-bit address add (a global load needs 64-bit address arithmetic to fold it),
// and the 64-bit temporaries' registers are freed.  The resource's record count, 2^32 - 1
// bytes, lets every fetch of a tree through: kMaxNodes packed nodes end at 2^31.
struct NodeFetch {
    __amdgpu_buffer_rsrc_t rsrc;
    __device__ __forceinline__ explicit NodeFetch(const NodeQ* nodes)
        // word 3 of a gfx9 raw buffer resource: 32-bit data format, no swizzle, no stride.
        : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<NodeQ*>(nodes), short(0), -1, 0x00020000)) {}
    __device__ __forceinline__ float4 operator()(uint32_t off) const {
        return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0));
    }
};

// Slab tests of the four children of packed node `cur`, sorted into entries (key = entry distance,
// reference), nearest first; a missed child's key is +inf.  Per axis the direction's sign selects
// the planes entered first and left last of all four children, so the entry and exit distances
// need no min / max per axis; the inverted box of an empty slot is entered only by rounding or NaN.
__device__ __forceinline__ void node_children(const NodeFetch& fetch, uint32_t cur, const Slab& s, float tmin, float tmax,
                                              double e[4]) {
    // 32-bit byte offsets from the node array (at most kMaxNodes nodes, checked by the builder).
    const uint32_t o = cur * uint32_t(sizeof(NodeQ));
    const float4 q0 = fetch(o), q1 = fetch(o + 16u), q2 = fetch(o + 32u), q3 = fetch(o + 48u);
    const PackedAxis x = packed_axis(q0.x, q0.w, __float_as_uint(q1.z), __float_as_uint(q1.w), s.ix, s.nx, s.fx);
    const PackedAxis y = packed_axis(q0.y, q1.x, __float_as_uint(q2.x), __float_as_uint(q2.y), s.iy, s.ny, s.fy);
    const PackedAxis z = packed_axis(q0.z, q1.y, __float_as_uint(q2.z), __float_as_uint(q2.w), s.iz, s.nz, s.fz);
    const float c[4] = {q3.x, q3.y, q3.z, q3.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float tn, tf;
        packed_span(x, y, z, i, tmin, tmax, tn, tf);
        e[i] = pack_entry(tn <= widened(tf, kBoxRobust) ? tn : INFINITY, __float_as_uint(c[i]));
    }
    cswap(e[0], e[1]);
    cswap(e[2], e[3]);
    cswap(e[0], e[2]);
    cswap(e[1], e[3]);
    cswap(e[1], e[2]);
}

// Records a triangle that trace_brute accepted in h; closest hit also keeps the watertight test's
// scaled weights V and W of v1 and v2 and their sum det, which hit_weights turns into barycentric
// weights once the ray is done.
template <bool kAny>
__device__ __forceinline__ void accept_hit(HitOut& h, float t, uint32_t rec, uint32_t prim, float V, float W,
                                           float det) {
    h.t = t;
    h.rec = rec;
    h.prim = prim;
    if (!kAny) {
        h.b0 = V;
        h.b1 = W;
        h.det = det;
    }
}
__device__ __forceinline__ void hit_weights(HitOut& h) {
    const float inv = 1.f / h.det;
    h.b0 *= inv;
    h.b1 *= inv;
}

// A BVH record's hit as the descent saw it: the same test gives the same t and weights.
__device__ __forceinline__ HitOut hit_at(const LeafTri* tris, uint32_t rec, const RayIn& r) {
    const float4* tp = reinterpret_cast<const float4*>(tris + rec);
    const float4 v0 = tp[0], v1 = tp[1], v2 = tp[2];
    HitOut h{-1.f, rec, __float_as_uint(v0.w), 0.f, 0.f, 1.f};
    float U;
    (void)watertight(make_shear_cyclic(r), v0, v1, v2, r.tmin, r.tmax, h.t, U, h.b0, h.b1, h.det);
    hit_weights(h);
    return h;
}

// The LDS of one traversal block: the stacks' LDS levels ([level][thread]), for closest hit
// with the entry distance in an entry's upper half.
template <bool kKeys> struct StackLevels;
template <> struct StackLevels<true> {
    using Entry = double;
    static constexpr uint32_t kLds = 12;
};
template <> struct StackLevels<false> {
    using Entry = uint32_t;
    static constexpr uint32_t kLds = 16;
};
template <bool kKeys> struct TraceShared {
    typename StackLevels<kKeys>::Entry stack[StackLevels<kKeys>::kLds * kTraceBlock];
};

// The per-lane traversal stack: the first levels live in LDS (`lds` is this lane's column,
// lds[level * kTraceBlock]), deeper ones in private memory.  The builder bounds
// 3 * depth <= kStackTotal, so the guard in push never fires.
// With kKeys (closest hit) every entry carries the entry distance of its box, and pop skips
// entries whose distance exceeds the current tmax * kBoxRobust: the box test would reject
// them now that a nearer hit shrank tmax, so they are never fetched.
// The spill array is owned by the caller (a separate private array, so the stack pointer and
// the LDS columns stay in registers).
template <bool kKeys> struct TraceStack {
    using Entry = typename StackLevels<kKeys>::Entry;
    static constexpr uint32_t kLds = StackLevels<kKeys>::kLds;
    // Spelled with its address space: from two generic pointers the compiler made one flat access
    // of each push and pop, which goes through the vector memory path.
    __attribute__((address_space(3))) Entry* lds;
    Entry* spill;
    uint32_t sp = 0;

    static __device__ __forceinline__ Entry entry(double e) {
        if constexpr (kKeys) return e;
        else return entry_ref(e);
    }
    __device__ __forceinline__ void push(double e) {
        if (sp < kLds) lds[sp * kTraceBlock] = entry(e);
        else if (sp < uint32_t(kStackTotal)) spill[sp - kLds] = entry(e);
        else return;
        sp++;
    }
    // Pushes the hit ones of the sorted entries e[3], e[2], e[1], in that order.
    __device__ __forceinline__ void push_sorted(const double e[4]) {
        if (sp + 3u <= kLds) {
#pragma unroll
            for (int i = 3; i > 0; i--)
                if (entry_key(e[i]) < INFINITY) lds[sp++ * kTraceBlock] = entry(e[i]);
        } else {
            for (int i = 3; i > 0; i--)
                if (entry_key(e[i]) < INFINITY) push(e[i]);
        }
    }
    // Takes the top entry: its reference, kPop when the entry is skipped, kDone when there is none.
    __device__ __forceinline__ uint32_t pop(float tmax) {
        if (sp == 0u) return kDone;
        sp--;
        Entry e;
        if (sp < kLds) e = lds[sp * kTraceBlock];
        else e = spill[sp - kLds];
        if constexpr (kKeys) return entry_key(e) > fmaxf(tmax * kBoxRobust, 0.f) ? kPop : entry_ref(e);
        else return e;
    }
};

// Descends from a node: pushes the farther hit children (the keys matter for closest hit
// only) and returns the nearest, or kPop when none is hit.
// Any hit descends nearest first too: it finds an occluder sooner (any-hit batch -1.7 %).
template <class Stack> __device__ __forceinline__ uint32_t descend(const double e[4], Stack& st) {
    st.push_sorted(e);
    return entry_key(e[0]) < INFINITY ? entry_ref(e[0]) : kPop;
}

__device__ __forceinline__ void cswap(float& ka, uint32_t& va, float& kb, uint32_t& vb) {
    const bool s = kb < ka;
    const float tk = s ? kb : ka;
    const uint32_t tv = s ? vb : va;
    kb = s ? ka : kb;
    vb = s ? va : vb;
    ka = tk;
    va = tv;
}

// The built node's children nearest first; equal keys as this network leaves them.
__device__ __forceinline__ void sort4(float key[4], uint32_t val[4]) {
    cswap(key[0], val[0], key[1], val[1]);
    cswap(key[2], val[2], key[3], val[3]);
    cswap(key[0], val[0], key[2], val[2]);
    cswap(key[1], val[1], key[3], val[3]);
    cswap(key[1], val[1], key[2], val[2]);
}

// Child `i` of a built node along the ray: its entry distance (+inf if it is missed or empty), its
// reference and its exit distance.
__device__ __forceinline__ float built_child(const BvhDev& bvh, const Slab& s, uint32_t node, uint32_t i, float tmin,
                                             float tmax, uint32_t& child, float& tf) {
    const float* nd = reinterpret_cast<const float*>(bvh.exact + node) + i;
    child = __float_as_uint(nd[24]);
    float tn;
    box_span(s, nd[0], nd[4], nd[8], nd[12], nd[16], nd[20], tmin, tmax, tn, tf);
    return child != kEmptyChild && tn <= widened(tf, kBoxRobustExact) ? tn : INFINITY;
}

// Whether a ray meets the box of a record's leaf as it was built (lx, hx: its x range, the fourth
// column of v1 and v2), by built_child's operations, and where it enters (`tn`).  The built boxes
// above contain this one and their tests round monotonically, so they accept whatever it accepts.
__device__ __forceinline__ bool in_leaf_box(const LeafTri& rec, float lx, float hx, const Slab& s, float tmin, float tmax,
                                            float& tn) {
    const float4 b = *reinterpret_cast<const float4*>(rec.box_yz);
    float tf;
    box_span(s, lx, hx, b.x, b.y, b.z, b.w, tmin, tmax, tn, tf);
    return tn <= widened(tf, kBoxRobustExact);
}

// What orders a ray's hits: the distance, but no less than where the ray enters the hit's leaf.  The
// FP32 test of a triangle that is large, thin or seen edge-on can place a hit before its own box;
// a descent that has met a hit between the two by then leaves the box out, another finds it first.
// Ordered so, no box test leaves out a hit that comes before the nearest one so far, whatever the
// order of the descent (kOrderPrune), and every kernel finds the same one.
__device__ __forceinline__ float hit_order(float t, float tn) { return fmaxf(t, tn * kOrderScale); }

// A descent that takes hits by their distance alone, and through packed boxes, ends at the first hit
// in that order if the record it ends at (`rec`, at distance t) is in its leaf's box and not before
// it: another that comes before in the order is nearer too, and was not left out unless a nearer
// one still was accepted.  The few other rays are traced again (trace_exact).  For any hit the box
// alone counts.
template <bool kAny>
__device__ __forceinline__ bool sound_hit(const BvhDev& bvh, uint32_t rec, const Slab& s, const RayIn& r, float t) {
    const LeafTri& l = bvh.tris[rec];
    float tn;
    return in_leaf_box(l, l.v1[3], l.v2[3], s, r.tmin, r.tmax, tn) && (kAny || tn * kOrderScale <= t);
}

// 2^-21 of the coordinates involved in a distance along r, which is known to a few units of 2^-24
// of them.
__device__ __forceinline__ float distance_band(const BvhDev& bvh, const RayIn& r, const ShearCyclic& sh) {
    return 4.76837158203125e-7f * fabsf(sh.Sz) * (fmaxf(fmaxf(fabsf(r.ox), fabsf(r.oy)), fabsf(r.oz)) + bvh.reach);
}

// The built boxes say which records a ray may hit and which of two at one place in the order
// (hit_order) comes first: the one that their descent meets first.  A ray whose hit is in doubt is
// traced again here, one node or leaf after the other in that order (kDone: none): to the first record at `t_hit`
// where only that is in doubt, through the whole interval where t_hit is -inf (sound_hit is false).
// Boxes away from t_hit by more than 1e-3 of it and `band`, a thousand times what a distance
// commonly is off by, are left out at first: after the node's children are sorted, so that the others
// keep their order.  Should no record be found so, the whole interval is traced.
// Ties are 1 in 10^6 of the rays in a city, but all of those that meet two lights in one plane:
// 1.1M camera rays over 16 overlapping lights 222 us with the whole interval, 212 us so; where a group
// of lanes looks for it together (trace_grouped), 45824 rays 70 and 37 us.
template <class Stack>
__device__ __forceinline__ uint32_t trace_exact(const BvhDev& bvh, const RayIn& r, float t_hit, Stack& st) {
    const Slab s = make_slab(r);
    const ShearCyclic sh = make_shear_cyclic(r);
    const float band = 1000.f * distance_band(bvh, r, sh);
    uint32_t rec = kDone;
    float best = t_hit, far = fminf(fmaf(t_hit, 1.f + 1e-3f, band), r.tmax), near = fmaf(t_hit, 1.f - 1e-3f, -band);
    bool first = t_hit > -INFINITY;  // the first record at t_hit is looked for
    uint32_t cur = first ? 0u : kDone;
    bool all = false;  // the whole interval
    st.sp = 0u;
    for (;;) {
        if (cur == kDone) {
            if (all) break;
            first = false;
            all = true;
            best = INFINITY;
            far = r.tmax;
            near = -INFINITY;
            cur = 0u;
        }
        if (is_inner(cur)) {
            const float4* n = reinterpret_cast<const float4*>(bvh.exact + cur);
            const uint32_t x = s.ix >= 0.f ? 0u : 1u, y = s.iy >= 0.f ? 0u : 1u, z = s.iz >= 0.f ? 0u : 1u;
            const float4 nxv = n[x], fxv = n[1u - x], nyv = n[2u + y], fyv = n[3u - y], nzv = n[4u + z], fzv = n[5u - z];
            const float4 cv = n[6];
            const float nx[4] = {nxv.x, nxv.y, nxv.z, nxv.w}, fx[4] = {fxv.x, fxv.y, fxv.z, fxv.w};
            const float ny[4] = {nyv.x, nyv.y, nyv.z, nyv.w}, fy[4] = {fyv.x, fyv.y, fyv.z, fyv.w};
            const float nz[4] = {nzv.x, nzv.y, nzv.z, nzv.w}, fz[4] = {fzv.x, fzv.y, fzv.z, fzv.w};
            const float c[4] = {cv.x, cv.y, cv.z, cv.w};
            float key[4];
            uint32_t val[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float tn = fmaxf(fmaxf(fmaf(nx[i], s.ix, s.nx), fmaf(ny[i], s.iy, s.ny)),
                                       fmaxf(fmaf(nz[i], s.iz, s.nz), r.tmin));
                const float tf = fminf(fminf(fmaf(fx[i], s.ix, s.fx), fmaf(fy[i], s.iy, s.fy)),
                                       fminf(fmaf(fz[i], s.iz, s.fz), far));
                val[i] = __float_as_uint(c[i]);
                key[i] = val[i] != kEmptyChild && tn <= widened(tf, kBoxRobustExact) ? tn : INFINITY;
                if (tf < near) val[i] = kEmptyChild;
            }
            sort4(key, val);
            cur = kDone;
#pragma unroll
            for (int i = 3; i >= 0; i--) {
                if (!(key[i] < INFINITY) || val[i] == kEmptyChild) continue;
                if (cur != kDone) st.push(pack_entry(-INFINITY, cur));
                cur = val[i];
            }
        } else {
            const uint32_t begin = cur & kMaxLeafFirst, end = begin + ((cur >> 27) & 0xfu) + 1u;
            for (uint32_t k = begin; k < end; k++) {
                const float4* tp = reinterpret_cast<const float4*>(bvh.tris + k);
                const float4 v0 = tp[0], v1 = tp[1], v2 = tp[2];
                float t, U, V, W, det, tn;
                if (!watertight(sh, v0, v1, v2, r.tmin, far, t, U, V, W, det) || !(t < r.tmax)) continue;
                (void)in_leaf_box(bvh.tris[k], v1.w, v2.w, s, r.tmin, r.tmax, tn);
                const float at = hit_order(t, tn);
                if (first ? at == t_hit : at < best) {
                    best = at;
                    far = fminf(widened(at, kOrderPrune), r.tmax);
                    rec = k;
                    if (first) return rec;
                }
            }
            cur = kDone;
        }
        if (cur == kDone) cur = st.pop(far);
    }
    return rec;
}

// The same for any hit, where no order counts: whether a record of a leaf whose built box the ray
// meets is hit.
template <class Stack> __device__ __forceinline__ bool occluded_exact(const BvhDev& bvh, const RayIn& r, Stack& st) {
    const Slab s = make_slab(r);
    const ShearCyclic sh = make_shear_cyclic(r);
    uint32_t cur = 0u;
    st.sp = 0u;
    while (cur != kDone) {
        uint32_t next = kDone;
        if (is_inner(cur)) {
#pragma unroll 1
            for (uint32_t i = 0; i < 4u; i++) {
                uint32_t child;
                float tf;
                if (!(built_child(bvh, s, cur, i, r.tmin, r.tmax, child, tf) < INFINITY)) continue;
                if (next != kDone) st.push(pack_entry(-INFINITY, next));
                next = child;
            }
        } else {
            const uint32_t begin = cur & kMaxLeafFirst, end = begin + ((cur >> 27) & 0xfu) + 1u;
#pragma unroll 1
            for (uint32_t k = begin; k < end; k++) {
                const float4* tp = reinterpret_cast<const float4*>(bvh.tris + k);
                const float4 v0 = tp[0], v1 = tp[1], v2 = tp[2];
                float t, U, V, W, det;
                if (watertight(sh, v0, v1, v2, r.tmin, r.tmax, t, U, V, W, det) && t < r.tmax) return true;
            }
        }
        cur = next != kDone ? next : st.pop(r.tmax);
    }
    return false;
}

// A wave fetches new rays once this many of its lanes are idle: fetching costs the setup of the
// rays' constants for the idle lanes only, waiting leaves lanes out of every step.  16M rays: 12
// idle lanes 3.14 ms, 16: 3.08, 28: 3.25; extension rays of the 96k-triangle room 10.6, 10.6, 10.9.
constexpr uint32_t kRefillIdle = 16;
// A wave takes a node step while at least this many times more lanes wait at nodes than hold a
// leaf: a leaf step is shorter and frees its lanes to shrink tmax.  2 against 1: extension rays
// 11.8 -> 11.5 ms, 1M-triangle city 2.65 -> 2.49 ms, 16M rays the same; 3: 11.8 ms.
constexpr uint32_t kLeafWeight = 2;

// Persistent traversal with per-lane ray refill (Aila & Laine, "Understanding the
// efficiency of ray traversal on GPUs", HPG 2009): every wave of the grid loops over its rays,
// and lanes whose rays have finished fetch new ones once kRefillIdle of the wave's lanes are
// idle.  A batch of up to kEvenRounds rays per lane is dealt out beforehand; a larger one gives
// each wave 64 rays and the rest in ranges claimed from `next` (which counts from 64 x the
// number of waves) one range ahead of need, so that a refill waits for no atomic.
// A lane visits nodes until it meets a leaf, and goes on visiting nodes while the leaf's
// triangles are still to be tested (speculative traversal, same paper); a second leaf stops
// it.  Each step of the wave serves the larger of the two groups.  A lane whose node left
// nothing to descend into takes one entry off its stack a step: a loop until every lane had
// one ran 102 times per 64 rays with 4 lanes each.
// `src(i)` returns ray i, `sink(i, found, h, r)` consumes its result.  Every wave exits
// once the batch is exhausted and its own lanes are done.  With kCount, `cnt` sums the
// lane's node visits and triangle tests over all rays it traced.
// n is at most kMaxBatch: a claim past the end then never wraps the counter.
constexpr uint32_t kMaxBatch = 0x80000000u;
// Up to this many rays per lane of the grid a wave's rays are fixed beforehand, consecutive and as
// many for each: 0.9M camera rays 240 -> 153 us, extension rays of the 96k-triangle room 12.0 ->
// 10.6 ms, shadow rays of a 1M-triangle city 1.10 -> 0.85 ms.  Beyond, ranges claimed as they are
// needed balance better (24 instead of 16: extension rays 11.3 ms; 64: 16M rays 3.09 -> 3.25 ms).
constexpr uint32_t kEvenRounds = 16;
template <bool kAny, bool kCount, class Source, class Sink>
__device__ __forceinline__ void trace_persistent(const BvhDev& bvh, uint32_t n, uint32_t* next, TraceShared<!kAny>& sm, Source& src,
                                                 Sink& sink, TraceCounters& cnt) {
    typename TraceStack<!kAny>::Entry spill[kStackTotal - TraceStack<!kAny>::kLds];
    TraceStack<!kAny> st{(__attribute__((address_space(3))) typename TraceStack<!kAny>::Entry*)(sm.stack + threadIdx.x), spill};
    constexpr uint32_t kNone = 0xffffffffu;
    const uint32_t lane = __lane_id();
    uint32_t id = kNone;
    RayIn r{0.f, 0.f, 0.f, 0.f, 0.f, 1.f, 0.f, 0.f};
    float tmax = 0.f;
    Slab sl = make_slab(r);
    ShearCyclic sh = make_shear_cyclic(r);
    HitOut h{};
    bool found = false;
    bool tie = false;  // closest hit: another triangle at the nearest distance
    // Closed rays that trace_exact decides, kTies at most; a lane with a full list takes no further ray.
    constexpr uint32_t kTies = 4;
    uint32_t ties[kTies];
    float ties_at[kAny ? 1 : kTies];
    uint32_t num_ties = 0u;
    uint32_t cur = kDone;   // next node or leaf reference to visit
    uint32_t tri = 0u, tri_end = 0u;  // records left of the leaf being tested
    const NodeFetch fetch(bvh.nodes);
    // A leaf next in line becomes the one being tested if there is none.
    auto take_leaf = [&]() {
        if (is_leaf(cur) && tri >= tri_end) {
            tri = cur & kMaxLeafFirst;
            tri_end = tri + ((cur >> 27) & 0xfu) + 1u;
            cur = kPop;
        }
    };
    auto start = [&](uint32_t k) {
        id = k;
        r = src(k);
        sl = make_slab(r);
        sh = make_shear_cyclic(r);
        tmax = r.tmax;
        found = tie = false;
        tri = tri_end = 0u;
        st.sp = 0u;
        cur = 0u;
    };
    // A triangle passed at t in (tmin, tmax].
    auto meet = [&](uint32_t k, float t) {
        if (t < tmax) {
            tie = false;
            found = true;
            if (!kAny) tmax = t;
            h.rec = k;
        } else if (!kAny) {
            tie = found;
        }
    };
    const uint32_t waves = gridDim.x * (blockDim.x >> 6);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    const uint32_t static_total = waves * 64u;
    // A batch of up to kEvenRounds rays per lane is spread evenly over all waves, each taking
    // ceil(n / waves) consecutive ones, 64 at least: ranges would give some waves a round more than
    // others.  (Fewer rays in more waves: 112000 camera rays of a city 62 instead of 52 us.)
    const bool even = n <= static_total * kEvenRounds;
    const uint32_t chunk = even ? max((n + waves - 1u) / waves, 64u) : 64u;
    uint32_t cur_next = min(wave * chunk + min(chunk, 64u), n);
    uint32_t cur_end = even ? uint32_t(min(uint64_t(wave + 1u) * chunk, uint64_t(n))) : cur_next;
    if (lane < min(chunk, 64u) && wave * chunk + lane < n) start(wave * chunk + lane);
    bool exhausted = cur_next >= (even ? cur_end : n);  // no ray is taken (wave-uniform)
    // Ranges: [cur_next, cur_end) is being handed out; `pend` (held by lane 0) is the base of the
    // next one, of pend_size rays.  A range holds a share of what is left, between 64
    // and kMaxRange rays, so a long batch costs few atomics and its end stays balanced.
    constexpr uint32_t kMaxRange = 1024u;
    const uint32_t share = 33u - uint32_t(__clz(int(waves)));  // log2 of 2 to 4 times the waves
    uint32_t pend = 0u, pend_size = 0u;
    auto range_size = [&](uint32_t at) {
        const uint32_t left = at < n ? n - at : 0u;
        return min(max((left >> share) & ~63u, 64u), kMaxRange);
    };
    auto refill = [&]() {
        const bool need = id == kNone && num_ties < kTies;
        const unsigned long long mask = __ballot(need);
        const uint32_t want = uint32_t(__popcll(mask));
        if (want == 0u) {
            // The waiting lanes' lists are full: no more rays until those under way are done and the
            // lists resolved, or the wave would come back at every step.
            exhausted = true;
            return;
        }
        const uint32_t rank = uint32_t(__popcll(mask & ((1ull << lane) - 1ull)));
        const uint32_t avail = cur_end - cur_next;
        uint32_t k = cur_next + rank;
        if (even) {
            if (need && rank < avail) start(k);
            cur_next = min(cur_next + want, cur_end);
            exhausted = cur_next >= cur_end;
            return;
        }
        if (want > avail) {
            uint32_t base = 0u, size = pend_size;
            if (size != 0u) {
                base = __builtin_amdgcn_readfirstlane(pend);
                pend_size = 0u;
            } else {
                size = range_size(max(cur_end, static_total));
                if (lane == 0u) base = static_total + atomicAdd(next, size);
                base = __builtin_amdgcn_readfirstlane(base);
            }
            if (rank >= avail) k = base + (rank - avail);
            cur_next = base + (want - avail);
            cur_end = base + size;
        } else {
            cur_next += want;
        }
        if (need && k < n) start(k);
        if (cur_next >= n) {
            exhausted = true;
        } else if (pend_size == 0u && cur_end < n && n - cur_end > static_total) {
            pend_size = range_size(max(cur_end, static_total));
            if (lane == 0u) pend = static_total + atomicAdd(next, pend_size);
        }
    };
    for (;;) {
        for (;;) {
            const unsigned long long nm = __ballot(is_inner(cur)), lm = __ballot(tri < tri_end);
            const unsigned long long pm = __ballot(cur == kPop);
            const uint32_t nn = uint32_t(__popcll(nm)), nl = uint32_t(__popcll(lm)), busy = uint32_t(__popcll(nm | lm | pm));
            if (busy == 0u || (!exhausted && busy <= 64u - kRefillIdle)) {
                if (id != kNone && cur == kDone && tri >= tri_end) {
                    const bool sound = !found || sound_hit<kAny>(bvh, h.rec, sl, r, tmax);
                    if (tie || !sound) {
                        if (!kAny) ties_at[num_ties] = sound ? tmax : -INFINITY;
                        ties[num_ties++] = id;
                    } else {
                        sink(id, found, h, r);
                    }
                    id = kNone;
                }
                if (busy == 0u && exhausted) break;
                refill();
            } else if (nn >= nl * kLeafWeight) {
                if (is_inner(cur)) {
                    if (kCount) cnt.nodes++;
                    double e[4];
                    node_children(fetch, cur, sl, r.tmin, tmax, e);
                    cur = descend(e, st);
                    take_leaf();
                }
            } else {
                if (tri < tri_end) {
                    // Two records a step: they share a line unless the second starts the next one.
                    const bool two = tri + 1u < tri_end;
                    const float4* ap = reinterpret_cast<const float4*>(bvh.tris + tri);
                    const float4* bp = ap + (two ? sizeof(LeafTri) / 16 : 0);
                    const float4 a0 = ap[0], a1 = ap[1], a2 = ap[2];
                    const float4 b0 = bp[0], b1 = bp[1], b2 = bp[2];
                    float t, U, V, W, det;
                    if (kCount) cnt.tris++;
                    if (watertight(sh, a0, a1, a2, r.tmin, tmax, t, U, V, W, det))
                        meet(tri, t);
                    if (two && !(kAny && found)) {
                        if (kCount) cnt.tris++;
                        if (watertight(sh, b0, b1, b2, r.tmin, tmax, t, U, V, W, det))
                            meet(tri + 1u, t);
                    }
                    tri += 2u;
                    if (kAny && found) {
                        cur = kDone;
                        tri_end = 0u;
                    }
                    take_leaf();
                }
            }
            if (cur == kPop) {
                cur = st.pop(tmax);
                take_leaf();
            }
        }
        // All lanes are idle: nothing of the loop above is live here.
        while (num_ties > 0u) {
            num_ties--;
            const RayIn q = src(ties[num_ties]);
            if constexpr (kAny) {
                sink(ties[num_ties], occluded_exact(bvh, q, st), h, q);
            } else {
                h.rec = trace_exact(bvh, q, ties_at[num_ties], st);
                sink(ties[num_ties], h.rec != kDone, h, q);
            }
        }
        exhausted = cur_next >= (even ? cur_end : n);
        if (exhausted) break;
        r = RayIn{0.f, 0.f, 0.f, 0.f, 0.f, 1.f, 0.f, 0.f};
        sl = Slab{};
        sh = ShearCyclic{};
        h = HitOut{};
        tmax = 0.f;
        found = tie = false;
        id = kNone;
        cur = kDone;
        tri = tri_end = 0u;
        st.sp = 0u;
        refill();
    }
}

// ---- Several lanes per ray ----------------------------------------------------------------
// Batches with few rays for the chip -- a probe, a late bounce -- last as long as one ray's
// chain of dependent fetches.  Here kLanes lanes follow one ray: each round takes up to
// kLanes / 4 nodes off the ray's stack, nearest on top, and every lane tests one child of one
// of them; the leaves found are tested at once, one triangle per lane.  With 64 lanes the chain
// is about the tree's depth instead of every node and leaf the ray visits.  The boxes are the
// built ones, so a leaf is met exactly if a depth-first descent could meet it; ties go to
// trace_exact.  The lanes of a ray are consecutive and every branch is uniform among them.
// Measured on device rays with the FP64 evaluation (1k to 1M triangles), us a batch: 81 rays 76-106
// one lane each, 8-14 with 64 lanes each; 1000 rays 98-136 -> 9-14; 32768 rays 97-193 -> 22-33 with
// 16 lanes each.  With three streams in flight the one-lane kernel overlaps its tails: 41-75 at 32768
// rays, 35-87 at 65549 against 42-67 with 16 lanes, hence the bounds:
constexpr uint32_t kGroup64Rays = 8192;     // 64 lanes per ray (4000 rays: 6-9 against 8-16 with 16 lanes; 16384: 18-24, 12-19)
constexpr uint32_t kGroup16Closest = 65536;  // 16 lanes per ray, closest hit
constexpr uint32_t kGroup16Any = 98304;      // any hit (65549 rays: 27-48 against 36-72; 131072: 53-94, 42-82)
template <int kLanes> struct GroupShared {
    static constexpr uint32_t kRays = kTraceBlock / kLanes;
    // Entries that one node at a time can add (3 * depth), and as much again for kLanes / 4.
    static constexpr uint32_t kDeep = 96, kRoom = kLanes == 64 ? 160 : 48;
    uint2 node[kRays][kDeep + kRoom];  // reference, entry distance
    uint32_t leaf[kRays][kLanes];
};

// Orders a wave's LDS writes before its later reads (the hardware keeps them in order).
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Group g of the grid traces rays g, g + groups, ...; as in trace_persistent, `sink` is called once
// per ray, by one lane.  With kCount the lanes count the children and triangles they test.
template <bool kAny, bool kCount, int kLanes, class Source, class Sink>
__device__ __forceinline__ void trace_grouped(const BvhDev& bvh, uint32_t n, GroupShared<kLanes>& sm, Source& src,
                                              Sink& sink, TraceCounters& cnt) {
    constexpr uint32_t kNodes = kLanes / 4;
    const uint32_t lane = __lane_id() & (kLanes - 1u), base = __lane_id() & ~(kLanes - 1u);
    const uint32_t sub = lane & 3u, slot = lane >> 2, quad = lane & ~3u;
    const uint32_t in_block = threadIdx.x / kLanes, groups = gridDim.x * (kTraceBlock / kLanes);
    auto ballot = [&](bool p) -> unsigned long long {
        const unsigned long long m = __ballot(p);
        if constexpr (kLanes == 64) return m;
        else return (m >> base) & ((1ull << kLanes) - 1ull);
    };
    uint2* stack = sm.node[in_block];
    uint32_t* leaves = sm.leaf[in_block];
    for (uint32_t i = blockIdx.x * (kTraceBlock / kLanes) + in_block; i < n; i += groups) {
        const RayIn r = src(i);
        const Slab sl = make_slab(r);
        const ShearCyclic sh = make_shear_cyclic(r);
        float tmax = r.tmax, limit = r.tmax;  // boxes that begin beyond `limit` hold no hit before tmax
        HitOut h{};
        float nearest = INFINITY;         // of the triangles this lane met: h.rec
        bool found = false, tie = false;  // of the ray
        uint32_t sp = 1u;
        wave_fence();
        if (lane == 0u) stack[0] = make_uint2(0u, 0xff800000u);
        while (sp > 0u && !(kAny && found)) {
            // As many nodes as their children are sure to fit for.
            const uint32_t take = sp + 3u * kNodes <= GroupShared<kLanes>::kRoom ? min(sp, kNodes) : 1u;
            wave_fence();
            const uint2 e = stack[slot < take ? sp - 1u - slot : 0u];
            sp -= take;
            bool hit = false;
            float tn = INFINITY;
            uint32_t child = kEmptyChild;
            if (slot < take && !(__uint_as_float(e.y) > widened(limit, kBoxRobustExact))) {
                if (kCount) cnt.nodes += sub == 0u ? 1u : 0u;
                float tf;
                tn = built_child(bvh, sl, e.x, sub, r.tmin, limit, child, tf);
                hit = tn < INFINITY;
            }
            const bool inner = hit && is_inner(child), leaf = hit && !is_inner(child);
            // Inner children: the top node's on top, each node's nearest uppermost.
            const unsigned long long im = ballot(inner);
            const uint32_t key = inner ? __float_as_uint(fmaxf(tn, 0.f)) : 0x7f800000u;
            uint32_t rank = 0u;
#pragma unroll
            for (uint32_t k = 1; k < 4u; k++) {
                const uint32_t other = uint32_t(__shfl_xor(int(key), int(k), 64));
                rank += other < key || (other == key && (sub ^ k) < sub) ? 1u : 0u;
            }
            const uint32_t below = uint32_t(__popcll(im >> quad));  // in this node and the ones under it
            wave_fence();
            if (inner) stack[sp + below - 1u - rank] = make_uint2(child, __float_as_uint(tn));
            sp += uint32_t(__popcll(im));
            const unsigned long long lm = ballot(leaf);
            const uint32_t nl = uint32_t(__popcll(lm));
            if (nl == 0u) continue;
            if (leaf) leaves[__popcll(lm & ((1ull << lane) - 1ull))] = child;
            wave_fence();
            for (uint32_t l = 0; l < nl && !(kAny && found); l += kNodes) {
                const uint32_t ref = l + slot < nl ? leaves[l + slot] : kDone;
                uint32_t tri = (ref & kMaxLeafFirst) + sub, end = tri - sub + ((ref >> 27) & 0xfu) + 1u;
                if (ref == kDone) end = tri = 0u;
                for (; ballot(tri < end) != 0ull; tri += 4u) {
                    float t = INFINITY, U, V, W, det;
                    bool met = false, same = false;
                    if (tri < end) {
                        if (kCount) cnt.tris++;
                        const float4* tp = reinterpret_cast<const float4*>(bvh.tris + tri);
                        const float4 v0 = tp[0], v1 = tp[1], v2 = tp[2];
                        if (watertight(sh, v0, v1, v2, r.tmin, tmax, t, U, V, W, det)) {
                            met = t < tmax;
                            same = !met && found;
                            if (met) {
                                nearest = t;
                                h.rec = tri;
                            }
                        }
                    }
                    const bool any_met = ballot(met) != 0ull;
                    if (kAny) {
                        found = found || any_met;
                        if (found) break;
                        continue;
                    }
                    tie = tie || ballot(same) != 0ull;
                    if (any_met) {
                        found = true;
                        float m = met ? t : INFINITY;
#pragma unroll
                        for (int off = kLanes / 2; off > 0; off >>= 1) m = fminf(m, __shfl_xor(m, off, 64));
                        tmax = m;
                        limit = fminf(widened(m, kOrderPrune), r.tmax);
                        tie = __popcll(ballot(met && t == tmax)) > 1;
                    }
                }
            }
        }
        if (kAny) {
            if (lane == 0u) sink(i, found, h, r);
            continue;
        }
        unsigned long long holders = ballot(found && nearest == tmax);
        // The boxes were the built ones, but a hit before its own may have kept another from being met.
        const bool sound = !found || ballot(nearest == tmax && !sound_hit<false>(bvh, h.rec, sl, r, tmax)) == 0ull;
        if (tie || !sound) {
            // As trace_exact, with a node's children or a leaf's records at once.
            const float band = 1000.f * distance_band(bvh, r, sh);
            float far = fminf(fmaf(tmax, 1.f + 1e-3f, band), r.tmax), near = fmaf(tmax, 1.f - 1e-3f, -band);
            bool first = sound;
            for (;;) {
                if (!first) {
                    tmax = INFINITY;
                    far = r.tmax;
                    near = -INFINITY;
                }
                found = false;
                if (lane == 0u) stack[0] = make_uint2(0u, 0u);
                for (sp = 1u; sp > 0u && !(first && found);) {
                    wave_fence();
                    const uint32_t ref = stack[--sp].x;
                    wave_fence();
                    if (is_inner(ref)) {
                        float tf;
                        uint32_t child;
                        float key = built_child(bvh, sl, ref, sub, r.tmin, far, child, tf);
                        if (tf < near) child = kEmptyChild;
                        float k[4];
                        uint32_t v[4];
#pragma unroll
                        for (uint32_t c = 0; c < 4u; c++) {
                            k[c] = __shfl(key, int(base + quad + c), 64);
                            v[c] = uint32_t(__shfl(int(child), int(base + quad + c), 64));
                        }
                        sort4(k, v);
#pragma unroll
                        for (int c = 3; c >= 0; c--) {
                            if (!(k[c] < INFINITY) || v[c] == kEmptyChild) continue;
                            if (lane == 0u) stack[sp] = make_uint2(v[c], 0u);
                            sp++;
                        }
                    } else {
                        const uint32_t tri = (ref & kMaxLeafFirst) + lane;
                        float at = INFINITY;
                        if (lane <= ((ref >> 27) & 0xfu)) {
                            const float4* tp = reinterpret_cast<const float4*>(bvh.tris + tri);
                            const float4 v0 = tp[0], v1 = tp[1], v2 = tp[2];
                            float t, U, V, W, det, tn;
                            if (watertight(sh, v0, v1, v2, r.tmin, far, t, U, V, W, det) && t < r.tmax) {
                                (void)in_leaf_box(bvh.tris[tri], v1.w, v2.w, sl, r.tmin, r.tmax, tn);
                                at = hit_order(t, tn);
                            }
                        }
                        float best = at;
#pragma unroll
                        for (int off = kLanes / 2; off > 0; off >>= 1) best = fminf(best, __shfl_xor(best, off, 64));
                        if (first ? ballot(at == tmax) != 0ull : best < tmax) {
                            if (!first) {
                                tmax = best;
                                far = fminf(widened(best, kOrderPrune), r.tmax);
                            }
                            found = true;
                            // Of equal ones the first record, the lowest lane's.
                            holders = ballot(at == tmax);
                            if (at == tmax) h.rec = tri;
                        }
                    }
                }
                if (found || !first) break;
                first = false;
            }
        }
        const bool lead = found ? lane == uint32_t(__ffsll(static_cast<long long>(holders)) - 1) : lane == 0u;
        if (lead) sink(i, found, h, r);
    }
}

// Scenes of at most kBruteMaxTris triangles skip the BVH: every lane tests every triangle
// record, in the same order, so the records are read at wave-uniform addresses and no lane
// idles in a divergent descent -- the loop of the reference's NaiveScene
// (scene.naive.cpp:31-124) with the watertight test.  A box room of a few dozen triangles
// costs a BVH descent through overlapping wall boxes that several times this loop costs.
// Every triangle against the BVH today, us: 1M closest hits (FP64) 42 triangles of the room 68 and
// 99, 90 113 and 103, soups of 60 84 and 106, 90 116 and 123, 128 157 and 149; any hits 42 60 and
// 55, soups of 36 52 and 58, 60 79 and 79, 128 159 and 111; 65,549 closest hits 42 19 and 34,
// 128 43 and 60.  Batches of up to 8192 rays are faster through trace_grouped at any size (81 rays:
// 36 triangles 13 and 8, 128 40 and 9), but a scene takes one way for all its batches: the two tests
// round differently, and a ray's result must not depend on its batch.  Renders of 256 x 256 x 16:
// pt 42 335 and 738, 138 511 and 698, 186 616 and 765; pt.direct 810 and 1520, 1226 and 1472, 1470
// and 1571.  The lines are those drawn on the descent of 128-byte nodes, where pt.direct crossed at
// 130 triangles and closest hits at 140; on today's closest hits cross at 75 to 110, any hits at 40
// to 60 and pt.direct beyond 186.
constexpr uint32_t kBruteMaxTris = 128;    // ray batches, pt.direct / pt.mis
constexpr uint32_t kBruteMaxTrisPt = 192;  // pt (and the LDS copy of the records)

// One ray per thread over grid-strided chunks of the batch; `active` lanes past the end test
// nothing.  Any hit stops once every active lane of the wave has a hit.
template <bool kAny, class Source, class Sink>
__device__ __forceinline__ void trace_brute(const TriRecord* __restrict__ tris, uint32_t ntris, uint32_t n,
                                            Source& src, Sink& sink) {
    const uint32_t waves = gridDim.x * (blockDim.x >> 6);
    if (n <= waves) {
        // At most one ray per wave (a late bounce, a small batch): the lanes share the ray and
        // split the triangles, so the ray costs one pass over ceil(ntris / 64) records instead
        // of a lane's walk over all of them.  The nearest hit (the lowest record among equal
        // distances, as in the lane-per-ray loop below) or, for any hit, the lowest lane with a
        // hit reports the ray.
        const uint32_t w = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
        if (w >= n) return;  // wave-uniform
        const uint32_t lane = __lane_id();
        const RayIn r = src(w);
        const ShearRows sh = make_shear_rows(r, make_shear(r));
        float tmax = r.tmax;
        HitOut h{tmax, 0u, 0xffffffffu, 0.f, 0.f, 1.f};
        bool found = false;
        for (uint32_t j = lane; j < ntris; j += 64u) {
            const float4* tp = reinterpret_cast<const float4*>(tris + j);
            const float4 v0 = tp[0], v1 = tp[1], v2 = tp[2];
            float t, U, V, W, det;
            if (!(kAny && found) && watertight_rows(sh, v0, v1, v2, r.tmin, tmax, t, U, V, W, det) && t < tmax) {
                found = true;
                tmax = t;
                accept_hit<kAny>(h, t, j, __float_as_uint(v0.w), V, W, det);
            }
        }
        const unsigned long long hits = __ballot(found);
        if (hits == 0ull) {
            if (lane == 0u) sink(w, false, h, r);
            return;
        }
        int winner = __ffsll(static_cast<long long>(hits)) - 1;
        if (!kAny) {
            // Lane L tested records L, L + 64, ...; its h.rec is the first of its records at its
            // nearest distance, so the minimum of (t, rec) over the lanes is the record the
            // lane-per-ray loop keeps (it replaces a hit only by a strictly nearer one).
            float best = found ? h.t : __builtin_inff();
            for (int off = 32; off > 0; off >>= 1) best = fminf(best, __shfl_xor(best, off, 64));
            uint32_t rec = found && h.t == best ? h.rec : 0xffffffffu;
            for (int off = 32; off > 0; off >>= 1) rec = min(rec, uint32_t(__shfl_xor(int(rec), off, 64)));
            winner = __ffsll(static_cast<long long>(__ballot(found && h.t == best && h.rec == rec))) - 1;
        }
        if (int(lane) == winner) {
            if (!kAny) hit_weights(h);
            sink(w, true, h, r);
        }
        return;
    }
    for (uint32_t base = blockIdx.x * blockDim.x; base < n; base += gridDim.x * blockDim.x) {
        const uint32_t i = base + threadIdx.x;
        const bool active = i < n;
        const RayIn r = active ? src(i) : RayIn{0.f, 0.f, 0.f, 0.f, 0.f, 1.f, 0.f, 0.f};
        const ShearRows sh = make_shear_rows(r, make_shear(r));
        float tmax = r.tmax;
        HitOut h{tmax, 0u, 0xffffffffu, 0.f, 0.f, 1.f};
        bool found = false;
        for (uint32_t j = 0; j < ntris; j++) {
            const float4* tp = reinterpret_cast<const float4*>(tris + j);
            const float4 v0 = tp[0], v1 = tp[1], v2 = tp[2];
            float t, U, V, W, det;
            if (active && !(kAny && found) && watertight_rows(sh, v0, v1, v2, r.tmin, tmax, t, U, V, W, det) && t < tmax) {
                found = true;
                tmax = t;
                accept_hit<kAny>(h, t, j, __float_as_uint(v0.w), V, W, det);
            }
            if (kAny && __ballot(active && !found) == 0ull) break;
        }
        if (!kAny && found) hit_weights(h);
        if (active) sink(i, found, h, r);
    }
}

// ---- Transform-record tests (XformRecord, bvh_build.h) of the tiny-scene path tracer ----
// The ray meets the triangle's plane where r2 . (o + t d) + r2.w = 0, i.e. at
// t = -(r2 . o + r2.w) / (r2 . d); the point's (r0, r1) coordinates are the weights u, v of v1
// and v2, and the hit counts when t lies strictly inside (tmin, tmax) and u, v >= 0,
// u + v <= 1.  About 20 VALU instructions per triangle against some 55 of the watertight
// test, for scenes whose rays test every triangle.  Like the reference's own tests
// (Moeller-Trumbore in its QBVH, TriAccel in its BVH) it is not watertight: a ray through a
// shared edge can pass both triangles, about as often as the edge's FP32 rounding decides.
__device__ __forceinline__ bool xform_test(const XformRecord& x, const RayIn& r, float tmax, float& t, float& u,
                                           float& v) {
    const float4 r0 = *reinterpret_cast<const float4*>(x.r0);
    const float4 r1 = *reinterpret_cast<const float4*>(x.r1);
    const float4 r2 = *reinterpret_cast<const float4*>(x.r2);
    const float dz = fmaf(r2.z, r.dz, fmaf(r2.y, r.dy, r2.x * r.dx));
    const float oz = fmaf(r2.z, r.oz, fmaf(r2.y, r.oy, fmaf(r2.x, r.ox, r2.w)));
    t = -oz * __builtin_amdgcn_rcpf(dz);
    const float px = fmaf(t, r.dx, r.ox), py = fmaf(t, r.dy, r.oy), pz = fmaf(t, r.dz, r.oz);
    u = fmaf(r0.z, pz, fmaf(r0.y, py, fmaf(r0.x, px, r0.w)));
    v = fmaf(r1.z, pz, fmaf(r1.y, py, fmaf(r1.x, px, r1.w)));
    return t > r.tmin && t < tmax && u >= 0.f && v >= 0.f && u + v <= 1.f;
}

// Closest hit over every record: (t, u, v, id bits), id 0xffffffff for a miss; a hit replaces
// another only when strictly nearer, so the lowest record wins a tie.  With group > 1 the
// group's lanes (consecutive, a power of two dividing 64, all holding the same ray) split the
// records and reduce to the same hit.  Every lane of the wave calls it (uniform trip count).
__device__ __forceinline__ float4 xform_closest(const XformRecord* __restrict__ xf, uint32_t n, const RayIn& r,
                                                bool active, uint32_t group = 1u, uint32_t sub = 0u) {
    float tmax = r.tmax, bu = 0.f, bv = 0.f;
    uint32_t rec = 0xffffffffu, id = 0xffffffffu;
    if (group == 1u) {
        // Every lane walks every record, four per iteration so that the tests' dependency
        // chains interleave; each replaces the result so far only when strictly nearer, in
        // record order, as one record at a time would.
        uint32_t j = 0;
        for (; j + 3u < n; j += 4u) {
            float t4[4], u4[4], v4[4];
            bool h4[4];
#pragma unroll
            for (int q = 0; q < 4; q++) h4[q] = xform_test(xf[j + q], r, tmax, t4[q], u4[q], v4[q]);
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (h4[q] && t4[q] < tmax) {
                    tmax = t4[q];
                    bu = u4[q];
                    bv = v4[q];
                    rec = j + q;
                }
        }
        for (; j < n; j++) {
            float t, u, v;
            if (xform_test(xf[j], r, tmax, t, u, v)) {
                tmax = t;
                bu = u;
                bv = v;
                rec = j;
            }
        }
        if (!active || rec == 0xffffffffu) return make_float4(0.f, 0.f, 0.f, __uint_as_float(0xffffffffu));
        return make_float4(tmax, bu, bv, __uint_as_float(xf[rec].id));
    }
    for (uint32_t j0 = 0; j0 < n; j0 += group) {
        const uint32_t j = j0 + sub;
        if (!active || j >= n) continue;
        float t, u, v;
        if (xform_test(xf[j], r, tmax, t, u, v)) {
            tmax = t;
            bu = u;
            bv = v;
            rec = j;
            id = xf[j].id;
        }
    }
    const bool found = rec != 0xffffffffu;
    if (group == 1u)
        return found ? make_float4(tmax, bu, bv, __uint_as_float(id)) : make_float4(0.f, 0.f, 0.f, __uint_as_float(id));
    float best = found ? tmax : __builtin_inff();
    for (uint32_t off = group >> 1; off > 0; off >>= 1) best = fminf(best, __shfl_xor(best, int(off), 64));
    uint32_t low = found && tmax == best ? rec : 0xffffffffu;
    for (uint32_t off = group >> 1; off > 0; off >>= 1) low = min(low, uint32_t(__shfl_xor(int(low), int(off), 64)));
    const uint32_t lane = __lane_id();
    const uint32_t base = lane & ~(group - 1u);
    const unsigned long long gmask = group >= 64u ? ~0ull : ((1ull << group) - 1ull);
    const unsigned long long win = (__ballot(found && tmax == best && rec == low) >> base) & gmask;
    const int src = win ? int(base) + __ffsll(static_cast<long long>(win)) - 1 : int(lane);
    const float4 out = make_float4(__shfl(tmax, src, 64), __shfl(bu, src, 64), __shfl(bv, src, 64),
                                   __uint_as_float(uint32_t(__shfl(int(id), src, 64))));
    return win ? out : make_float4(0.f, 0.f, 0.f, __uint_as_float(0xffffffffu));
}

// Whether any record blocks the ray; the wave stops once every active lane (with group > 1:
// every active group) has a hit.
__device__ __forceinline__ bool xform_any(const XformRecord* __restrict__ xf, uint32_t n, const RayIn& r, bool active,
                                          uint32_t group = 1u, uint32_t sub = 0u) {
    if (group == 1u) {
        // Four records per iteration (independent chains), until every active lane has a hit.
        bool found = false;
        for (uint32_t j = 0; j < n; j += 4u) {
            float t, u, v;
#pragma unroll
            for (uint32_t q = 0; q < 4u; q++)
                if (j + q < n && xform_test(xf[j + q], r, r.tmax, t, u, v)) found = true;
            if (__ballot(active && !found) == 0ull) break;
        }
        return active && found;
    }
    const uint32_t base = __lane_id() & ~(group - 1u);
    const unsigned long long gmask = group >= 64u ? ~0ull : ((1ull << group) - 1ull);
    bool found = false, group_found = false;
    for (uint32_t j0 = 0; j0 < n; j0 += group) {
        const uint32_t j = j0 + sub;
        if (active && !group_found && j < n) {
            float t, u, v;
            if (xform_test(xf[j], r, r.tmax, t, u, v)) found = true;
        }
        group_found = group == 1u ? found : ((__ballot(found) >> base) & gmask) != 0ull;
        if (__ballot(active && !group_found) == 0ull) break;
    }
    return active && group_found;
}

// Barycentrics of the recorded winner (weights of v1 and v2): the FP32 weights kept at
// acceptance, or the winner re-evaluated in FP64.
template <class Tri>
__device__ __forceinline__ void winner_barycentrics(const Tri* __restrict__ tris, const RayIn& r,
                                                    const HitOut& h, bool fp64, float& t, float& b0, float& b1) {
    t = h.t;
    b0 = h.b0;
    b1 = h.b1;
    if (fp64) {
        const float4* tp = reinterpret_cast<const float4*>(tris + h.rec);
        refine_fp64(r, tp[0], tp[1], tp[2], t, b0, b1);
    }
}

}  // namespace lmgpu
