// Wavefront path tracer: the reference's per-sample loops restated as stage kernels
// over structure-of-arrays path queues in HBM.
//
//   gen     -- camera vertex of every path of a batch        (pathtrace.cpp:167-192,
//              pathtrace.direct.cpp:172-303 for the camera vertex of pt.direct / pt.mis)
//   extend  -- closest-hit traversal of the live queue        (Scene::Intersect, scene.cpp:67-72)
//   shade   -- emission, NEE, Russian roulette, BSDF sampling (pathtrace.cpp:203-262,
//              pathtrace.direct.cpp:188-336, pathtrace.mis.cpp:185-367); live paths are
//              compacted into the next queue with one atomic per block
//   shadow  -- any-hit traversal of the NEE queue, then the film update
//              (RenderUtils::Visible, renderutils.cpp:58-70)
//   resolve -- film sums * W*H/N into the caller's film        (sched.mt.cpp:250-256)
//
// Scene-dependent forms of the same stages: on a BVH of 4 MB or more the camera stage hands
// out path slots in screen-tile order (k_tile_keys + a radix sort); in a scene of at most
// kBruteMaxTris triangles the shade kernels trace their own segment's rays over every
// triangle's transform record (xform_closest; no extend launch), and the render shadow-tests
// its connections where it makes them (xform_any; no shadow launch).  The next-event renderers add the camera vertex's light
// connections to film replicas (splat_add) that are folded into the film at the end.
//
// Each path sample owns a Philox4x32-10 stream keyed by (seed, global sample index) and
// draws from it in exactly the order the reference estimator calls Sampler::Next(), so
// the GPU traces the same path as the CPU restatement for the same sample index.
//
// The same stage kernels, instantiated per mode, also run the adjoint (path replay, no
// counterpart in the reference): for a loss L(I) of the rendered film I and its gradient
// g = dL/dI, every path sample is traced twice more from its own stream.
//   kAdjTotal -- Q_s = sum over the sample's contributions v (film pixel p) of g[p] * v,
//                per colour channel, into a per-sample FP64 slot;
//   kAdjGrad  -- the replay subtracts each contribution from Q_s as it is made, so at a
//                surface vertex Q_s holds exactly the contributions made after it, each of
//                which carries the vertex's reflectance R once as a factor (BSDF weight,
//                or the BSDF value of the vertex's own next-event connection).  Hence
//                dL/dR[m] += Q_s / R[m] at every vertex of material m, and
//                dL/dLe[l] += g[p] * v / Le[l] for every contribution lit by light l.
// Russian-roulette probabilities are held constant (the estimator stays unbiased for any
// probability), MIS weights and all sampling pdfs do not depend on R or Le, so the
// replay is exact for the path it retraces.  Gradients are scattered with FP64 atomics.
#include "context.hpp"
#include "traverse.hpp"

#include <algorithm>
#include <type_traits>
#include <cmath>
#include <chrono>

// Path state arithmetic of this file is not contracted into FMAs, so the render and both
// adjoint passes (different instantiations) compute bit-identical paths.
#pragma clang fp contract(off)

namespace lmgpu {

enum PTMode : int { kRender = 0, kAdjTotal = 1, kAdjGrad = 2 };

constexpr int kPTBlock = 256;
constexpr uint32_t kMiss = 0xffffffffu;
constexpr uint32_t kBlackMat = 0xffffffffu;  // the black diffuse BSDF of the environment sphere
constexpr uint32_t kFlagDegenerate = 1u;     // previous vertex is the pinhole camera
constexpr uint32_t kFlagSpecular = 2u;       // previous BSDF sample was specular
constexpr uint32_t kFlagLit = 4u;            // pt render: the path has gathered light (aux)

// GeneralizedBSDFType bits (include/lightmetrica/generalizedbsdf.h:34-72)
constexpr int kDiffuseReflection = 1 << 0;
constexpr int kSpecularReflection = 1 << 2;

struct PTConsts {
    BvhDev bvh;
    const XformRecord* xform;  // scenes of at most kBruteMaxTrisPt triangles: the records' transforms
    const ShadeTri* shade;
    const MaterialDev* mats;
    const LightDev* lights;
    const LightTri* light_tris;
    uint32_t num_lights;
    CameraDev cam;
    EnvDev env;
    void* film;
    int film_mode;       // LMGPU_FILM_*
    float* film_comp;    // FP32_COMPENSATED: the rounding-error sums beside the FP32 sums
    const float* dLdI;   // adjoint: dL/dI, W*H*3
    double* qacc;        // adjoint: per batch sample, 4 doubles (Q.xyz)
    double* grad_mat;    // adjoint: num_materials * 3
    double* grad_light;  // adjoint: num_lights * 3
    float4* record;      // pt render: per batch sample (radiance, pixel bits), or nullptr
    void* splat;         // NEE render: splat_k film replicas of splat_vals values (FP32 for the FP32 film, else FP64)
    int conn_lds;        // NEE render: the camera vertex's connections go through k_conn_reduce (their rectangle
                         // fits the kernel's LDS), written per shadow slot as (rgb with Le, pixel bits)
    uint32_t splat_k;
    size_t splat_vals;
    uint32_t splat_x0, splat_y0, splat_w, splat_h;  // the film rectangle the replicas cover
    const uint32_t* order;  // pt: batch sample of each camera-stage thread (screen-tile order), or nullptr
    uint32_t ntris;         // triangle records (the shading kernels trace their own rays up to kBruteMaxTrisPt)
    uint64_t seed;
    uint64_t base;  // global index of the batch's first sample
    uint32_t batch;  // samples in this batch
    int max_pv;
    int rr_depth;
    int renderer;
};

// Path queue: structure of arrays of 16-byte records.  The shading stages are bound by their traffic,
// so a vertex moves 48 bytes in and 48 out beside its hit, and `aux` only where it holds something:
// with five full records each the shading of a training step (59M vertices, twice) took 4.29 ms, now
// 4.09, the camera stage 0.80 -> 0.57, the whole step 16.8 -> 15.9 ms.  A segment's rays have one tmin, which the host passes.
struct Queue {
    float4* ray_o;  // o.xyz, throughput x
    float4* ray_d;  // d.xyz, throughput y
    uint4* meta;    // sample index in batch, path_bits, pixel, throughput z
    float4* aux;    // pt render: L.xyz of a path that has kFlagLit;  pt.mis: shading normal of the ray
                    // origin, pdf of the BSDF sample that produced the ray
};

// Vertex count n <= kMaxSegments, flags and stream dimension (at most a dozen numbers a vertex).
__device__ __forceinline__ uint32_t path_bits(uint32_t n, uint32_t flags, uint32_t dim) {
    return n | flags << 8 | dim << 16;
}

struct ShadowQueue {
    float4* o;      // origin, tmax
    float4* d;      // direction, pixel (bits)
    float4* c;      // contribution without the light's Le, light index (bits)
    uint32_t* sid;  // sample index in the batch
    uint32_t* vis;  // adjoint passes: 1 = unoccluded
};

struct PTBuffers {
    Queue q[2];
    uint32_t* hits;  // records of the segment's hits
    ShadowQueue sq;
    uint32_t* counters;  // [0, 64): live-queue sizes per segment, [64, 128): shadow sizes per segment,
                         // [128, 192): work counters of the extension launches, [192, 257): of the shadow launches
    unsigned long long* totals;  // closest rays, shadow rays
};

// Segment launches per batch at most: counters of 4 * kMaxSegments words fill the 2 KB
// counter block of the path buffers.
constexpr int kMaxSegments = 128;

// max_path_vertices = -1 (pathtrace.cpp:126) leaves the path length to Russian roulette,
// which keeps a path with probability min(0.5, Luminance(T)) <= 1/2 at every vertex from
// rr_depth on (pathtrace.cpp:250-260).  The render stops a path after kRouletteTail such
// vertices, where it survives with probability <= 2^-kRouletteTail: 2^-60 of the 2.1G
// samples of a 4K x 256 spp render is 2e-9 paths.
constexpr int kRouletteTail = 60;

// ---------------------------------------------------------------------------------

// Block-aggregated queue append: one atomic per block of kPTBlock threads instead of one
// per wavefront (same-address atomics serialise in L2).  Every thread of the block must call
// it -- it synchronises the block -- and each call site of a kernel needs its own kSite.
template <int kSite>
__device__ __forceinline__ uint32_t block_append(uint32_t* counter, bool pred) {
    __shared__ uint32_t wave_off[kPTBlock / 64];
    __shared__ uint32_t base;
    const unsigned long long mask = __ballot(pred);
    const uint32_t lane = __lane_id(), wave = threadIdx.x >> 6;
    if (lane == 0) wave_off[wave] = uint32_t(__popcll(mask));
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int w = 0; w < kPTBlock / 64; w++) {
            const uint32_t c = wave_off[w];
            wave_off[w] = t;
            t += c;
        }
        base = t ? atomicAdd(counter, t) : 0u;
    }
    __syncthreads();
    return base + wave_off[wave] + uint32_t(__popcll(mask & ((1ull << lane) - 1ull)));
}

// The rounding error of the FP32 sum old + x.
__device__ __forceinline__ float two_sum_error(float old, float x) {
    const float s = old + x;  // the value the atomic stored (round to nearest even)
    const float bp = s - old;
    return (old - (s - bp)) + (x - bp);
}

// Compensated FP32 accumulation: the atomic returns the sum it replaced, so the rounding
// error of the stored sum is recovered exactly by TwoSum (Knuth, TAOCP vol. 2, 4.2.2) and
// accumulated in a second FP32 array; the film value is sum + error.
__device__ __forceinline__ void comp_add(float* sum, float* err, float x) {
    if (x == 0.f) return;
    const float e = two_sum_error(unsafeAtomicAdd(sum, x), x);
    if (e != 0.f) unsafeAtomicAdd(err, e);
}

__device__ __forceinline__ void film_add(const PTConsts& c, uint32_t pixel, V3 v) {
    if (v.x == 0.f && v.y == 0.f && v.z == 0.f) return;
    if (c.film_mode == LMGPU_FILM_FP64) {
        double* f = static_cast<double*>(c.film) + 3ull * pixel;
        unsafeAtomicAdd(f + 0, double(v.x));
        unsafeAtomicAdd(f + 1, double(v.y));
        unsafeAtomicAdd(f + 2, double(v.z));
    } else if (c.film_mode == LMGPU_FILM_FP32_COMPENSATED) {
        float* f = static_cast<float*>(c.film) + 3ull * pixel;
        float* e = c.film_comp + 3ull * pixel;
        comp_add(f + 0, e + 0, v.x);
        comp_add(f + 1, e + 1, v.y);
        comp_add(f + 2, e + 2, v.z);
    } else {
        float* f = static_cast<float*>(c.film) + 3ull * pixel;
        unsafeAtomicAdd(f + 0, v.x);
        unsafeAtomicAdd(f + 1, v.y);
        unsafeAtomicAdd(f + 2, v.z);
    }
}

// The camera vertex's light connections (pt.direct / pt.mis) all land on the pixels that
// show the lights, so their film atomics pile onto a few cache lines and serialise there.
// Block b adds them to replica b mod splat_k (a multiple of the 8 XCDs when at least 8, so
// each replica is written from one XCD) of the film rectangle that the lights project to,
// and k_resolve adds the replicas to the film's values after the last batch.  A pixel outside
// the rectangle (never, up to rounding) goes to the film directly.
__device__ __forceinline__ void splat_add(const PTConsts& c, uint32_t pixel, V3 v) {
    if (v.x == 0.f && v.y == 0.f && v.z == 0.f) return;
    const uint32_t w = uint32_t(c.cam.width);
    const uint32_t x = pixel % w - c.splat_x0, y = pixel / w - c.splat_y0;  // wraps below the rectangle
    if (x >= c.splat_w || y >= c.splat_h) {
        film_add(c, pixel, v);
        return;
    }
    const size_t off = size_t(blockIdx.x % c.splat_k) * c.splat_vals + 3ull * (y * c.splat_w + x);
    if (c.film_mode == LMGPU_FILM_FP32) {
        float* f = static_cast<float*>(c.splat) + off;
        unsafeAtomicAdd(f + 0, v.x);
        unsafeAtomicAdd(f + 1, v.y);
        unsafeAtomicAdd(f + 2, v.z);
    } else {
        double* f = static_cast<double*>(c.splat) + off;
        unsafeAtomicAdd(f + 0, double(v.x));
        unsafeAtomicAdd(f + 1, double(v.y));
        unsafeAtomicAdd(f + 2, double(v.z));
    }
}

// Sample records.  pt: one float4 per sample, (radiance, pixel bits), written when the path
// ends.  pt.direct / pt.mis: two float4 per sample, (sum of contributions, pixel bits) for at
// most two pixels -- the path's own pixel, set by the camera stage, and the pixel of the
// camera vertex's light connection -- which are all the pixels a sample of these estimators
// touches.  A sample's contributions come one per launch, so the updates need no atomics.
constexpr uint32_t kNoPixel = 0xffffffffu;

__device__ __forceinline__ void record_add(const PTConsts& c, uint32_t sid, uint32_t pixel, V3 v) {
    if (v.x == 0.f && v.y == 0.f && v.z == 0.f) return;
    float4* r = c.record + 2ull * sid;
    float4 a = r[0];
    if (__float_as_uint(a.w) != pixel) {
        r += 1;
        a = r[0];
    }
    r[0] = make_float4(a.x + v.x, a.y + v.y, a.z + v.z, __uint_as_float(pixel));
}

// One contribution v of batch sample `sid` to film pixel `pixel`: the film in the render,
// +/- g[pixel] * v into the sample's Q in the adjoint passes.  Per launch a sample makes at
// most one call, so the read-modify-write of its Q slot needs no atomics.
template <int kMode>
__device__ __forceinline__ void contribute(const PTConsts& c, uint32_t sid, uint32_t pixel, V3 v) {
    if (kMode == kRender) {
        film_add(c, pixel, v);
        if (c.record) record_add(c, sid, pixel, v);
        return;
    }
    if (is_zero(v)) return;
    const float* g = c.dLdI + 3ull * pixel;
    double* q = c.qacc + 4ull * sid;
    const double x = double(g[0]) * double(v.x), y = double(g[1]) * double(v.y), z = double(g[2]) * double(v.z);
    if (kMode == kAdjTotal) {
        q[0] += x;
        q[1] += y;
        q[2] += z;
    } else {
        q[0] -= x;
        q[1] -= y;
        q[2] -= z;
    }
}

// Gradient accumulation of one block: an open-addressing hash table in LDS keyed by
// material id, or by kLightKey | light id, holding FP64 sums.  Paths of a block share
// few hot parameters (walls, lights), so the table turns most device-scope FP64 atomics
// into LDS atomics; each block adds its table to the gradient once, at its end.  A key
// that finds no slot within kGradProbes goes straight to the device atomics.
constexpr int kGradSlots = 512;
constexpr int kGradProbes = 8;
constexpr uint32_t kEmptyKey = 0xffffffffu;
constexpr uint32_t kLightKey = 0x80000000u;

struct GradCache {
    uint32_t keys[kGradSlots];
    double vals[3 * kGradSlots];
};

__device__ __forceinline__ double* grad_target(const PTConsts& c, uint32_t key) {
    return (key & kLightKey) ? c.grad_light + 3ull * (key & ~kLightKey) : c.grad_mat + 3ull * key;
}

__device__ __forceinline__ void gc_init(GradCache& g) {
    for (int i = threadIdx.x; i < kGradSlots; i += blockDim.x) {
        g.keys[i] = kEmptyKey;
        g.vals[3 * i] = g.vals[3 * i + 1] = g.vals[3 * i + 2] = 0.0;
    }
    __syncthreads();
}

// Adds to the sums of `key`; false if there is no slot for it.
__device__ __forceinline__ bool gc_put(GradCache& g, uint32_t key, double x, double y, double z) {
    uint32_t slot = (key * 2654435761u) >> 23;  // 9 bits: kGradSlots = 512
    for (int probe = 0; probe < kGradProbes; probe++) {
        uint32_t k = __hip_atomic_load(&g.keys[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (k == kEmptyKey) {
            const uint32_t prev = atomicCAS(&g.keys[slot], kEmptyKey, key);
            k = prev == kEmptyKey ? key : prev;
        }
        if (k == key) {
            atomicAdd(&g.vals[3 * slot + 0], x);
            atomicAdd(&g.vals[3 * slot + 1], y);
            atomicAdd(&g.vals[3 * slot + 2], z);
            return true;
        }
        slot = (slot + 1) & (kGradSlots - 1);
    }
    return false;
}

__device__ __forceinline__ void gc_add(GradCache& g, const PTConsts& c, uint32_t key, double x, double y, double z) {
    if (x == 0.0 && y == 0.0 && z == 0.0) return;
    if (gc_put(g, key, x, y, z)) return;
    double* d = grad_target(c, key);
    if (x != 0.0) unsafeAtomicAdd(d + 0, x);
    if (y != 0.0) unsafeAtomicAdd(d + 1, y);
    if (z != 0.0) unsafeAtomicAdd(d + 2, z);
}

__device__ __forceinline__ void gc_flush(GradCache& g, const PTConsts& c) {
    __syncthreads();
    for (int i = threadIdx.x; i < kGradSlots; i += blockDim.x) {
        const uint32_t key = g.keys[i];
        if (key == kEmptyKey) continue;
        double* d = grad_target(c, key);
        for (int k = 0; k < 3; k++)
            if (g.vals[3 * i + k] != 0.0) unsafeAtomicAdd(d + k, g.vals[3 * i + k]);
    }
}

// The same table over the pixels on which a tile of paths ends (keys: pixel indices), added to an
// FP64 or compensated film once per tile and emptied.  Paths in screen-tile order end four to a
// pixel and tile, and the film's atomics, six a path where it is compensated, took longer than all
// the rest of the shading: 1920 x 1080 x 8 of the terrain 2.90 -> 1.22 ms compensated, 2.04 ->
// 1.07 FP64 (0.81 without a film).  An FP32 film keeps its sums' order, and its atomics.
__device__ __forceinline__ void film_flush(GradCache& g, const PTConsts& c) {
    constexpr int kEach = 3 * kGradSlots / kPTBlock;
    static_assert(kEach * kPTBlock == 3 * kGradSlots, "a thread flushes kEach values");
    __syncthreads();
    double x[kEach];
    uint32_t pixel[kEach];
    auto channel = [](int j) { return uint32_t(j * kPTBlock + int(threadIdx.x)) % 3u; };
#pragma unroll
    for (int j = 0; j < kEach; j++) {
        const int i = j * kPTBlock + int(threadIdx.x);
        pixel[j] = g.keys[i / 3];
        x[j] = 0.0;
        if (pixel[j] == kEmptyKey) continue;
        x[j] = g.vals[i];
        g.vals[i] = 0.0;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kGradSlots; i += kPTBlock) g.keys[i] = kEmptyKey;
    if (c.film_mode == LMGPU_FILM_FP64) {
#pragma unroll
        for (int j = 0; j < kEach; j++)
            if (x[j] != 0.0) unsafeAtomicAdd(static_cast<double*>(c.film) + 3ull * pixel[j] + channel(j), x[j]);
    } else {
        // comp_add, with all the sums' old values under way before the first is needed.
        float old[kEach];
#pragma unroll
        for (int j = 0; j < kEach; j++)
            if (x[j] != 0.0) old[j] = unsafeAtomicAdd(static_cast<float*>(c.film) + 3ull * pixel[j] + channel(j), float(x[j]));
#pragma unroll
        for (int j = 0; j < kEach; j++) {
            if (x[j] == 0.0) continue;
            const float v = float(x[j]);
            const float e = two_sum_error(old[j], v) + float(x[j] - double(v));
            if (e != 0.f) unsafeAtomicAdd(c.film_comp + 3ull * pixel[j] + channel(j), e);
        }
    }
    __syncthreads();
}

// dL/dLe of a contribution v = w * Le (w: the contribution without Le) of light `li`.
__device__ __forceinline__ void grad_emission(GradCache& g, const PTConsts& c, uint32_t pixel, V3 w, int li) {
    const float* dl = c.dLdI + 3ull * pixel;
    gc_add(g, c, kLightKey | uint32_t(li), double(dl[0]) * double(w.x), double(dl[1]) * double(w.y),
           double(dl[2]) * double(w.z));
}

// HDRBitmapFilm pixel of a raster position (hdrfilm.cpp:160-166); y = 0 is the bottom row.
__device__ __forceinline__ uint32_t pixel_of(const CameraDev& cam, float rx, float ry) {
    const int px = min(max(int(rx * float(cam.width)), 0), cam.width - 1);
    const int py = min(max(int(ry * float(cam.height)), 0), cam.height - 1);
    return uint32_t(py) * uint32_t(cam.width) + uint32_t(px);
}

// PerspectiveCamera::EvaluateImportance (perspectivecamera.cpp:325-353)
__device__ __forceinline__ float cam_importance(const CameraDev& cam, float cos_theta) {
    if (cos_theta <= 0.f) return 0.f;
    if (fabsf(cos_theta - 1.f) < kEpsLarge) cos_theta = 1.f;
    const float ic = 1.f / cos_theta;
    return cam.inv_A * ic * ic * ic;
}

// PerspectiveCamera::SampleAndEstimateDirection (perspectivecamera.cpp:216-240): direction
// for a raster position; `pdf` is the importance in the projected-solid-angle measure.
__device__ __forceinline__ V3 cam_direction(const CameraDev& cam, float u0, float u1, float& pdf) {
    float d4[4];
    mul4(cam.inv_proj, u0 * 2.f - 1.f, u1 * 2.f - 1.f, 0.f, 1.f, d4);
    const V3 d3 = normalize(v3(d4[0] / d4[3], d4[1] / d4[3], d4[2] / d4[3]));
    float w4[4];
    mul4(cam.inv_view, d3.x, d3.y, d3.z, 0.f, w4);
    pdf = cam_importance(cam, -d3.z);
    return normalize(v3(w4[0], w4[1], w4[2]));
}

// PerspectiveCamera::RayToRasterPosition (perspectivecamera.cpp:304-323)
__device__ __forceinline__ bool cam_ray_to_raster(const CameraDev& cam, V3 p, V3 d, float& rx, float& ry) {
    float c4[4], n4[4];
    mul4(cam.view, p.x + d.x, p.y + d.y, p.z + d.z, 1.f, c4);
    mul4(cam.proj, c4[0], c4[1], c4[2], c4[3], n4);
    rx = (n4[0] / n4[3] + 1.f) / 2.f;
    ry = (n4[1] / n4[3] + 1.f) / 2.f;
    return !(rx < 0.f || rx > 1.f || ry < 0.f || ry > 1.f);
}

// PerspectiveCamera::EvaluateDirection / EvaluateDirectionPDF (perspectivecamera.cpp:276-302, :355-383)
__device__ __forceinline__ float cam_eval_direction(const CameraDev& cam, V3 p, V3 wo) {
    float c4[4], n4[4];
    mul4(cam.view, p.x + wo.x, p.y + wo.y, p.z + wo.z, 1.f, c4);
    mul4(cam.proj, c4[0], c4[1], c4[2], c4[3], n4);
    const float rx = (n4[0] / n4[3] + 1.f) / 2.f, ry = (n4[1] / n4[3] + 1.f) / 2.f;
    if (rx < 0.f || rx > 1.f || ry < 0.f || ry > 1.f) return 0.f;
    return cam_importance(cam, -normalize(v3(c4[0], c4[1], c4[2])).z);
}

// ---------------------------------------------------------------------------------
// Surfaces

struct Surf {
    V3 p, gn;
    Frame f;
    uint32_t mat;
    int32_t light;
};

// Scene::StoreIntersectionFromBarycentricCoords (scene.cpp:101-149) for a triangle hit,
// or the environment sphere when the triangles are missed (emittershape.sphere.cpp:117-176).
__device__ __forceinline__ bool surface_at(const PTConsts& c, V3 o, V3 d, float tmin, float4 hit, Surf& s) {
    const uint32_t prim = __float_as_uint(hit.w);
    if (prim != kMiss) {
        const float4* sp = reinterpret_cast<const float4*>(c.shade + prim);
        const float4 a = sp[0], b = sp[1], e = sp[2], g = sp[3];
        const float t = hit.x, b0 = hit.y, b1 = hit.z;
        s.p = o + d * t;
        s.gn = v3(a.x, a.y, a.z);
        s.mat = __float_as_uint(a.w);
        s.light = __float_as_int(b.w);
        const float w0 = 1.f - b0 - b1;
        const V3 n = v3(b.x, b.y, b.z) * w0 + v3(e.x, e.y, e.z) * b0 + v3(g.x, g.y, g.z) * b1;
        s.f.build(normalize(n));
        return true;
    }
    if (c.env.index < 0) return false;
    const V3 ctr = v3(c.env.center[0], c.env.center[1], c.env.center[2]);
    const V3 oc = o - ctr;
    const float A = dot(d, d), B = 2.f * dot(oc, d), C = dot(oc, oc) - c.env.radius * c.env.radius;
    const float det = B * B - 4.f * A * C;
    if (det < 0.f) return false;
    const float e = sqrtf(det), den = 2.f * A;
    const float t0 = (-B - e) / den, t1 = (-B + e) / den;
    if (t0 > kInf || t1 < tmin) return false;
    float t = t0;
    if (t < tmin) {
        t = t1;
        if (t > kInf) return false;
    }
    s.p = o + d * t;
    const V3 n = normalize(ctr - s.p);
    s.gn = n;
    s.f.build(n);
    s.mat = kBlackMat;
    s.light = c.env.index;
    return true;
}

// BSDF::ShadingNormalCorrectionFactor for EL transport (bsdf.h:57-83): 1 or 0.
__device__ __forceinline__ bool sides_agree(V3 gn, V3 wi, V3 wo, float lwi_z, float lwo_z) {
    return !(dot(wi, gn) * lwi_z <= 0.f || dot(wo, gn) * lwo_z <= 0.f);
}

struct MatInfo {
    uint32_t type;
    V3 R;
};
__device__ __forceinline__ MatInfo mat_info(const PTConsts& c, uint32_t m) {
    if (m == kBlackMat) return MatInfo{LMGPU_BSDF_DIFFUSE, v3s(0.f)};
    const float4 x = reinterpret_cast<const float4*>(c.mats)[m];
    return MatInfo{__float_as_uint(x.x), v3(x.y, x.z, x.w)};
}

// SampleAndEstimateDirection (EL): diffuse.cpp:133-157, mirror.cpp:84-107,
// diffusemirror.cpp:84-125.  Returns the estimate f/p; zero means the path ends.
__device__ __forceinline__ V3 bsdf_sample(const MatInfo& m, const Surf& s, V3 wi, float u0, float u1, float uc,
                                          V3& wo, float& pdf, int& type) {
    const V3 lwi = s.f.to_local(wi);
    if (lwi.z <= 0.f) return v3s(0.f);
    V3 lwo;
    V3 est;
    if (m.type == LMGPU_BSDF_DIFFUSE || (m.type == LMGPU_BSDF_DIFFUSEMIRROR && uc < 0.5f)) {
        lwo = cosine_hemisphere(u0, u1);
        type = kDiffuseReflection;
        pdf = m.type == LMGPU_BSDF_DIFFUSE ? kInvPi : kInvPi * 0.5f;
        est = m.type == LMGPU_BSDF_DIFFUSE ? m.R : m.R * 0.5f / 0.5f;
    } else {
        lwo = v3(-lwi.x, -lwi.y, lwi.z);  // ReflectZUp (math.vector.inl:532-536)
        type = kSpecularReflection;
        pdf = m.type == LMGPU_BSDF_MIRROR ? 1.f / lwo.z : 0.5f / fabsf(lwi.z);
        est = m.type == LMGPU_BSDF_MIRROR ? m.R : m.R * 0.5f / 0.5f;
    }
    wo = s.f.to_world(lwo);
    if (!sides_agree(s.gn, wi, wo, lwi.z, lwo.z)) return v3s(0.f);
    return est;
}

// EvaluateDirection / EvaluateDirectionPDF with type NonDelta (diffuse.cpp:192-220,
// mirror.cpp:141-215 -> 0, diffusemirror.cpp:188-274).
__device__ __forceinline__ V3 bsdf_eval_nondelta(const MatInfo& m, const Surf& s, V3 wi, V3 wo, float& pdf) {
    pdf = 0.f;
    if (m.type == LMGPU_BSDF_MIRROR) return v3s(0.f);
    const V3 lwi = s.f.to_local(wi), lwo = s.f.to_local(wo);
    if (lwi.z <= 0.f || lwo.z <= 0.f) return v3s(0.f);
    pdf = m.type == LMGPU_BSDF_DIFFUSE ? kInvPi : kInvPi * 0.5f;
    if (!sides_agree(s.gn, wi, wo, lwi.z, lwo.z)) return v3s(0.f);
    return m.type == LMGPU_BSDF_DIFFUSE ? m.R * kInvPi : m.R * kInvPi * 0.5f;
}

__device__ __forceinline__ bool mat_nondelta(const MatInfo& m) { return m.type != LMGPU_BSDF_MIRROR; }

// Emission toward -d at a surface: EvaluateDirection * EvaluatePosition = (1/pi) * (Le pi)
// on the front side (light.area.cpp:233-252, light.env.const.cpp:174-209).
__device__ __forceinline__ V3 light_Le(const PTConsts& c, int li) {
    const float4 x = reinterpret_cast<const float4*>(c.lights)[2 * li];
    return v3(x.y, x.z, x.w);
}

// ---------------------------------------------------------------------------------
// Next-event estimation at a vertex (pathtrace.direct.cpp:197-248, pathtrace.mis.cpp:194-262).

struct NEEVertex {
    V3 p;
    Surf s;           // valid when !camera
    bool camera;      // the pinhole camera vertex (degenerated, no cosine)
    MatInfo m;
    V3 wi;
};

struct ShadowRec {
    bool emit;
    float4 o, d, c;
};

// Returns the shadow-ray record of the connection: its contribution without the light's Le
// and the light index.  emit = false when the contribution is 0 (in the adjoint passes:
// when it is 0 whatever Le is); the caller appends emitted records to the shadow queue.
__device__ __forceinline__ ShadowRec nee(const PTConsts& c, const NEEVertex& v, V3 T, int n, uint32_t pixel,
                                         SampleStream& rng, bool mis, bool active, bool adjoint) {
    V3 contrib = v3s(0.f);
    V3 Le = v3s(0.f);
    int li = 0;
    V3 target = v.p;
    uint32_t pix = pixel;
    if (active) {
        // Scene::SampleLightSelection (scene.cpp:79-86)
        float lu0 = rng.next(), lu1 = rng.next();
        const int nl = int(c.num_lights);
        li = min(int(lu0 * float(nl)), nl - 1);
        lu0 = lu0 * float(nl) - float(li);
        const float sel_pdf = 1.f / float(nl);
        const float4 L0 = reinterpret_cast<const float4*>(c.lights)[2 * li];
        const float4 L1 = reinterpret_cast<const float4*>(c.lights)[2 * li + 1];
        const uint32_t ltype = __float_as_uint(L0.x);
        Le = v3(L0.y, L0.z, L0.w);
        V3 lp, ln;
        float pdf_pl;
        if (ltype == LMGPU_LIGHT_ENV_CONST) {  // light.env.const.cpp:196-204
            const V3 dir = uniform_sphere(lu0, lu1);
            lp = v3(c.env.center[0], c.env.center[1], c.env.center[2]) + dir * c.env.radius;
            ln = -dir;
            pdf_pl = c.env.inv_area;
        } else {  // light.area.cpp:146-179
            const uint32_t tb = __float_as_uint(L1.x), tc = __float_as_uint(L1.y);
            pdf_pl = L1.z;
            // upper_bound over the cumulative area fractions
            uint32_t lo = 0, hi = tc;
            while (lo < hi) {
                const uint32_t mid = (lo + hi) >> 1;
                if (c.light_tris[tb + mid].p2[3] <= lu1) lo = mid + 1;
                else hi = mid;
            }
            const uint32_t k = min(lo, tc - 1);
            const LightTri lt = c.light_tris[tb + k];
            const float ylo = lt.p1[3], yhi = lt.p2[3];
            const float y = (lu1 - ylo) / (yhi - ylo);
            float b0, b1;
            uniform_triangle(lu0, y, b0, b1);
            const V3 p1 = v3(lt.p1[0], lt.p1[1], lt.p1[2]), p2 = v3(lt.p2[0], lt.p2[1], lt.p2[2]),
                     p3 = v3(lt.p3[0], lt.p3[1], lt.p3[2]);
            lp = p1 * (1.f - b0 - b1) + p2 * b0 + p3 * b1;
            ln = normalize(cross(p2 - p1, p3 - p1));
        }
        pdf_pl *= sel_pdf;
        const V3 ppl = normalize(lp - v.p);
        bool vis = true;
        if (n == 1) {
            float rx, ry;
            vis = cam_ray_to_raster(c.cam, v.p, ppl, rx, ry);
            pix = pixel_of(c.cam, rx, ry);
        }
        if (vis) {
            V3 fsE;
            float pdf_bsdf;
            if (v.camera) {
                const float w = cam_eval_direction(c.cam, v.p, ppl);
                fsE = v3s(w);
                pdf_bsdf = w;
            } else {
                fsE = bsdf_eval_nondelta(v.m, v.s, v.wi, ppl, pdf_bsdf);
            }
            // Light frame: shading normal = geometric normal (light.area.cpp:170-172).
            const float fsL = dot(ln, -ppl) <= 0.f ? 0.f : kInvPi;
            // RenderUtils::GeneralizedGeometryTerm (renderutils.cpp:29-56)
            V3 dv = lp - v.p;
            const float l2 = dot(dv, dv);
            const float l = sqrtf(l2);
            dv = dv / l;
            float num = 1.f;
            if (!v.camera) num *= fabsf(dot(v.s.f.sn, dv));
            num *= fabsf(dot(ln, -dv));
            const float G = fabsf(l) < kEps ? 0.f : num / l2;
            // T fsE G fsL LeP / pdf with LeP = Le pi; Le is applied where the ray is resolved.
            if (!mis) {
                contrib = T * fsE * G * fsL * kPi / pdf_pl;
            } else if (G != 0.f) {
                const float pdf_dl = pdf_pl / G;
                const float w = pdf_dl / (pdf_dl + pdf_bsdf);
                contrib = T * w * fsE * G * fsL * kPi / pdf_pl;
            }
            target = lp;
        }
    }
    ShadowRec rec;
    rec.emit = active && !is_zero(contrib) && (adjoint || !is_zero(Le));
    if (rec.emit) {
        // RenderUtils::Visible: d = (p2 - p1) / |p2 - p1|, (Eps, |p2 - p1| (1 - Eps))
        const V3 dv = target - v.p;
        const float len = length(dv);
        const V3 d = dv / len;
        rec.o = make_float4(v.p.x, v.p.y, v.p.z, len * (1.f - kEps));
        rec.d = make_float4(d.x, d.y, d.z, __uint_as_float(pix));
        rec.c = make_float4(contrib.x, contrib.y, contrib.z, __int_as_float(li));
    }
    return rec;
}

__device__ __forceinline__ void put_shadow(const ShadowQueue& sq, uint32_t slot, const ShadowRec& r, uint32_t sid) {
    sq.o[slot] = r.o;
    sq.d[slot] = r.d;
    sq.c[slot] = r.c;
    sq.sid[slot] = sid;
}

// Render of a scene of at most kBruteMaxTris triangles: the connection's shadow ray is traced
// at once (any hit over every triangle record) and its unoccluded contribution added, as
// ShadowSink does for a queued ray; kSplat: the camera vertex's connections (splat_add).
// Every lane calls shadow_visible: the triangle loop is wave-uniform.
// With group > 1 the group's lanes (all holding the same record) split the triangle loop.
__device__ __forceinline__ bool shadow_visible(const PTConsts& c, const XformRecord* xf, const ShadowRec& rec,
                                               uint32_t group = 1u, uint32_t sub = 0u) {
    const RayIn r{rec.o.x, rec.o.y, rec.o.z, rec.d.x, rec.d.y, rec.d.z, kEps, rec.o.w};
    return rec.emit && !xform_any(xf, c.ntris, r, rec.emit, group, sub);
}

template <bool kSplat>
__device__ __forceinline__ void add_connection(const PTConsts& c, const ShadowRec& rec, uint32_t sid) {
    const V3 Le = light_Le(c, __float_as_int(rec.c.w));
    const uint32_t pixel = __float_as_uint(rec.d.w);
    const V3 x = v3(rec.c.x, rec.c.y, rec.c.z) * Le;
    if (kSplat) splat_add(c, pixel, x);
    else film_add(c, pixel, x);
    if (c.record) record_add(c, sid, pixel, x);
}

// The camera vertex's connection of shadow slot `slot` when c.conn_lds: its contribution (Le
// applied) and pixel, or no pixel when occluded, into the slot's record for k_conn_reduce; the
// sample record (c.record) is updated at once.
__device__ __forceinline__ void stage_connection(const PTConsts& c, const ShadowQueue& sq, uint32_t slot,
                                                 const ShadowRec& rec, bool lit, uint32_t sid) {
    if (!lit) {
        sq.c[slot] = make_float4(0.f, 0.f, 0.f, __uint_as_float(kNoPixel));
        return;
    }
    const V3 Le = light_Le(c, __float_as_int(rec.c.w));
    const uint32_t pixel = __float_as_uint(rec.d.w);
    const V3 x = v3(rec.c.x, rec.c.y, rec.c.z) * Le;
    sq.c[slot] = make_float4(x.x, x.y, x.z, __uint_as_float(pixel));
    if (c.record) record_add(c, sid, pixel, x);
}

// ---------------------------------------------------------------------------------
// Kernels

// The triangle records of a scene of at most kMax triangles (kBruteMaxTrisPt for pt,
// kBruteMaxTris for pt.direct / pt.mis) copied into the block's LDS, for the kernels that test
// every record per ray (kFuse): the loops then read them at LDS latency.  Every thread of the
// block must call it (it synchronises the block).
template <uint32_t kMax>
__device__ __forceinline__ const XformRecord* stage_xform(const PTConsts& c, XformRecord* lds) {
    const uint32_t n = min(c.ntris, kMax);
    for (uint32_t k = threadIdx.x; k < n; k += blockDim.x) lds[k] = c.xform[k];
    __syncthreads();
    return lds;
}

__device__ __forceinline__ void store_path(const Queue& q, uint32_t slot, V3 o, V3 d, V3 T, uint32_t sid, uint32_t bits,
                                           uint32_t pixel) {
    q.ray_o[slot] = make_float4(o.x, o.y, o.z, T.x);
    q.ray_d[slot] = make_float4(d.x, d.y, d.z, T.y);
    q.meta[slot] = make_uint4(sid, bits, pixel, __float_as_uint(T.z));
}

// Interleaves the bits of x and y (each < 2^16): the Z-order (Morton) index of (x, y).
__device__ __forceinline__ uint32_t morton2(uint32_t x, uint32_t y) {
    auto spread = [](uint32_t v) {
        v = (v | (v << 8)) & 0x00ff00ffu;
        v = (v | (v << 4)) & 0x0f0f0f0fu;
        v = (v | (v << 2)) & 0x33333333u;
        v = (v | (v << 1)) & 0x55555555u;
        return v;
    };
    return spread(x) | (spread(y) << 1);
}

// Sort keys of the camera stage on large scenes: the Z-order index of the 8x8-pixel tile
// that each batch sample's raster position falls in -- numbers `skip` and skip + 1 of its
// stream: 0 for pt (pathtrace.cpp:167-173); for pt.direct / pt.mis the camera position, the
// light selection and sample of the camera vertex's connection and, when rr_depth <= 1, the
// roulette come first (pathtrace.direct.cpp:175-262).  Tracing the camera rays tile by tile
// lets a wave's lanes share BVH nodes in the caches; the samples and their streams are
// unchanged.
__global__ void k_tile_keys(PTConsts c, int skip, uint32_t* __restrict__ keys, uint32_t* __restrict__ vals) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= c.batch) return;
    SampleStream rng;
    rng.init(c.seed, c.base + i, 0);
    for (int k = 0; k < skip; k++) rng.next();
    const float r0 = rng.next(), r1 = rng.next();
    const uint32_t p = pixel_of(c.cam, r0, r1), w = uint32_t(c.cam.width);
    keys[i] = morton2((p % w) >> 3, (p / w) >> 3);
    vals[i] = i;
}

// Camera vertex.  pt: pathtrace.cpp:167-192.  pt.direct / pt.mis: the first loop
// iteration of pathtrace.direct.cpp:172-303 (NEE from the camera, RR, camera sampling).
// kFuse (render of a scene of at most kBruteMaxTris triangles): the camera vertex's
// connection is shadow-tested here (shadow_visible) instead of queued, and added after the
// sample's record is set up.
template <int kMode, bool kFuse = false>
__global__ __launch_bounds__(kPTBlock) void k_gen(PTConsts c, Queue out, uint32_t* live_count, ShadowQueue sq,
                                                  uint32_t* shadow_count) {
    // Only the next-event renderers trace here (the camera vertex's connection).
    __shared__ XformRecord xf_lds[kFuse ? kBruteMaxTris : 1];
    const XformRecord* xf = kFuse && c.renderer != LMGPU_PT ? stage_xform<kBruteMaxTris>(c, xf_lds) : c.xform;
    const uint32_t slot0 = blockIdx.x * kPTBlock + threadIdx.x;
    const bool valid = slot0 < c.batch;
    const uint32_t i = c.order && valid ? c.order[slot0] : slot0;  // the batch sample of this thread
    SampleStream rng;
    rng.init(c.seed, c.base + i, 0);
    const V3 cam_p = v3(c.cam.pos[0], c.cam.pos[1], c.cam.pos[2]);
    const bool start = !(c.max_pv != -1 && 1 >= c.max_pv);
    if (c.renderer == LMGPU_PT) {
        // Every path of pt survives its camera vertex: slot = thread, no compaction.
        if (!valid) return;
        if (!start) {  // max_path_vertices = 1: no segment, the sample contributes nothing
            if (kMode == kRender && c.record) c.record[i] = make_float4(0.f, 0.f, 0.f, __uint_as_float(kNoPixel));
            return;
        }
        if (slot0 == 0) *live_count = c.batch;
        const float r0 = rng.next(), r1 = rng.next();
        rng.next();  // Camera::SamplePosition draws a Vec2 (pathtrace.cpp:173)
        rng.next();
        float pdf;
        const V3 d = cam_direction(c.cam, r0, r1, pdf);
        const uint32_t pixel = pixel_of(c.cam, r0, r1);
        // The path's record is written where it ends.
        store_path(out, slot0, cam_p, d, v3s(1.f), i, path_bits(1u, 0u, rng.dim), pixel);
        return;
    }
    const bool mis = c.renderer == LMGPU_PT_MIS;
    rng.next();  // Camera::SamplePosition (pathtrace.direct.cpp:175)
    rng.next();
    V3 T = v3s(1.f);
    bool alive = valid && start;
    NEEVertex v;
    v.p = cam_p;
    v.camera = true;
    v.wi = v3s(0.f);
    const ShadowRec rec = nee(c, v, T, 1, 0u, rng, mis, alive, kMode != kRender);
    bool lit = false;  // kFuse: the connection is unoccluded; added once the record is set up
    uint32_t cslot = 0;  // kFuse: its shadow slot
    if constexpr (kMode == kRender && kFuse) {
        cslot = block_append<0>(shadow_count, rec.emit);  // counts the shadow rays traced
        lit = shadow_visible(c, xf, rec);
    } else {
        const uint32_t sslot = block_append<0>(shadow_count, rec.emit);
        if (rec.emit) put_shadow(sq, sslot, rec, i);
    }
    if (alive && c.rr_depth != -1 && 1 >= c.rr_depth) {
        const float q = fminf(0.5f, luminance(T));
        if (rng.next() > q) alive = false;
        else T = T / q;
    }
    V3 d = v3s(0.f);
    float pdf = 0.f;
    uint32_t pixel = 0;
    if (alive) {
        const float u0 = rng.next(), u1 = rng.next();
        rng.next();  // uComp
        d = cam_direction(c.cam, u0, u1, pdf);
        float rx, ry;
        if (!cam_ray_to_raster(c.cam, cam_p, d, rx, ry)) alive = false;
        pixel = pixel_of(c.cam, rx, ry);
    }
    const uint32_t slot = block_append<1>(live_count, alive);
    if (alive) {
        store_path(out, slot, cam_p, d, T, i, path_bits(1u, kFlagDegenerate, rng.dim), pixel);
        if (mis) out.aux[slot] = make_float4(0.f, 0.f, 0.f, pdf);
    }
    if (kMode == kRender && c.record && valid) {
        c.record[2ull * i] = make_float4(0.f, 0.f, 0.f, __uint_as_float(alive ? pixel : kNoPixel));
        c.record[2ull * i + 1] = make_float4(0.f, 0.f, 0.f, __uint_as_float(kNoPixel));
    }
    if (kMode == kRender && kFuse) {
        if (c.conn_lds) {
            if (rec.emit) stage_connection(c, sq, cslot, rec, lit, i);
        } else if (lit) {
            add_connection<true>(c, rec, i);
        }
    }
}

// Extension rays: closest hit of every live path (persistent, refilling lanes).
struct QueueSource {
    Queue q;
    float tmin;
    __device__ __forceinline__ RayIn operator()(uint32_t i) const {
        const float4 o = q.ray_o[i], d = q.ray_d[i];
        return RayIn{o.x, o.y, o.z, d.x, d.y, d.z, tmin, kInf};
    }
};

// A segment's hits: the winner's record (kMiss for none), a word per path.  The shading stages repeat
// its test (hit_of), which gives the traversal's t and weights: a training step's extension rays
// 10.52 -> 10.15 ms without the four-word results and their registers, its shading 4.10 -> 4.18.
struct HitSink {
    uint32_t* recs;
    __device__ __forceinline__ void operator()(uint32_t i, bool found, const HitOut& h, const RayIn&) const {
        recs[i] = found ? h.rec : kMiss;
    }
};

// (t, b0, b1, triangle bits) of record `rec` along r.
__device__ __forceinline__ float4 hit_of(const LeafTri* tris, uint32_t rec, const RayIn& r) {
    if (rec == kMiss) return make_float4(0.f, 0.f, 0.f, __uint_as_float(kMiss));
    const HitOut h = hit_at(tris, rec, r);
    return make_float4(h.t, h.b0, h.b1, __uint_as_float(h.prim));
}

// The LDS of a stage that traces a queue, whatever the number of rays makes of it: late bounces
// hold few rays, which several lanes follow each (trace_grouped).
template <bool kKeys> union QueueShared {
    TraceShared<kKeys> lane;
    GroupShared<64> group64;
    GroupShared<16> group16;
    __device__ QueueShared() {}
};

// The traversal counters of a wave added to counts[0] (node visits) and counts[1] (triangle
// tests), one atomic per wave each (the counting forms of the extension and shadow stages).
__device__ __forceinline__ void add_wave_counts(const TraceCounters& cnt, unsigned long long* counts) {
    unsigned long long a = cnt.nodes, b = cnt.tris;
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_down(a, off, 64);
        b += __shfl_down(b, off, 64);
    }
    if (__lane_id() == 0) {
        atomicAdd(&counts[0], a);
        atomicAdd(&counts[1], b);
    }
}

// kCount (lmgpu_enable_counting): also counts node visits and triangle tests into `counts`.
// 6 waves per SIMD, as the LDS stack allows (the bound keeps the kernel within 80 VGPRs).
template <bool kCount = false>
__global__ __launch_bounds__(kTraceBlock, 6) void k_extend(BvhDev bvh, Queue q, float tmin,
                                                        const uint32_t* __restrict__ count, uint32_t* next,
                                                        uint32_t* __restrict__ hits, unsigned long long* counts) {
    __shared__ QueueShared<true> sm;
    const uint32_t n = *count;
    QueueSource src{q, tmin};
    HitSink sink{hits};
    TraceCounters cnt{0, 0};
    if (n <= kGroup64Rays) trace_grouped<false, kCount, 64>(bvh, n, sm.group64, src, sink, cnt);
    else if (n <= kGroup16Closest) trace_grouped<false, kCount, 16>(bvh, n, sm.group16, src, sink, cnt);
    else trace_persistent<false, kCount>(bvh, n, next, sm.lane, src, sink, cnt);
    if (kCount) add_wave_counts(cnt, counts);
}

// dL/dR of the vertex's material: Q / R per channel (the contributions still in Q all carry
// R once).
__device__ __forceinline__ void grad_material(GradCache& g, const PTConsts& c, uint32_t sid, uint32_t mat, V3 R) {
    const double* q = c.qacc + 4ull * sid;
    gc_add(g, c, mat, R.x != 0.f ? q[0] / double(R.x) : 0.0, R.y != 0.f ? q[1] / double(R.y) : 0.0,
           R.z != 0.f ? q[2] / double(R.z) : 0.0);
}

// One vertex of pt (pathtrace.cpp:203-262) at the hit `hit` of the ray o + t d: the emission
// seen there, BSDF sampling and Russian roulette.  T and n are the path's throughput and
// vertex count, updated when the path goes on (`alive`, along the ray s.p + t wo).
struct PtVertex {
    Surf s;
    MatInfo m;
    bool emits;  // the hit is on the front of a light: emit = T * Le (T before the vertex)
    V3 emit, Le_w;  // the emission and the emission without Le
    V3 wo;
    float pdf;
    bool alive;
};

__device__ __forceinline__ PtVertex pt_vertex(const PTConsts& c, V3 o, V3 d, float tmin, float4 hit, bool valid, V3& T,
                                              int& n, SampleStream& rng) {
    PtVertex v;
    v.s.mat = kBlackMat;
    v.s.light = -1;
    v.m = MatInfo{LMGPU_BSDF_DIFFUSE, v3s(0.f)};
    v.emits = false;
    v.emit = v3s(0.f);
    v.Le_w = v3s(0.f);
    v.wo = v3s(0.f);
    v.pdf = 0.f;
    v.alive = false;
    if (valid && surface_at(c, o, d, tmin, hit, v.s)) {
        if (v.s.light >= 0 && dot(v.s.f.sn, -d) > 0.f) {
            v.emits = true;
            const V3 Le = light_Le(c, v.s.light);
            v.Le_w = T * v3s(kInvPi) * kPi;
            v.emit = T * v3s(kInvPi) * (Le * kPi);
        }
        const float u0 = rng.next(), u1 = rng.next(), uc = rng.next();
        int type;
        v.m = mat_info(c, v.s.mat);
        const V3 fs = bsdf_sample(v.m, v.s, -d, u0, u1, uc, v.wo, v.pdf, type);
        if (!is_zero(fs)) {
            T = T * fs;
            v.alive = true;
            if (c.rr_depth != -1 && n >= c.rr_depth) {
                const float q = fminf(0.5f, luminance(T));
                if (rng.next() > q) v.alive = false;
                else T = T / q;
            }
            n++;
            if (c.max_pv != -1 && n >= c.max_pv) v.alive = false;
        }
    }
    return v;
}

// Lanes per path of the shading kernels that trace their own rays (kFuse): a segment of
// `count` paths gives each path a group of G lanes -- the largest power of two up to
// kSplitMax with count * G <= kSplitLanes -- which split the triangle loop of its rays
// (xform_closest, xform_any with group > 1).  kSplitLanes is two wavefronts per SIMD of the
// 1024 SIMDs: segments with fewer lanes' worth of paths leave the SIMDs too few waves to hide
// latency, and each launch lasts about one ray's walk over every record.
constexpr uint32_t kSplitLanes = 1u << 17;
constexpr uint32_t kSplitMax = 16;
__device__ __forceinline__ uint32_t lanes_per_path(uint32_t count) {
    uint32_t g = 1u;
    while (g < kSplitMax && uint64_t(count) * uint64_t(2u * g) <= uint64_t(kSplitLanes)) g *= 2u;
    return g;
}

// pt: pathtrace.cpp:203-262 for one segment.
// The shade kernels walk the queue in tiles of kPTBlock paths, tile t by block t mod grid,
// over a device-filling grid (16 blocks per CU; 4 for the gradient pass, so that each
// block's gradient table collects many paths before it is flushed): a late segment's
// nearly empty queue then costs a launch of that grid, not of one block per queue slot.
// kTable: the film's sums go through film_flush.
template <int kMode, bool kFuse = false, bool kTable = false>
__global__ __launch_bounds__(kPTBlock) void k_shade_pt(PTConsts c, Queue in, float tmin, const uint32_t* __restrict__ in_count,
                                                       const uint32_t* __restrict__ hits, Queue out,
                                                       uint32_t* out_count) {
    const uint32_t count = *in_count;
    // kFuse: a segment of few paths gives each path a group of lanes (lanes_per_path).
    const uint32_t group = kFuse ? lanes_per_path(count) : 1u;
    const uint32_t per_tile = kPTBlock / group;  // paths per tile
    if (blockIdx.x * per_tile >= count) return;  // a block without paths (block-uniform)
    __shared__ XformRecord xf_lds[kFuse ? kBruteMaxTrisPt : 1];
    const XformRecord* xf = kFuse ? stage_xform<kBruteMaxTrisPt>(c, xf_lds) : c.xform;
    __shared__ GradCache gc;
    if (kMode == kAdjGrad || kTable) gc_init(gc);
    auto tile_body = [&](uint32_t tile) {
    const uint32_t i = tile * per_tile + threadIdx.x / group;
    const uint32_t sub = threadIdx.x & (group - 1u);
    const bool valid = i < count;
    const bool lead = sub == 0u;  // the lane of the group that applies the path's effects
    const uint32_t j = valid ? i : 0u;  // invalid lanes read slot 0 and discard it
    const float4 ro = in.ray_o[j], rd = in.ray_d[j];
    const uint4 meta = in.meta[j];
    const V3 o = v3(ro.x, ro.y, ro.z), d = v3(rd.x, rd.y, rd.z);
    V3 T = v3(ro.w, rd.w, __uint_as_float(meta.w)), L = v3s(0.f);
    int n = int(meta.y & 0xffu);
    if (kMode == kRender && (meta.y >> 8 & kFlagLit)) {
        const float4 ax = in.aux[j];
        L = v3(ax.x, ax.y, ax.z);
    }
    SampleStream rng;
    rng.init(c.seed, c.base + meta.x, meta.y >> 16);
    // kFuse (scenes of at most kBruteMaxTris triangles): the segment's ray is traced here
    // instead of by a separate extension launch.
    const RayIn ray{ro.x, ro.y, ro.z, rd.x, rd.y, rd.z, tmin, kInf};
    const float4 hit = kFuse ? xform_closest(xf, c.ntris, ray, valid, group, sub) : hit_of(c.bvh.tris, hits[j], ray);
    // Every lane of a group shades the same path the same way; the lead lane applies it.
    const PtVertex v = pt_vertex(c, o, d, tmin, hit, valid, T, n, rng);
    if (v.emits) {
        if (kMode == kRender) L = L + v.emit;
        else if (lead) contribute<kMode>(c, meta.x, meta.z, v.emit);
    }
    const bool alive = v.alive && lead;
    if (kMode == kAdjGrad && lead) {
        if (v.emits) grad_emission(gc, c, meta.z, v.Le_w, v.s.light);
        if (alive && v.s.mat != kBlackMat) grad_material(gc, c, meta.x, v.s.mat, v.m.R);
    }
    const uint32_t slot = block_append<0>(out_count, alive);
    if (alive) {
        const bool lit = kMode == kRender && (L.x != 0.f || L.y != 0.f || L.z != 0.f);
        store_path(out, slot, v.s.p, v.wo, T, meta.x, path_bits(uint32_t(n), lit ? kFlagLit : 0u, rng.dim), meta.z);
        if (lit) out.aux[slot] = make_float4(L.x, L.y, L.z, 0.f);
    } else if (kMode == kRender && valid && lead) {
        if (!kTable || is_zero(L) || !gc_put(gc, meta.z, L.x, L.y, L.z)) film_add(c, meta.z, L);
        if (c.record) c.record[meta.x] = make_float4(L.x, L.y, L.z, __uint_as_float(meta.z));
    }
    if (kTable) film_flush(gc, c);
    };
    for (uint32_t tile = blockIdx.x; tile * per_tile < count; tile += gridDim.x) tile_body(tile);
    if (kMode == kAdjGrad) gc_flush(gc, c);
}

// pt.direct / pt.mis: the hit half of one loop iteration (pathtrace.direct.cpp:304-336,
// pathtrace.mis.cpp:318-367) followed by the next iteration up to the next ray
// (NEE :197-248 / :194-262, RR, BSDF sampling).
// 5 waves per SIMD: the bound keeps the kernel within 96 VGPRs (it needed 97, i.e. 4 waves;
// the room's pt.direct / pt.mis renders 3 % faster).
template <int kMode, bool kFuse = false>
__global__ __launch_bounds__(kPTBlock, 5) void k_shade_nee(PTConsts c, Queue in, float tmin, const uint32_t* __restrict__ in_count,
                                                        const uint32_t* __restrict__ hits, Queue out,
                                                        uint32_t* out_count, ShadowQueue sq, uint32_t* shadow_count) {
    const uint32_t count = *in_count;
    // kFuse: a segment of few paths gives each path a group of lanes (lanes_per_path).
    const uint32_t group = kFuse ? lanes_per_path(count) : 1u;
    const uint32_t per_tile = kPTBlock / group;  // paths per tile
    if (blockIdx.x * per_tile >= count) return;  // a block without paths (block-uniform)
    __shared__ XformRecord xf_lds[kFuse ? kBruteMaxTris : 1];
    const XformRecord* xf = kFuse ? stage_xform<kBruteMaxTris>(c, xf_lds) : c.xform;
    __shared__ GradCache gc;
    if (kMode == kAdjGrad) gc_init(gc);
    auto tile_body = [&](uint32_t tile) {
    const uint32_t i = tile * per_tile + threadIdx.x / group;
    const uint32_t sub = threadIdx.x & (group - 1u);
    const bool valid = i < count;
    // Every lane of a group shades the same path the same way; the lead lane applies it.
    const bool lead = sub == 0u;
    const uint32_t j = valid ? i : 0u;  // invalid lanes read slot 0 and discard it
    const bool mis = c.renderer == LMGPU_PT_MIS;
    const float4 ro = in.ray_o[j], rd = in.ray_d[j];
    const uint4 meta = in.meta[j];
    const V3 o = v3(ro.x, ro.y, ro.z), d = v3(rd.x, rd.y, rd.z);
    V3 T = v3(ro.w, rd.w, __uint_as_float(meta.w));
    const uint32_t pixel = meta.z;
    int n = int(meta.y & 0xffu);
    const uint32_t flags = meta.y >> 8 & 0xffu;
    SampleStream rng;
    rng.init(c.seed, c.base + meta.x, meta.y >> 16);
    Surf s;
    s.mat = kBlackMat;
    s.light = -1;
    const RayIn ray{ro.x, ro.y, ro.z, rd.x, rd.y, rd.z, tmin, kInf};
    const float4 hit = kFuse ? xform_closest(xf, c.ntris, ray, valid, group, sub) : hit_of(c.bvh.tris, hits[j], ray);
    bool alive = valid && surface_at(c, o, d, tmin, hit, s);
    bool emits = false;
    V3 Le_w = v3s(0.f);
    if (alive && s.light >= 0) {
        const float LeD = dot(s.f.sn, -d) > 0.f ? kInvPi : 0.f;
        const V3 Le = light_Le(c, s.light);
        if (flags & kFlagSpecular) {
            emits = true;
            Le_w = T * v3s(LeD) * kPi;
        } else if (mis) {
            // GeneralizedGeometryTerm(previous vertex, hit) and the light-sampling pdf
            const float4 ax = in.aux[j];
            V3 dv = s.p - o;
            const float l2 = dot(dv, dv);
            const float l = sqrtf(l2);
            dv = dv / l;
            float num = 1.f;
            if (!(flags & kFlagDegenerate)) num *= fabsf(dot(v3(ax.x, ax.y, ax.z), dv));
            num *= fabsf(dot(s.f.sn, -dv));
            const float G = fabsf(l) < kEps ? 0.f : num / l2;
            const float pos_pdf = s.light == c.env.index ? c.env.inv_area
                                                         : reinterpret_cast<const float4*>(c.lights)[2 * s.light + 1].z;
            const float pdf_dl = G == 0.f ? 0.f : (1.f / float(c.num_lights)) * pos_pdf / G;
            const float w = ax.w / (ax.w + pdf_dl);
            emits = true;
            Le_w = T * v3s(LeD) * kPi * w;
        }
        if (emits && lead) contribute<kMode>(c, meta.x, pixel, Le_w * Le);
    }
    if (kMode == kAdjGrad && emits && lead) grad_emission(gc, c, pixel, Le_w, s.light);
    if (alive) {
        n++;
        if (c.max_pv != -1 && n >= c.max_pv) alive = false;
    }
    NEEVertex v;
    v.p = s.p;
    v.s = s;
    v.camera = false;
    v.wi = -d;
    v.m = alive ? mat_info(c, s.mat) : MatInfo{LMGPU_BSDF_MIRROR, v3s(0.f)};
    const ShadowRec rec = nee(c, v, T, n, pixel, rng, mis, alive && mat_nondelta(v.m), kMode != kRender);
    if constexpr (kMode == kRender && kFuse) {
        (void)block_append<0>(shadow_count, rec.emit && lead);  // counts the shadow rays traced
        if (shadow_visible(c, xf, rec, group, sub) && lead) add_connection<false>(c, rec, meta.x);
    } else {
        const uint32_t sslot = block_append<0>(shadow_count, rec.emit && lead);
        if (rec.emit && lead) put_shadow(sq, sslot, rec, meta.x);
    }
    if (alive && c.rr_depth != -1 && n >= c.rr_depth) {
        const float q = fminf(0.5f, luminance(T));
        if (rng.next() > q) alive = false;
        else T = T / q;
    }
    V3 wo = v3s(0.f);
    float pdf = 0.f;
    int type = 0;
    if (alive) {
        const float u0 = rng.next(), u1 = rng.next(), uc = rng.next();
        const V3 fs = bsdf_sample(v.m, s, -d, u0, u1, uc, wo, pdf, type);
        if (is_zero(fs)) alive = false;
        else T = T * fs;
    }
    if (kMode == kAdjGrad && lead && (rec.emit || alive) && s.mat != kBlackMat)
        grad_material(gc, c, meta.x, s.mat, v.m.R);
    alive = alive && lead;
    const uint32_t slot = block_append<1>(out_count, alive);
    if (alive) {
        const uint32_t bits = path_bits(uint32_t(n), (type & (1 << 2)) ? kFlagSpecular : 0u, rng.dim);
        store_path(out, slot, s.p, wo, T, meta.x, bits, pixel);
        if (mis) out.aux[slot] = make_float4(s.f.sn.x, s.f.sn.y, s.f.sn.z, pdf);
    }
    };
    for (uint32_t tile = blockIdx.x; tile * per_tile < count; tile += gridDim.x) tile_body(tile);
    if (kMode == kAdjGrad) gc_flush(gc, c);
}

// NEE shadow rays: any hit over the triangles.  The render adds the unoccluded
// contributions to the film right away; the adjoint passes record visibility and apply
// it in k_shadow_apply, where the wavefront is converged for the gradient scatter.
struct ShadowSource {
    ShadowQueue sq;
    __device__ __forceinline__ RayIn operator()(uint32_t i) const {
        const float4 o = sq.o[i], d = sq.d[i];
        return RayIn{o.x, o.y, o.z, d.x, d.y, d.z, kEps, o.w};
    }
};

// kSplat: the camera vertex's connections, added to the film replicas (splat_add).
template <int kMode, bool kSplat>
struct ShadowSink {
    PTConsts c;
    ShadowQueue sq;
    __device__ __forceinline__ void operator()(uint32_t i, bool found, const HitOut&, const RayIn&) const {
        if (kMode != kRender) {
            sq.vis[i] = found ? 0u : 1u;
            return;
        }
        if (kSplat && c.conn_lds) {
            // the slot's record becomes the connection for k_conn_reduce
            const float4 v = sq.c[i];
            const V3 x = found ? v3s(0.f) : v3(v.x, v.y, v.z) * light_Le(c, __float_as_int(v.w));
            const uint32_t pixel = found ? kNoPixel : __float_as_uint(sq.d[i].w);
            sq.c[i] = make_float4(x.x, x.y, x.z, __uint_as_float(pixel));
            if (!found && c.record) record_add(c, sq.sid[i], pixel, x);
            return;
        }
        if (found) return;
        const float4 v = sq.c[i];
        const V3 Le = light_Le(c, __float_as_int(v.w));
        const uint32_t pixel = __float_as_uint(sq.d[i].w);
        const V3 x = v3(v.x, v.y, v.z) * Le;
        if (kSplat) splat_add(c, pixel, x);
        else film_add(c, pixel, x);
        if (c.record) record_add(c, sq.sid[i], pixel, x);
    }
};

// 7 waves per SIMD: the bound keeps the kernel within 72 VGPRs (its LDS allows 9).
template <int kMode, bool kSplat = false, bool kCount = false>
__global__ __launch_bounds__(kTraceBlock, 7) void k_shadow(PTConsts c, ShadowQueue sq, const uint32_t* __restrict__ count,
                                                        uint32_t* next, unsigned long long* counts) {
    __shared__ QueueShared<false> sm;
    const uint32_t n = *count;
    ShadowSource src{sq};
    ShadowSink<kMode, kSplat> sink{c, sq};
    TraceCounters cnt{0, 0};
    if (n <= kGroup64Rays) trace_grouped<true, kCount, 64>(c.bvh, n, sm.group64, src, sink, cnt);
    else if (n <= kGroup16Any) trace_grouped<true, kCount, 16>(c.bvh, n, sm.group16, src, sink, cnt);
    else trace_persistent<true, kCount>(c.bvh, n, next, sm.lane, src, sink, cnt);
    if (kCount) add_wave_counts(cnt, counts);
}

// Shadow rays of a scene of at most kBruteMaxTris triangles (the adjoint passes' queue): every
// triangle's transform record from the block's LDS, the same test as the render's
// shadow_visible; a launch of few rays splits each ray's records over a group of lanes.
template <int kMode, bool kSplat = false>
__global__ __launch_bounds__(kTraceBlock) void k_shadow_brute(PTConsts c, uint32_t ntris, ShadowQueue sq,
                                                              const uint32_t* __restrict__ count) {
    const uint32_t n = *count;
    const uint32_t group = lanes_per_path(n);
    const uint32_t per_block = kTraceBlock / group;  // rays per block and pass
    if (blockIdx.x * per_block >= n) return;  // block-uniform
    __shared__ XformRecord xf_lds[kBruteMaxTris];
    const XformRecord* xf = stage_xform<kBruteMaxTris>(c, xf_lds);
    ShadowSource src{sq};
    ShadowSink<kMode, kSplat> sink{c, sq};
    const uint32_t sub = threadIdx.x & (group - 1u);
    for (uint32_t base = blockIdx.x * per_block; base < n; base += gridDim.x * per_block) {
        const uint32_t i = base + threadIdx.x / group;
        const bool active = i < n;
        const RayIn r = src(active ? i : 0u);
        const bool found = xform_any(xf, ntris, r, active, group, sub);
        if (active && sub == 0u) sink(i, found, HitOut{}, r);
    }
}

// Adjoint passes: the unoccluded shadow contributions into Q, and dL/dLe.
template <int kMode>
__global__ __launch_bounds__(kPTBlock) void k_shadow_apply(PTConsts c, ShadowQueue sq,
                                                           const uint32_t* __restrict__ count) {
    __shared__ GradCache gc;
    if (kMode == kAdjGrad) gc_init(gc);
    const uint32_t n = *count;
    for (uint32_t i = blockIdx.x * kPTBlock + threadIdx.x; i < n; i += gridDim.x * kPTBlock) {
        if (sq.vis[i] == 0u) continue;
        const float4 cv = sq.c[i];
        const uint32_t pixel = __float_as_uint(sq.d[i].w);
        const int li = __float_as_int(cv.w);
        const V3 w = v3(cv.x, cv.y, cv.z);
        contribute<kMode>(c, sq.sid[i], pixel, w * light_Le(c, li));
        if (kMode == kAdjGrad) grad_emission(gc, c, pixel, w, li);
    }
    if (kMode == kAdjGrad) gc_flush(gc, c);
}

// The raycast renderer (RaycastRenderer_RenderProcess::ProcessSinglePixel,
// src/liblightmetrica/raycast.cpp:96-137, under the deterministic per-pixel scheduler,
// sched.pixel.cpp:79-126): the ray through each pixel centre, |sn . -d| on a hit --
// triangles first, then the environment sphere -- and black otherwise.  Every pixel is a
// function of its own ray only, so the image is bit-identical from run to run.
struct RaycastSource {
    CameraDev cam;
    __device__ __forceinline__ RayIn operator()(uint32_t i) const {
        const uint32_t x = i % uint32_t(cam.width), y = i / uint32_t(cam.width);
        float pdf;
        const V3 d = cam_direction(cam, (0.5f + float(x)) / float(cam.width), (0.5f + float(y)) / float(cam.height), pdf);
        return RayIn{cam.pos[0], cam.pos[1], cam.pos[2], d.x, d.y, d.z, 0.f, kInf};
    }
};

template <class Out>
struct RaycastSink {
    PTConsts c;
    Out* out;
    __device__ __forceinline__ void operator()(uint32_t i, bool found, const HitOut& h, const RayIn& r) const {
        const V3 o = v3(r.ox, r.oy, r.oz), d = v3(r.dx, r.dy, r.dz);
        const float4 hit = hit_of(c.bvh.tris, found ? h.rec : kMiss, r);
        Surf s;
        float v = 0.f;
        if (surface_at(c, o, d, 0.f, hit, s)) v = fabsf(dot(s.f.sn, -d));
        out[3ull * i + 0] = Out(v);
        out[3ull * i + 1] = Out(v);
        out[3ull * i + 2] = Out(v);
    }
};

template <class Out>
__global__ __launch_bounds__(kTraceBlock, 5) void k_raycast(PTConsts c, uint32_t n, uint32_t* next, Out* out) {
    __shared__ QueueShared<true> sm;
    RaycastSource src{c.cam};
    RaycastSink<Out> sink{c, out};
    TraceCounters cnt{0, 0};
    if (n <= kGroup64Rays) trace_grouped<false, false, 64>(c.bvh, n, sm.group64, src, sink, cnt);
    else if (n <= kGroup16Closest) trace_grouped<false, false, 16>(c.bvh, n, sm.group16, src, sink, cnt);
    else trace_persistent<false, false>(c.bvh, n, next, sm.lane, src, sink, cnt);
}

__global__ void k_zero_u32(uint32_t* p, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

__global__ void k_zero_bytes(uint4* p, size_t n16) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n16) p[i] = make_uint4(0u, 0u, 0u, 0u);
}

// What a render or an adjoint starts from: two accumulators and the path buffers' counters and
// totals, cleared in one launch.  Launches are what a small render waits for, some 5 us each: 64 x 64 x 8
// with 18 of them took 195 us, with 12 180.
__global__ void k_clear(uint4* a, size_t na, uint4* b, size_t nb, uint32_t* words, uint32_t nw) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < na) a[i] = make_uint4(0u, 0u, 0u, 0u);
    else if (i - na < nb) b[i - na] = make_uint4(0u, 0u, 0u, 0u);
    if (i < nw) words[i] = 0u;
}

// Adds a batch's queue sizes to the totals, by the first wave of a launch; `out` may be `totals`.
__device__ __forceinline__ void add_totals(const uint32_t* counters, int segments, const unsigned long long* totals,
                                           unsigned long long* out) {
    unsigned long long a = 0, b = 0;
    for (int k = int(threadIdx.x); k < segments; k += 64) {
        a += counters[k];
        b += counters[kMaxSegments + k];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_xor(a, off, 64);
        b += __shfl_xor(b, off, 64);
    }
    if (threadIdx.x == 0) {
        out[0] = totals[0] + a;
        out[1] = totals[1] + b;
    }
}

// After every batch but the last, whose counters the run's last kernel adds.
__global__ void k_accumulate_totals(const uint32_t* counters, int segments, unsigned long long* totals) {
    add_totals(counters, segments, totals, totals);
}

struct RunTotals {
    const uint32_t* counters;
    int segments;
    const unsigned long long* totals;
    unsigned long long* out;  // device or pinned host memory
};

// HDRBitmapFilm::Rescale after the master-film reduction (sched.mt.cpp:250-256): weight =
// Float(W*H) / Float(N), data *= weight, in the film's arithmetic type; the compensated FP32 film
// as (sum + error) * weight, evaluated in FP64 and rounded once.  kSplat: the replicas of splat_add
// are first added to the film's values in their rectangle; the compensated film takes sum + error
// + replicas in FP64, rounded to an FP32 pair.
template <class Acc, class Out, bool kComp, bool kSplat>
__global__ void k_resolve(PTConsts c, Out* __restrict__ out, size_t n, std::conditional_t<kComp, double, Acc> weight,
                          RunTotals run) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (blockIdx.x == 0 && threadIdx.x < 64) add_totals(run.counters, run.segments, run.totals, run.out);
    if (i >= n) return;
    using Rep = std::conditional_t<kComp, double, Acc>;  // the replicas' type
    Rep s = Rep(0);
    bool in = false;
    if constexpr (kSplat) {
        const uint32_t w = uint32_t(c.cam.width);
        const uint32_t pixel = uint32_t(i / 3), ch = uint32_t(i % 3);
        const uint32_t x = pixel % w - c.splat_x0, y = pixel / w - c.splat_y0;  // wraps below the rectangle
        in = x < c.splat_w && y < c.splat_h;
        if (in) {
            const Rep* r = static_cast<const Rep*>(c.splat) + 3ull * (y * c.splat_w + x) + ch;
#pragma unroll 8
            for (uint32_t k = 0; k < c.splat_k; k++) s += r[k * c.splat_vals];
        }
    }
    if constexpr (kComp) {
        const float f = static_cast<const float*>(c.film)[i], e = c.film_comp[i];
        double v = double(f) + double(e);
        if (in) {
            const double t = v + s;
            const float hi = float(t);
            v = double(hi) + double(float(t - double(hi)));
        }
        out[i] = Out(v * weight);
    } else {
        Acc v = static_cast<const Acc*>(c.film)[i];
        if (in) v += s;
        out[i] = Out(v * weight);
    }
}

// The camera vertex's connections of a batch (c.conn_lds; shadow slots [0, *count), each
// (rgb, pixel bits) or no pixel) summed per block in an LDS copy of the film rectangle the
// lights project to, then added to the block's film replica (block mod splat_k) with one
// atomic per touched value: instead of three device atomics per connection on the few
// hundred pixels that show the lights, where they serialise, about one per value per block.
// FP32 sums for the FP32 film, FP64 otherwise (the replicas' type).  A pixel outside the
// rectangle (never, up to rounding) goes to the film directly.
constexpr uint32_t kConnLdsBytes = 32768;
template <class Acc>
__global__ __launch_bounds__(kPTBlock) void k_conn_reduce(PTConsts c, const float4* __restrict__ conn,
                                                          const uint32_t* __restrict__ count) {
    __shared__ Acc acc[kConnLdsBytes / sizeof(Acc)];
    const uint32_t n = *count;
    const uint32_t vals = 3u * c.splat_w * c.splat_h;  // <= the LDS array (checked by the host)
    for (uint32_t k = threadIdx.x; k < vals; k += kPTBlock) acc[k] = Acc(0);
    __syncthreads();
    const uint32_t w = uint32_t(c.cam.width);
    for (uint32_t i = blockIdx.x * kPTBlock + threadIdx.x; i < n; i += gridDim.x * kPTBlock) {
        const float4 v = conn[i];
        const uint32_t pixel = __float_as_uint(v.w);
        if (pixel == kNoPixel) continue;
        const uint32_t x = pixel % w - c.splat_x0, y = pixel / w - c.splat_y0;  // wraps below the rectangle
        if (x >= c.splat_w || y >= c.splat_h) {
            film_add(c, pixel, v3(v.x, v.y, v.z));
            continue;
        }
        Acc* a = acc + 3u * (y * c.splat_w + x);
        if (v.x != 0.f) atomicAdd(a + 0, Acc(v.x));
        if (v.y != 0.f) atomicAdd(a + 1, Acc(v.y));
        if (v.z != 0.f) atomicAdd(a + 2, Acc(v.z));
    }
    __syncthreads();
    Acc* rep = static_cast<Acc*>(c.splat) + size_t(blockIdx.x % c.splat_k) * c.splat_vals;
    for (uint32_t k = threadIdx.x; k < vals; k += kPTBlock)
        if (acc[k] != Acc(0)) unsafeAtomicAdd(rep + k, acc[k]);
}

// *out += the sum of v over a block of 256 threads.
__device__ __forceinline__ void block_sum_to(double v, double* out) {
    __shared__ double part[256 / 64];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if (__lane_id() == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) unsafeAtomicAdd(out, part[0] + part[1] + part[2] + part[3]);
}

// sum over samples of |Q.x| + |Q.y| + |Q.z| (the replay check of the adjoint).
__global__ __launch_bounds__(256) void k_abs_sum(const double* __restrict__ q, uint32_t n, double* out) {
    double v = 0.0;
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
        v += fabs(q[4ull * i]) + fabs(q[4ull * i + 1]) + fabs(q[4ull * i + 2]);
    block_sum_to(v, out);
}

// Adjoint pass 1 from a sample record (`stride` float4 per sample):
// Q = sum over the record's pixels of dL/dI[pixel] * contribution.
// A pixel index outside the film (a record the render did not write) contributes nothing.
// *sum += its k_abs_sum (one atomic a block, of 4096 at most).
__global__ __launch_bounds__(256) void k_q_from_record(const float4* __restrict__ rec, uint32_t stride, const float* __restrict__ dLdI,
                                uint32_t npix, uint32_t n, double* __restrict__ q, double* sum) {
    double total = 0.0;
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        double x = 0.0, y = 0.0, z = 0.0;
        for (uint32_t k = 0; k < stride; k++) {
            const float4 r = rec[size_t(stride) * i + k];
            const uint32_t pixel = __float_as_uint(r.w);
            if (pixel >= npix) continue;
            const float* g = dLdI + 3ull * pixel;
            x += double(g[0]) * double(r.x);
            y += double(g[1]) * double(r.y);
            z += double(g[2]) * double(r.z);
        }
        q[4ull * i + 0] = x;
        q[4ull * i + 1] = y;
        q[4ull * i + 2] = z;
        q[4ull * i + 3] = 0.0;
        total += fabs(x) + fabs(y) + fabs(z);
    }
    block_sum_to(total, sum);
}

// The gradients (materials, then lights) times w, to where they go; the replay check's sums and the
// totals after them.
__global__ void k_grad_out(const double* p, uint32_t nmat, uint32_t n, double w, double* mat, double* light,
                           const double* sums, double* sums_out, RunTotals run) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (blockIdx.x == 0 && threadIdx.x < 64) add_totals(run.counters, run.segments, run.totals, run.out);
    if (i < 2) sums_out[i] = sums[i];
    if (i < nmat) mat[i] = p[i] * w;
    else if (i < n) light[i - nmat] = p[i] * w;
}

// ---------------------------------------------------------------------------------
// Host driver

// The camera stage orders its rays by screen tile from this size of the tree as it is built (Node4 and
// TriRecord, some 55,000 triangles) on.  One XCD's L2 is as large; with the 128-byte nodes that the
// kernels read when the line was drawn a smaller tree stayed in the caches whatever the order (room:
// 0.90 -> 1.01 ms; 96k triangles: 11.35 -> 10.72).  With packed nodes the samples matter more than
// the tree, in ms ordered and not: 4.1M samples, terrain of 0.5M triangles 2.09 and 1.91 (compensated
// film 1.90 and 2.02), city of 1M 2.22 and 1.98, 48k to 55k triangles 3.61 and 3.36; 8.4M, 96k
// triangles 7.22 and 6.98; 7.4M, city of 1M 3.04 and 3.14; 16.6M, terrain 6.08 and 6.29 (FP64 film
// 5.29 and 6.07); 66M, city of 16M 26.6 and 29.4; 133M, terrain of 2M 42.0 and 48.2.
constexpr uint64_t kOrderMinBvhBytes = uint64_t(4) << 20;

hipError_t sort_tile_keys(void* temp, size_t& temp_bytes, const uint32_t* keys_in, uint32_t* keys_out,
                          const uint32_t* vals_in, uint32_t* vals_out, uint32_t n, int bits, hipStream_t stream);

// Film replicas of the NEE renders' camera connections (splat_add).
constexpr size_t kSplatMax = 32;
constexpr size_t kSplatMinBytes = size_t(32) << 20;
constexpr size_t kSplatMaxBytes = size_t(1) << 30;

// The film rectangle {x0, y0, x1, y1} (inclusive) that the camera vertex's light connections
// can reach: the raster bounding box of the area lights' triangles, widened by a pixel on
// each side for rounding (a point of a triangle in front of the camera projects inside the
// projected triangle); the whole film with an environment light, or when a light vertex is
// not in front of the camera.
static void connection_rect(const lmgpu_ctx* ctx, uint32_t r[4]) {
    const CameraDev& cam = ctx->cam;
    r[0] = 0;
    r[1] = 0;
    r[2] = uint32_t(cam.width - 1);
    r[3] = uint32_t(cam.height - 1);
    if (ctx->env.index >= 0 || ctx->host_light_tris.empty()) return;
    double lo[2] = {INFINITY, INFINITY}, hi[2] = {-INFINITY, -INFINITY};
    auto mul = [](const M4& m, const double x[4], double o[4]) {
        for (int i = 0; i < 4; i++)
            o[i] = m.m[i] * x[0] + m.m[4 + i] * x[1] + m.m[8 + i] * x[2] + m.m[12 + i] * x[3];
    };
    for (const LightTri& t : ctx->host_light_tris) {
        for (const float* p : {t.p1, t.p2, t.p3}) {
            const double q[4] = {p[0], p[1], p[2], 1.0};
            double v[4], n[4];
            mul(cam.view, q, v);
            if (!(v[2] < 0.0)) return;  // the camera looks down -z
            mul(cam.proj, v, n);
            if (!(n[3] > 0.0)) return;
            const double rx = (n[0] / n[3] + 1.0) / 2.0 * cam.width, ry = (n[1] / n[3] + 1.0) / 2.0 * cam.height;
            if (!std::isfinite(rx) || !std::isfinite(ry)) return;
            lo[0] = std::min(lo[0], rx);
            hi[0] = std::max(hi[0], rx);
            lo[1] = std::min(lo[1], ry);
            hi[1] = std::max(hi[1], ry);
        }
    }
    const double size[2] = {double(cam.width), double(cam.height)};
    for (int a = 0; a < 2; a++) {
        const double l = std::min(std::max(std::floor(lo[a]) - 1.0, 0.0), size[a] - 1.0);
        const double h = std::min(std::max(std::floor(hi[a]) + 1.0, 0.0), size[a] - 1.0);
        r[a] = uint32_t(l);
        r[2 + a] = uint32_t(h);
    }
}

static size_t queue_bytes(uint32_t cap) { return size_t(cap) * 16 * 4; }
static size_t hit_bytes(uint32_t cap) { return (size_t(cap) * 4 + 15) / 16 * 16; }

static void carve(void* base, uint32_t cap, PTBuffers& b) {
    char* p = static_cast<char*>(base);
    for (int k = 0; k < 2; k++) {
        b.q[k].ray_o = reinterpret_cast<float4*>(p); p += size_t(cap) * 16;
        b.q[k].ray_d = reinterpret_cast<float4*>(p); p += size_t(cap) * 16;
        b.q[k].aux = reinterpret_cast<float4*>(p); p += size_t(cap) * 16;
        b.q[k].meta = reinterpret_cast<uint4*>(p); p += size_t(cap) * 16;
    }
    b.hits = reinterpret_cast<uint32_t*>(p); p += hit_bytes(cap);
    b.sq.o = reinterpret_cast<float4*>(p); p += size_t(cap) * 16;
    b.sq.d = reinterpret_cast<float4*>(p); p += size_t(cap) * 16;
    b.sq.c = reinterpret_cast<float4*>(p); p += size_t(cap) * 16;
    b.sq.sid = reinterpret_cast<uint32_t*>(p); p += size_t(cap) * 4;
    b.sq.vis = reinterpret_cast<uint32_t*>(p); p += size_t(cap) * 4;
    b.counters = reinterpret_cast<uint32_t*>(p); p += 4096;
    b.totals = reinterpret_cast<unsigned long long*>(p);
}

static size_t pt_bytes(uint32_t cap) { return 2 * queue_bytes(cap) + hit_bytes(cap) + size_t(cap) * (16 * 3 + 8) + 4096 + 64; }

// Paths in flight per batch when the caller leaves it to the library: the whole render in one
// batch, up to 2^26 paths (12.6 GB of queues) and a quarter of the device memory free for the
// queues and the adjoint's per-sample totals.  Wide batches keep every segment's launch full:
// with RR the late segments of a 2^21-path batch hold a few hundred thousand paths, fewer than
// the persistent traversal grid has lanes.
static uint32_t auto_width(const lmgpu_ctx* ctx, uint64_t num_samples) {
    uint64_t cap = std::min<uint64_t>(num_samples, 1ull << 26);
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) == hipSuccess) {
        const uint64_t per_path = pt_bytes(1) - 4096 - 64 + 32 + 24;  // + camera-ray order
        const uint64_t by_mem = (uint64_t(free_b) + ctx->pt_buf_bytes + ctx->adj_buf_bytes) / 4 / per_path;
        cap = std::min<uint64_t>(cap, std::max<uint64_t>(by_mem, 1ull << 20));
    }
    return uint32_t(cap);
}

// (Re)allocates a context-owned device buffer to at least `bytes`.
static lmgpu_status ensure(lmgpu_ctx* ctx, void** buf, size_t* have, size_t bytes, const char* what) {
    if (bytes <= *have) return LMGPU_OK;
    dev_free(*buf);
    *buf = nullptr;
    *have = 0;
    lmgpu_status s = dev_alloc(ctx, buf, bytes, what);
    if (s != LMGPU_OK) return s;
    *have = bytes;
    return LMGPU_OK;
}

// The path-vertex bound the kernels run with: max_path_vertices, or for -1 (unbounded) the
// vertex after kRouletteTail roulette vertices.  Roulette starts at the vertex count
// max(rr_depth, 1) (the camera vertex counts 1), so a path reaches vertex
// max(rr_depth, 1) + kRouletteTail only after kRouletteTail roulette survivals.
static int effective_max_pv(const lmgpu_pt_params* p) {
    if (p->max_path_vertices != -1) return p->max_path_vertices;
    return std::max(p->rr_depth, 1) + kRouletteTail;
}

static lmgpu_status validate(lmgpu_ctx* ctx, const lmgpu_pt_params* p, const char* fn) {
    const std::string f(fn);
    if (!p) return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, f + ": params is NULL");
    if (!ctx->has_bvh) return fail(ctx, LMGPU_ERR_NO_BVH, f + ": build the BVH first");
    if (!ctx->has_shading || !ctx->has_camera)
        return fail(ctx, LMGPU_ERR_NO_SCENE, f + ": scene has no materials or camera");
    if (p->renderer < LMGPU_PT || p->renderer > LMGPU_PT_MIS)
        return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, f + ": unknown renderer");
    if (p->renderer != LMGPU_PT && ctx->num_lights == 0)
        return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, f + ": pt.direct / pt.mis need at least one light");
    if (p->film_precision != LMGPU_FILM_FP32 && p->film_precision != LMGPU_FILM_FP64 &&
        p->film_precision != LMGPU_FILM_FP32_COMPENSATED)
        return fail(ctx, LMGPU_ERR_UNSUPPORTED, f + ": film precision not supported");
    if (p->num_samples == 0) return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, f + ": num_samples is 0");
    if (p->max_path_vertices == 0 || p->max_path_vertices < -1)
        return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, f + ": max_path_vertices must be -1 or >= 1");
    if (p->max_path_vertices > kMaxSegments)
        return fail(ctx, LMGPU_ERR_UNSUPPORTED,
                    f + ": max_path_vertices must be -1 or in [1, " + std::to_string(kMaxSegments) + "]");
    if (p->max_path_vertices == -1 && p->rr_depth == -1)
        return fail(ctx, LMGPU_ERR_UNSUPPORTED,
                    f + ": max_path_vertices = -1 needs Russian roulette (rr_depth != -1): the paths would not end");
    if (p->max_path_vertices == -1 && effective_max_pv(p) > kMaxSegments)
        return fail(ctx, LMGPU_ERR_UNSUPPORTED,
                    f + ": max_path_vertices = -1 supports rr_depth <= " + std::to_string(kMaxSegments - kRouletteTail));
    if (3u * ctx->bvh_max_depth > uint32_t(kStackTotal))
        return fail(ctx, LMGPU_ERR_BVH_TOO_DEEP, f + ": BVH deeper than the traversal stack");
    return LMGPU_OK;
}

// Shared state of one render / adjoint run.
struct Pipeline {
    lmgpu_ctx* ctx;
    PTConsts c;
    PTBuffers b;
    uint32_t cap;
    uint32_t trace_grid;
    int segments;
    bool is_pt;
    bool brute;  // at most kBruteMaxTrisPt (pt) / kBruteMaxTris triangles: no BVH descent
    // pt camera-stage order (large scenes): keys and samples in, sorted out, sort scratch.
    uint32_t *keys_in = nullptr, *keys_out = nullptr, *vals_in = nullptr, *vals_out = nullptr;
    void* sort_temp = nullptr;
    size_t sort_temp_bytes = 0;
    int key_bits = 0;
    int key_skip = 0;
    bool counters_clear = false;  // the next batch need not clear them

    // Clears what a run starts from (k_clear).
    void clear(void* a, size_t a_bytes, void* b2, size_t b2_bytes) {
        const size_t na = a_bytes / 16, nb = b2_bytes / 16;
        const uint32_t nw = (4096u + 64u) / 4u;
        hipLaunchKernelGGL(k_clear, dim3(uint32_t((std::max<size_t>(na + nb, nw) + 255) / 256)), dim3(256), 0, ctx->stream,
                           static_cast<uint4*>(a), na, static_cast<uint4*>(b2), nb, b.counters, nw);
        counters_clear = true;
    }
    RunTotals run_totals(unsigned long long* out) const { return {b.counters, segments + 1, b.totals, out}; }

    lmgpu_status setup(const lmgpu_pt_params* p) {
        cap = p->wavefront_width ? p->wavefront_width : auto_width(ctx, p->num_samples);
        cap = uint32_t(std::min<uint64_t>(cap, p->num_samples));
        cap = std::max<uint32_t>(cap, 64u);
        lmgpu_status st = ensure(ctx, &ctx->pt_buf, &ctx->pt_buf_bytes, pt_bytes(cap), "path queues");
        if (st != LMGPU_OK) return st;
        ctx->pt_capacity = cap;
        carve(ctx->pt_buf, cap, b);
        c = PTConsts{};
        c.bvh = bvh_of(ctx);
        c.xform = ctx->xform.ptr;
        c.shade = ctx->shade.ptr;
        c.mats = ctx->mats.ptr;
        c.lights = ctx->lights.ptr;
        c.light_tris = ctx->light_tris.ptr;
        c.num_lights = ctx->num_lights;
        c.cam = ctx->cam;
        c.env = ctx->env;
        c.seed = p->seed;
        c.max_pv = effective_max_pv(p);
        c.rr_depth = p->rr_depth;
        c.renderer = p->renderer;
        c.film_mode = p->film_precision;
        int occ_e = 0, occ_s = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ_e, k_extend<false>, kTraceBlock, 0) != hipSuccess ||
            occ_e < 1)
            occ_e = 1;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ_s, (k_shadow<kRender, false, false>), kTraceBlock, 0) !=
                hipSuccess ||
            occ_s < 1)
            occ_s = 1;
        trace_grid = uint32_t(std::max(ctx->num_cus, 1)) * uint32_t(std::min(occ_e, occ_s));
        // Segments traced per path: at most max_path_vertices - 1 (pathtrace.cpp:196-199).
        segments = c.max_pv - 1;
        is_pt = p->renderer == LMGPU_PT;
        brute = ctx->num_records <= (is_pt ? kBruteMaxTrisPt : kBruteMaxTris);
        c.ntris = ctx->num_records;
        // A BVH larger than the caches: camera rays in screen-tile order (k_tile_keys), whose
        // raster numbers follow key_skip others in each stream.
        c.order = nullptr;
        key_skip = is_pt ? 0 : 4 + (p->rr_depth != -1 && p->rr_depth <= 1 ? 1 : 0);
        const uint64_t bvh_bytes = uint64_t(ctx->nodes.count) * sizeof(Node4) + uint64_t(ctx->num_records) * sizeof(TriRecord);
        if (bvh_bytes >= kOrderMinBvhBytes) {
            const uint32_t tiles = uint32_t(std::max((ctx->cam.width + 7) / 8, (ctx->cam.height + 7) / 8));
            key_bits = 2;
            while ((1u << (key_bits / 2)) < tiles) key_bits += 2;
            size_t temp = 0;
            hipError_t e = sort_tile_keys(nullptr, temp, nullptr, nullptr, nullptr, nullptr, cap, key_bits, ctx->stream);
            if (e != hipSuccess) return hip_fail(ctx, e, "camera ray order (sort size)");
            const size_t arr = (size_t(cap) * 4 + 255) / 256 * 256;
            st = ensure(ctx, &ctx->order_buf, &ctx->order_buf_bytes, 4 * arr + temp, "camera ray order");
            if (st != LMGPU_OK) return st;
            char* base = static_cast<char*>(ctx->order_buf);
            keys_in = reinterpret_cast<uint32_t*>(base);
            keys_out = reinterpret_cast<uint32_t*>(base + arr);
            vals_in = reinterpret_cast<uint32_t*>(base + 2 * arr);
            vals_out = reinterpret_cast<uint32_t*>(base + 3 * arr);
            sort_temp = base + 4 * arr;
            sort_temp_bytes = temp;
            c.order = vals_out;
        }
        return LMGPU_OK;
    }

    // One batch [base, base + nb) of the global sample range through every stage.
    // counters[k]: queue entering segment k; counters[kMaxSegments + k]: shadow rays emitted
    // before segment k; [2 kMaxSegments, 4 kMaxSegments + 1): work counters of the launches.
    // `last`: the run's last kernel adds its counters to the totals.
    template <int kMode> lmgpu_status batch(uint64_t base, uint32_t nb, bool last) {
        hipStream_t s = ctx->stream;
        c.base = base;
        c.batch = nb;
        if (!counters_clear)
            hipLaunchKernelGGL(k_zero_u32, dim3(2), dim3(256), 0, s, b.counters, uint32_t(4 * kMaxSegments));
        counters_clear = false;
        const dim3 grid_b((nb + kPTBlock - 1) / kPTBlock);
        // Persistent traversal grids: the device fill, never more than the queue capacity needs with a
        // wave per ray.
        const dim3 grid_t(std::min<uint32_t>((cap + kTraceBlock / 64 - 1) / (kTraceBlock / 64), trace_grid));
        // Brute-force traversal grids: 16 blocks of kTraceBlock per CU, walking the queue.
        const dim3 grid_r(std::min<uint32_t>((cap + kTraceBlock - 1) / kTraceBlock, 16u * uint32_t(std::max(ctx->num_cus, 1))));
        const uint32_t ntris = ctx->num_records;
        // Shade grids: 16 blocks per CU; the gradient pass 4, each flushing its gradient table once.
        // Where few paths get a group of lanes each (lanes_per_path), a block for every kPTBlock lanes:
        // with one for as many paths a render of 64 x 64 x 8 used half the CUs, 269 us against 195.
        const uint32_t lanes = brute ? std::max(cap, std::min(cap, kSplitLanes / kSplitMax) * kSplitMax) : cap;
        const dim3 grid_s(std::min<uint32_t>((lanes + kPTBlock - 1) / kPTBlock, (kMode == kAdjGrad ? 4u : 16u) * uint32_t(std::max(ctx->num_cus, 1))));
        hipError_t sort_e = hipSuccess;
        // Render of a scene of at most kBruteMaxTris triangles: shadow rays are traced where
        // they are made (shadow_visible, add_connection), so no shadow launches.
        const bool fuse_shadow = brute && kMode == kRender;
        hipError_t e = timed(ctx, kKGen, [&]() {
            if (c.order) {
                hipLaunchKernelGGL(k_tile_keys, grid_b, dim3(kPTBlock), 0, s, c, key_skip, keys_in, vals_in);
                size_t tb = sort_temp_bytes;
                sort_e = sort_tile_keys(sort_temp, tb, keys_in, keys_out, vals_in, vals_out, nb, key_bits, s);
            }
            if (fuse_shadow)
                hipLaunchKernelGGL((k_gen<kMode, true>), grid_b, dim3(kPTBlock), 0, s, c, b.q[0], b.counters + 0, b.sq,
                                   b.counters + kMaxSegments + 0);
            else
                hipLaunchKernelGGL(k_gen<kMode>, grid_b, dim3(kPTBlock), 0, s, c, b.q[0], b.counters + 0, b.sq,
                                   b.counters + kMaxSegments + 0);
        });
        if (sort_e != hipSuccess) return hip_fail(ctx, sort_e, "camera ray order (sort)");
        if (e != hipSuccess) return hip_fail(ctx, e, "k_gen");
        // lmgpu_enable_counting: the BVH traversal stages in their counting forms.
        const bool counting = ctx->counting;
        unsigned long long* ext_counts = ctx->trav_counts;
        unsigned long long* shadow_counts = ctx->trav_counts + 2;
        auto shadow = [&](int k) -> lmgpu_status {
            hipError_t e2 = timed(ctx, kKShadow, [&]() {
                const uint32_t* cnt = b.counters + kMaxSegments + k;
                uint32_t* work = b.counters + 3 * kMaxSegments + k;
                if constexpr (kMode == kRender) {
                    if (k == 0 && c.splat) {
                        if (brute)
                            hipLaunchKernelGGL((k_shadow_brute<kRender, true>), grid_r, dim3(kTraceBlock), 0, s, c,
                                               ntris, b.sq, cnt);
                        else if (counting)
                            hipLaunchKernelGGL((k_shadow<kRender, true, true>), grid_t, dim3(kTraceBlock), 0, s, c,
                                               b.sq, cnt, work, shadow_counts);
                        else
                            hipLaunchKernelGGL((k_shadow<kRender, true>), grid_t, dim3(kTraceBlock), 0, s, c, b.sq,
                                               cnt, work, shadow_counts);
                        return;
                    }
                }
                if (brute)
                    hipLaunchKernelGGL(k_shadow_brute<kMode>, grid_r, dim3(kTraceBlock), 0, s, c, ntris, b.sq, cnt);
                else if (counting)
                    hipLaunchKernelGGL((k_shadow<kMode, false, true>), grid_t, dim3(kTraceBlock), 0, s, c, b.sq, cnt,
                                       work, shadow_counts);
                else
                    hipLaunchKernelGGL(k_shadow<kMode>, grid_t, dim3(kTraceBlock), 0, s, c, b.sq, cnt, work,
                                       shadow_counts);
            });
            if (e2 != hipSuccess) return hip_fail(ctx, e2, "k_shadow");
            if (kMode != kRender) {
                hipLaunchKernelGGL(k_shadow_apply<kMode>, grid_s, dim3(kPTBlock), 0, s, c, b.sq,
                                   b.counters + kMaxSegments + k);
                e2 = hipGetLastError();
                if (e2 != hipSuccess) return hip_fail(ctx, e2, "k_shadow_apply");
            }
            return LMGPU_OK;
        };
        if (!is_pt && !fuse_shadow) {
            lmgpu_status st = shadow(0);
            if (st != LMGPU_OK) return st;
        }
        if (kMode == kRender && !is_pt && c.conn_lds) {
            // The camera vertex's connections, staged per shadow slot by the camera stage (or its
            // shadow launch), summed before the first segment reuses the slots.
            const dim3 grid_cr(std::min<uint32_t>(grid_b.x, 2u * uint32_t(std::max(ctx->num_cus, 1))));
            e = timed(ctx, kKGen, [&]() {
                if (c.film_mode == LMGPU_FILM_FP32)
                    hipLaunchKernelGGL(k_conn_reduce<float>, grid_cr, dim3(kPTBlock), 0, s, c, b.sq.c,
                                       b.counters + kMaxSegments);
                else
                    hipLaunchKernelGGL(k_conn_reduce<double>, grid_cr, dim3(kPTBlock), 0, s, c, b.sq.c,
                                       b.counters + kMaxSegments);
            });
            if (e != hipSuccess) return hip_fail(ctx, e, "k_conn_reduce");
        }
        for (int k = 0; k < segments; k++) {
            const Queue& qi = b.q[k & 1];
            const Queue& qo = b.q[(k + 1) & 1];
            const float tmin = is_pt && k == 0 ? 0.f : kEps;  // pt's camera rays (pathtrace.cpp:187-192) start at 0
            // Scenes of at most kBruteMaxTris triangles: the shading kernel traces the segment's
            // rays itself (kFuse), so there is no extension launch and no hit record.
            if (!brute) {
                e = timed(ctx, kKExtend, [&]() {
                    if (counting)
                        hipLaunchKernelGGL(k_extend<true>, grid_t, dim3(kTraceBlock), 0, s, c.bvh, qi, tmin,
                                           b.counters + k, b.counters + 2 * kMaxSegments + k, b.hits, ext_counts);
                    else
                        hipLaunchKernelGGL(k_extend<false>, grid_t, dim3(kTraceBlock), 0, s, c.bvh, qi, tmin,
                                           b.counters + k, b.counters + 2 * kMaxSegments + k, b.hits, ext_counts);
                });
                if (e != hipSuccess) return hip_fail(ctx, e, "k_extend");
            }
            e = timed(ctx, kKShade, [&]() {
                if (is_pt && brute)
                    hipLaunchKernelGGL((k_shade_pt<kMode, true>), grid_s, dim3(kPTBlock), 0, s, c, qi, tmin, b.counters + k,
                                       b.hits, qo, b.counters + k + 1);
                else if (is_pt && kMode == kRender && c.order && c.film_mode != LMGPU_FILM_FP32)
                    hipLaunchKernelGGL((k_shade_pt<kMode, false, kMode == kRender>), grid_s, dim3(kPTBlock), 0, s, c, qi,
                                       tmin, b.counters + k, b.hits, qo, b.counters + k + 1);
                else if (is_pt)
                    hipLaunchKernelGGL(k_shade_pt<kMode>, grid_s, dim3(kPTBlock), 0, s, c, qi, tmin, b.counters + k, b.hits,
                                       qo, b.counters + k + 1);
                else if (brute)
                    hipLaunchKernelGGL((k_shade_nee<kMode, true>), grid_s, dim3(kPTBlock), 0, s, c, qi, tmin, b.counters + k,
                                       b.hits, qo, b.counters + k + 1, b.sq, b.counters + kMaxSegments + k + 1);
                else
                    hipLaunchKernelGGL(k_shade_nee<kMode>, grid_s, dim3(kPTBlock), 0, s, c, qi, tmin, b.counters + k,
                                       b.hits, qo, b.counters + k + 1, b.sq, b.counters + kMaxSegments + k + 1);
            });
            if (e != hipSuccess) return hip_fail(ctx, e, "k_shade");
            if (!is_pt && !fuse_shadow) {
                lmgpu_status st = shadow(k + 1);
                if (st != LMGPU_OK) return st;
            }
        }
        // k_shade_pt never enqueues a path whose vertex count reached max_path_vertices, so
        // the final queue is empty.
        if (!last) hipLaunchKernelGGL(k_accumulate_totals, dim3(1), dim3(64), 0, s, b.counters, segments + 1, b.totals);
        e = hipGetLastError();
        if (e != hipSuccess) return hip_fail(ctx, e, "k_accumulate_totals");
        return LMGPU_OK;
    }
};

// A film of up to this many bytes is resolved into pinned host memory: the link takes it as fast as
// a copy would, without the copy's launch.
constexpr size_t kDirectFilm = (size_t(1) << 20) - kPinnedWords;
constexpr double kDirectUs = 80.0;  // a MiB so saved: the room at 256 x 256 (768 KB) 395 -> 335 us

lmgpu_status run_raycast(lmgpu_ctx* ctx, lmgpu_film* film) {
    if (!ctx->has_bvh) return fail(ctx, LMGPU_ERR_NO_BVH, "lmgpu_raycast_render: build the BVH first");
    if (!ctx->has_shading || !ctx->has_camera)
        return fail(ctx, LMGPU_ERR_NO_SCENE, "lmgpu_raycast_render: scene has no materials or camera");
    if (!film || !film->data || film->width != uint32_t(ctx->cam.width) || film->height != uint32_t(ctx->cam.height))
        return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_raycast_render: film size differs from the camera's");
    if (film->precision != LMGPU_FILM_FP32 && film->precision != LMGPU_FILM_FP64)
        return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_raycast_render: output film precision");
    if (3u * ctx->bvh_max_depth > uint32_t(kStackTotal))
        return fail(ctx, LMGPU_ERR_BVH_TOO_DEEP, "lmgpu_raycast_render: BVH deeper than the traversal stack");
    const uint32_t n = uint32_t(ctx->cam.width) * uint32_t(ctx->cam.height);
    const size_t out_bytes = size_t(n) * 3 * (film->precision == LMGPU_FILM_FP64 ? 8 : 4);
    void* out_dev = film->data;
    if (!film->device) {
        lmgpu_status st = ensure(ctx, &ctx->film_out_staging, &ctx->film_out_staging_bytes, out_bytes, "film staging");
        if (st != LMGPU_OK) return st;
        out_dev = ctx->film_out_staging;
    }
    PTConsts c{};
    c.bvh = bvh_of(ctx);
    c.shade = ctx->shade.ptr;
    c.mats = ctx->mats.ptr;
    c.lights = ctx->lights.ptr;
    c.cam = ctx->cam;
    c.env = ctx->env;
    int occ = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, k_raycast<float>, kTraceBlock, 0) != hipSuccess || occ < 1)
        occ = 1;
    const uint32_t grid = std::min<uint32_t>((n + kTraceBlock / 64 - 1) / (kTraceBlock / 64),
                                             uint32_t(std::max(ctx->num_cus, 1)) * uint32_t(occ));
    hipStream_t s = ctx->stream;
    hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, s, ctx->next_counter, 1u);
    hipError_t e = timed(ctx, kKTraceClosest, [&]() {
        if (film->precision == LMGPU_FILM_FP64)
            hipLaunchKernelGGL(k_raycast<double>, dim3(grid), dim3(kTraceBlock), 0, s, c, n, ctx->next_counter,
                               static_cast<double*>(out_dev));
        else
            hipLaunchKernelGGL(k_raycast<float>, dim3(grid), dim3(kTraceBlock), 0, s, c, n, ctx->next_counter,
                               static_cast<float*>(out_dev));
    });
    if (e != hipSuccess) return hip_fail(ctx, e, "k_raycast");
    e = film->device ? hipStreamSynchronize(s) : read_back(ctx, film->data, out_dev, out_bytes, ring_pays(ctx, out_bytes));
    if (e != hipSuccess) return hip_fail(ctx, e, "raycast readback");
    return LMGPU_OK;
}

lmgpu_status run_pt(lmgpu_ctx* ctx, const lmgpu_pt_params* p, lmgpu_film* film, lmgpu_pt_stats* stats) {
    lmgpu_status st = validate(ctx, p, "lmgpu_pt_render");
    if (st != LMGPU_OK) return st;
    if (!film || !film->data || film->width != uint32_t(ctx->cam.width) || film->height != uint32_t(ctx->cam.height))
        return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_pt_render: film size differs from the camera's");
    if (film->precision != LMGPU_FILM_FP32 && film->precision != LMGPU_FILM_FP64)
        return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_pt_render: output film precision");

    Pipeline pl{ctx};
    st = pl.setup(p);
    if (st != LMGPU_OK) return st;
    const size_t npix = size_t(ctx->cam.width) * size_t(ctx->cam.height);
    const size_t nval = npix * 3;
    const bool comp = p->film_precision == LMGPU_FILM_FP32_COMPENSATED;
    const size_t acc_elem = p->film_precision == LMGPU_FILM_FP64 ? 8 : 4;
    const size_t acc_one = (nval * acc_elem + 15) / 16 * 16;
    const size_t acc_bytes = comp ? 2 * acc_one : acc_one;
    st = ensure(ctx, &ctx->film_acc, &ctx->film_acc_bytes, acc_bytes, "film accumulator");
    if (st != LMGPU_OK) return st;
    const size_t out_elem = film->precision == LMGPU_FILM_FP64 ? 8 : 4;
    const size_t out_bytes = nval * out_elem;
    void* out_dev = film->data;
    // The pinned memory is grown here, before it holds the words.
    const bool small = !film->device && out_bytes <= kDirectFilm;
    const bool ring = !film->device && ring_pays(ctx, out_bytes);
    const bool in_place = small && pinned_pays(ctx, kPinnedWords + out_bytes, double(out_bytes) * (kDirectUs / (1 << 20)));
    const bool pinned = ensure_pinned(ctx, kPinnedWords + (ring || in_place ? std::min(out_bytes, kReadSlots * kReadSlot) : 0));
    const bool direct = in_place && pinned;
    unsigned long long words_here[4];
    void* const words = pinned ? ctx->io->pinned : words_here;
    if (direct) {
        out_dev = static_cast<char*>(ctx->io->pinned) + kPinnedWords;
    } else if (!film->device) {
        st = ensure(ctx, &ctx->film_out_staging, &ctx->film_out_staging_bytes, out_bytes, "film staging");
        if (st != LMGPU_OK) return st;
        out_dev = ctx->film_out_staging;
    }
    pl.c.film = ctx->film_acc;
    pl.c.film_comp = comp ? reinterpret_cast<float*>(static_cast<char*>(ctx->film_acc) + acc_one) : nullptr;
    // NEE renderers: replicas of the film rectangle the lights project to, for the camera
    // vertex's light connections (splat_add): at most kSplatMax, within 8 bytes per sample
    // clamped to [kSplatMinBytes, kSplatMaxBytes], a multiple of 8 from 8 on.
    size_t splat_bytes = 0, splat_vals = 0;
    if (p->renderer != LMGPU_PT) {
        uint32_t r[4];
        connection_rect(ctx, r);
        pl.c.splat_x0 = r[0];
        pl.c.splat_y0 = r[1];
        pl.c.splat_w = r[2] - r[0] + 1;
        pl.c.splat_h = r[3] - r[1] + 1;
        splat_vals = size_t(pl.c.splat_w) * pl.c.splat_h * 3;
        const size_t elem = p->film_precision == LMGPU_FILM_FP32 ? 4 : 8;
        const size_t one = (splat_vals * elem + 255) / 256 * 256;
        const size_t budget = std::min(kSplatMaxBytes, std::max(kSplatMinBytes, size_t(p->num_samples) * 8));
        size_t k = std::min(kSplatMax, std::max<size_t>(1, budget / one));
        if (k >= 8) k &= ~size_t(7);
        splat_bytes = k * one;
        st = ensure(ctx, &ctx->splat_buf, &ctx->splat_buf_bytes, splat_bytes, "film replicas");
        if (st != LMGPU_OK) return st;
        pl.c.splat = ctx->splat_buf;
        pl.c.splat_k = uint32_t(k);
        pl.c.splat_vals = one / elem;
        // The connections' rectangle fits k_conn_reduce's LDS sums (elem bytes per value).
        pl.c.conn_lds = splat_vals * elem <= kConnLdsBytes ? 1 : 0;
    }

    hipStream_t s = ctx->stream;
    (void)hipEventRecord(ctx->run0, s);
    pl.clear(ctx->film_acc, acc_bytes, ctx->splat_buf, splat_bytes);
    const uint32_t rec_stride = p->renderer == LMGPU_PT ? 1u : 2u;  // float4 per sample in the record
    for (uint64_t base = 0; base < p->num_samples && st == LMGPU_OK; base += pl.cap) {
        pl.c.record = p->sample_record ? static_cast<float4*>(p->sample_record) + rec_stride * base : nullptr;
        const uint32_t nb = uint32_t(std::min<uint64_t>(pl.cap, p->num_samples - base));
        st = pl.batch<kRender>(p->sample_offset + base, nb, base + nb == p->num_samples);
    }
    if (st == LMGPU_OK) {
        // Resolve: sums * W*H/N into the output film.
        const dim3 rg(uint32_t((nval + 255) / 256));
        const double w = double(npix) / double(p->num_samples);
        const RunTotals run = pl.run_totals(pinned ? static_cast<unsigned long long*>(words) : pl.b.totals);
        auto resolve = [&](auto kernel, auto* out, auto weight) {
            hipLaunchKernelGGL(kernel, rg, dim3(256), 0, s, pl.c, out, nval, weight, run);
        };
        auto resolve_to = [&](auto* out) {
            using Out = std::remove_pointer_t<decltype(out)>;
            if (comp && splat_bytes) resolve(k_resolve<float, Out, true, true>, out, w);
            else if (comp) resolve(k_resolve<float, Out, true, false>, out, w);
            else if (p->film_precision == LMGPU_FILM_FP64 && splat_bytes) resolve(k_resolve<double, Out, false, true>, out, w);
            else if (p->film_precision == LMGPU_FILM_FP64) resolve(k_resolve<double, Out, false, false>, out, w);
            else if (splat_bytes) resolve(k_resolve<float, Out, false, true>, out, float(npix) / float(p->num_samples));
            else resolve(k_resolve<float, Out, false, false>, out, float(npix) / float(p->num_samples));
        };
        if (film->precision == LMGPU_FILM_FP64) resolve_to(static_cast<double*>(out_dev));
        else resolve_to(static_cast<float*>(out_dev));
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) st = hip_fail(ctx, e, "k_resolve");
    }
    (void)hipEventRecord(ctx->run1, s);
    unsigned long long totals[2] = {0, 0};
    if (st == LMGPU_OK) {
        hipError_t e = pinned ? hipSuccess : hipMemcpyAsync(words, pl.b.totals, sizeof(totals), hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = film->device || direct ? hipStreamSynchronize(s) : read_back(ctx, film->data, out_dev, out_bytes, ring);
        if (e != hipSuccess) st = hip_fail(ctx, e, "pt readback");
        else std::memcpy(totals, words, sizeof(totals));
        if (e == hipSuccess && direct) {
            const CopyJob job{static_cast<char*>(film->data), static_cast<const char*>(out_dev), out_bytes};
            ctx->io->team.run(&job, 1);
        }
    }
    float ms = 0.f;
    if (st == LMGPU_OK) (void)hipEventElapsedTime(&ms, ctx->run0, ctx->run1);
    if (st != LMGPU_OK) return st;
    if (stats) {
        stats->closest_rays = totals[0];
        stats->shadow_rays = totals[1];
        stats->samples = p->num_samples;
        stats->seconds = double(ms) / 1000.0;
    }
    return LMGPU_OK;
}

lmgpu_status run_pt_backward(lmgpu_ctx* ctx, const lmgpu_pt_params* p, lmgpu_adjoint* adj, lmgpu_pt_stats* stats) {
    lmgpu_status st = validate(ctx, p, "lmgpu_pt_backward");
    if (st != LMGPU_OK) return st;
    if (!adj || !adj->d_image || !adj->d_albedo || (ctx->num_lights > 0 && !adj->d_emission))
        return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_pt_backward: missing image gradient or outputs");

    Pipeline pl{ctx};
    st = pl.setup(p);
    if (st != LMGPU_OK) return st;
    const size_t npix = size_t(ctx->cam.width) * size_t(ctx->cam.height);
    const size_t nval = npix * 3;
    const uint32_t ngrad = 3u * (ctx->num_materials + ctx->num_lights);
    // Q per batch sample (4 doubles), the gradients, two residual sums, the staged dL/dI.
    const size_t q_bytes = size_t(pl.cap) * 32;
    const size_t g_bytes = (size_t(ngrad) * 8 + 15) / 16 * 16;
    const size_t img_bytes = adj->image_device ? 0 : (nval * 4 + 15) / 16 * 16;
    const size_t need = q_bytes + g_bytes + 16 + img_bytes;
    st = ensure(ctx, &ctx->adj_buf, &ctx->adj_buf_bytes, need, "adjoint buffers");
    if (st != LMGPU_OK) return st;
    char* ab = static_cast<char*>(ctx->adj_buf);
    pl.c.qacc = reinterpret_cast<double*>(ab);
    double* grad = reinterpret_cast<double*>(ab + q_bytes);
    double* sums = reinterpret_cast<double*>(ab + q_bytes + g_bytes);
    pl.c.grad_mat = grad;
    pl.c.grad_light = grad + 3ull * ctx->num_materials;
    hipStream_t s = ctx->stream;
    hipError_t e = hipSuccess;
    if (adj->image_device) {
        pl.c.dLdI = adj->d_image;
    } else {
        float* img = reinterpret_cast<float*>(ab + q_bytes + g_bytes + 16);
        e = hipMemcpyAsync(img, adj->d_image, nval * 4, hipMemcpyHostToDevice, s);
        if (e != hipSuccess) return hip_fail(ctx, e, "image gradient upload");
        pl.c.dLdI = img;
    }
    pl.c.film_mode = LMGPU_FILM_FP32;

    (void)hipEventRecord(ctx->run0, s);
    pl.clear(grad, g_bytes + 16, nullptr, 0);
    const uint32_t rec_stride = p->renderer == LMGPU_PT ? 1u : 2u;  // float4 per sample in the record
    for (uint64_t base = 0; base < p->num_samples && st == LMGPU_OK; base += pl.cap) {
        const uint32_t nb = uint32_t(std::min<uint64_t>(pl.cap, p->num_samples - base));
        const dim3 grid_sum(std::min<uint32_t>((nb + 255) / 256, 256u));
        if (p->sample_record) {
            // The forward's record holds every sample's contributions: Q without a replay.
            hipLaunchKernelGGL(k_q_from_record, dim3(std::min<uint32_t>((nb + 255) / 256, 4096u)), dim3(256), 0, s,
                               static_cast<const float4*>(p->sample_record) + rec_stride * base, rec_stride,
                               pl.c.dLdI, uint32_t(npix), nb, pl.c.qacc, sums + 0);
            e = hipGetLastError();
            if (e != hipSuccess) {
                st = hip_fail(ctx, e, "k_q_from_record");
                break;
            }
        } else {
            hipLaunchKernelGGL(k_zero_bytes, dim3(uint32_t((size_t(nb) * 2 + 255) / 256)), dim3(256), 0, s,
                               reinterpret_cast<uint4*>(pl.c.qacc), size_t(nb) * 2);
            st = pl.batch<kAdjTotal>(p->sample_offset + base, nb, false);
            if (st != LMGPU_OK) break;
            hipLaunchKernelGGL(k_abs_sum, grid_sum, dim3(256), 0, s, pl.c.qacc, nb, sums + 0);
        }
        st = pl.batch<kAdjGrad>(p->sample_offset + base, nb, base + nb == p->num_samples);
        if (st != LMGPU_OK) break;
        hipLaunchKernelGGL(k_abs_sum, grid_sum, dim3(256), 0, s, pl.c.qacc, nb, sums + 1);
    }
    unsigned long long totals[2] = {0, 0};
    double hs[2] = {0.0, 0.0};
    const uint32_t nmat = 3u * ctx->num_materials, nlight = ngrad - nmat;
    const bool pinned = ensure_pinned(ctx, kPinnedWords);
    // The sums and the totals, on the device where there is no pinned memory.
    double* const hs_out = pinned ? static_cast<double*>(ctx->io->pinned) : sums;
    unsigned long long* const totals_out = pinned ? reinterpret_cast<unsigned long long*>(hs_out + 2) : pl.b.totals;
    if (st == LMGPU_OK) {
        // The film is Sum * W*H/N (sched.mt.cpp:256): the same factor scales its gradient.
        hipLaunchKernelGGL(k_grad_out, dim3((ngrad + 255) / 256), dim3(256), 0, s, grad, nmat, ngrad,
                           double(npix) / double(p->num_samples), adj->grad_device ? adj->d_albedo : grad,
                           adj->grad_device ? adj->d_emission : grad + nmat, sums, hs_out, pl.run_totals(totals_out));
        e = hipGetLastError();
        if (e != hipSuccess) st = hip_fail(ctx, e, "k_grad_out");
    }
    (void)hipEventRecord(ctx->run1, s);
    if (st == LMGPU_OK) {
        if (!adj->grad_device) {
            e = hipMemcpyAsync(adj->d_albedo, grad, size_t(nmat) * 8, hipMemcpyDeviceToHost, s);
            if (e == hipSuccess && nlight > 0)
                e = hipMemcpyAsync(adj->d_emission, grad + nmat, size_t(nlight) * 8, hipMemcpyDeviceToHost, s);
        }
        if (!pinned) {
            if (e == hipSuccess) e = hipMemcpyAsync(hs, sums, sizeof(hs), hipMemcpyDeviceToHost, s);
            if (e == hipSuccess) e = hipMemcpyAsync(totals, pl.b.totals, sizeof(totals), hipMemcpyDeviceToHost, s);
        }
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e != hipSuccess) {
            st = hip_fail(ctx, e, "adjoint readback");
        } else if (pinned) {
            std::memcpy(hs, hs_out, sizeof(hs));
            std::memcpy(totals, totals_out, sizeof(totals));
        }
    }
    float ms = 0.f;
    if (st == LMGPU_OK) (void)hipEventElapsedTime(&ms, ctx->run0, ctx->run1);
    if (st != LMGPU_OK) return st;
    adj->replay_residual = hs[0] > 0.0 ? hs[1] / hs[0] : 0.0;
    if (stats) {
        stats->closest_rays = totals[0];
        stats->shadow_rays = totals[1];
        stats->samples = p->num_samples;
        stats->seconds = double(ms) / 1000.0;
    }
    return LMGPU_OK;
}

}  // namespace lmgpu
