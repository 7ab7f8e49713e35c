// Internal state of an lmgpu context and the device-side scene records.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/lmgpu.h"
#include "bvh_build.h"
#include "device_math.hpp"
#include "host_io.hpp"

namespace lmgpu {

// Per-triangle shading record in scene order (64 B): geometric normal (as the reference
// computes it, normalize(cross(p2 - p1, p3 - p1)), scene.cpp:121-127), material,
// light, and the three vertex normals for the interpolated shading normal (:130-133).
struct alignas(16) ShadeTri {
    float gn[3];
    uint32_t mat;
    float n1[3];
    int32_t light;
    float n2[3];
    float pad0;
    float n3[3];
    float pad1;
};
static_assert(sizeof(ShadeTri) == 64, "ShadeTri is 64 bytes");

struct alignas(16) MaterialDev {
    uint32_t type;
    float R[3];
};

// Area light: its triangles are light_tris[tri_begin, tri_begin + tri_count).
struct alignas(16) LightDev {
    uint32_t type;
    float Le[3];
    uint32_t tri_begin, tri_count;
    float inv_area;
    float pad;
};

// Light triangle: vertices, w of p1 = cumulative area fraction before it, w of p2 = after it
// (AreaLight::RegisterPrimitives, light.area.cpp:109-144).
struct alignas(16) LightTri {
    float p1[4];
    float p2[4];
    float p3[4];
};

struct CameraDev {
    M4 view, inv_view, proj, inv_proj;
    float pos[3];
    float inv_A;
    int width, height;
};

struct EnvDev {
    float center[3];
    float radius;
    float Le[3];
    float inv_area;
    int index;  // light index, -1 if there is no environment light
};

// Kernel classes for lmgpu_kernel_timing.
enum KernelClass : int {
    kKTraceClosest = 0,
    kKTraceAny = 1,
    kKShade = 2,
    kKGen = 3,
    kKShadow = 4,
    kKExtend = 5,
    kKNumClasses = 6
};

template <class T> struct DevBuf {
    T* ptr = nullptr;
    size_t count = 0;
};

}  // namespace lmgpu

struct lmgpu_ctx {
    int device = 0;
    int num_cus = 0;
    hipStream_t own_stream = nullptr;
    hipStream_t stream = nullptr;
    std::string err;
    int inject_alloc_failures = 0;

    // Host copies needed by the BVH build and the light / camera setup.
    std::vector<float> positions;
    std::vector<uint32_t> faces;
    uint32_t num_vertices = 0, num_triangles = 0;
    bool has_scene = false;
    bool has_shading = false;
    bool has_camera = false;

    // Device scene
    // One allocation, nodes.ptr: the packed nodes, the nodes as built (as many) and the records.
    lmgpu::DevBuf<lmgpu::NodeQ> nodes;
    lmgpu::Node4* exact_nodes = nullptr;
    float reach = 0.f;                        // the largest coordinate of the scene's box
    lmgpu::DevBuf<lmgpu::TriRecord> tris;  // scenes of at most kBruteMaxTris triangles, else empty
    struct {
        lmgpu::LeafTri* ptr;
        size_t count;
    } leaf_tris{nullptr, 0};
    uint32_t num_records = 0;  // triangle records of the built tree
    lmgpu::DevBuf<lmgpu::XformRecord> xform;  // scenes of at most kBruteMaxTrisPt triangles, else empty
    uint32_t bvh_max_depth = 0;
    bool has_bvh = false;
    lmgpu::DevBuf<lmgpu::ShadeTri> shade;
    lmgpu::DevBuf<lmgpu::MaterialDev> mats;
    lmgpu::DevBuf<lmgpu::LightDev> lights;
    lmgpu::DevBuf<lmgpu::LightTri> light_tris;
    uint32_t num_lights = 0, num_materials = 0;
    std::vector<lmgpu::MaterialDev> host_mats;  // copies for lmgpu_scene_set_params
    std::vector<lmgpu::LightDev> host_lights;
    std::vector<lmgpu::LightTri> host_light_tris;  // the area lights' triangles (camera-connection pixels)
    lmgpu::CameraDev cam{};
    lmgpu::EnvDev env{};

    // Staging of host rays / hits for the trace entry points.
    void* trace_staging = nullptr;
    size_t trace_staging_bytes = 0;
    lmgpu::HostIo* io = nullptr;  // acquired by ensure_pinned
    hipEvent_t io_events[7] = {};
    hipStream_t copy_streams[2] = {nullptr, nullptr};  // their uploads and read-backs
    uint64_t* count_buf = nullptr;  // 2 x u64 for lmgpu_trace_count
    uint32_t* next_counter = nullptr;  // work counter of the persistent traversal kernels
    // This device's address of the static scratch array of lmgpu_trace_closest_noalloc (its
    // work counter), resolved when the context is created; nullptr if that failed.
    uint32_t* noalloc_scratch = nullptr;

    // Path-tracing work buffers (capacity = wavefront width).
    uint32_t pt_capacity = 0;
    void* pt_buf = nullptr;
    size_t pt_buf_bytes = 0;
    void* film_acc = nullptr;
    size_t film_acc_bytes = 0;
    void* film_out_staging = nullptr;
    size_t film_out_staging_bytes = 0;
    void* adj_buf = nullptr;  // adjoint: per-sample Q, gradients, staged dL/dI
    size_t adj_buf_bytes = 0;
    void* splat_buf = nullptr;  // NEE renders: film replicas for the camera vertex's light connections
    size_t splat_buf_bytes = 0;
    void* order_buf = nullptr;  // pt on large scenes: tile keys, sample order and the sort's scratch
    size_t order_buf_bytes = 0;

    // Counting (lmgpu_enable_counting): node visits and triangle tests of the path tracer's
    // BVH stages, extension [0, 2) and shadow [2, 4), in the context's counter block.
    bool counting = false;
    unsigned long long* trav_counts = nullptr;

    // Timing
    bool timing = false;
    double kernel_ms[lmgpu::kKNumClasses] = {};
    uint64_t kernel_launches[lmgpu::kKNumClasses] = {};
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    hipEvent_t run0 = nullptr, run1 = nullptr;  // of a whole render or adjoint
};

namespace lmgpu {

inline BvhDev bvh_of(const lmgpu_ctx* ctx) {
    return BvhDev{ctx->nodes.ptr, ctx->leaf_tris.ptr, ctx->exact_nodes, ctx->reach};
}

// Status helpers: set ctx->err and return a status.
lmgpu_status fail(lmgpu_ctx* ctx, lmgpu_status s, const std::string& msg);
lmgpu_status hip_fail(lmgpu_ctx* ctx, hipError_t e, const char* what);
lmgpu_status dev_alloc(lmgpu_ctx* ctx, void** p, size_t bytes, const char* what);
void dev_free(void* p);

// Grows the context's pinned memory to at least `bytes` (its contents are lost); false if it cannot
// be had.
bool ensure_pinned(lmgpu_ctx* ctx, size_t bytes);
// HostIo::pays of the context's pinned memory.
bool pinned_pays(lmgpu_ctx* ctx, size_t need, double saved_us, double more_us = 0.0);
bool ensure_io_events(lmgpu_ctx* ctx);
constexpr size_t kReadSlot = size_t(2) << 20;
constexpr size_t kReadSlots = 4;
// Whether read_back takes a film of this many bytes through the ring of pinned slots (of at most
// kPinnedWords + kReadSlots * kReadSlot bytes).
bool ring_pays(lmgpu_ctx* ctx, size_t bytes);
// Copies device results to a host array, behind the work on the context's stream; returns when
// they are there.
hipError_t read_back(lmgpu_ctx* ctx, void* dst, const void* src, size_t bytes, bool ring);

// Times `launch` with HIP events on the context stream when timing is enabled.
template <class Fn> hipError_t timed(lmgpu_ctx* ctx, int cls, Fn&& launch) {
    if (!ctx->timing) {
        launch();
        return hipGetLastError();
    }
    (void)hipEventRecord(ctx->ev0, ctx->stream);
    launch();
    hipError_t e = hipGetLastError();
    (void)hipEventRecord(ctx->ev1, ctx->stream);
    (void)hipEventSynchronize(ctx->ev1);
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1);
    ctx->kernel_ms[cls] += double(ms);
    ctx->kernel_launches[cls] += 1;
    return e;
}

// Kernel launchers (trace_kernels.hip, pt_kernels.hip).
// The traversal's nodes and triangle records from the uploaded ones.
hipError_t launch_pack_nodes(lmgpu_ctx* ctx);
// `next`: the work counter of the persistent traversal.
hipError_t launch_trace_closest(lmgpu_ctx* ctx, const float* const* rays, uint32_t n, float* t, float* b0, float* b1,
                                int32_t* prim, bool refine, uint32_t* next);
hipError_t launch_trace_any(lmgpu_ctx* ctx, const float* const* rays, uint32_t n, uint8_t* occluded);
hipError_t launch_trace_count(lmgpu_ctx* ctx, const float* const* rays, uint32_t n, unsigned long long* counts);
lmgpu_status run_pt(lmgpu_ctx* ctx, const lmgpu_pt_params* p, lmgpu_film* film, lmgpu_pt_stats* stats);
lmgpu_status run_pt_backward(lmgpu_ctx* ctx, const lmgpu_pt_params* p, lmgpu_adjoint* adj, lmgpu_pt_stats* stats);
lmgpu_status run_raycast(lmgpu_ctx* ctx, lmgpu_film* film);

}  // namespace lmgpu
