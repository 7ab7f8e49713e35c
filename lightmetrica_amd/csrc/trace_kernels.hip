// Ray-batch traversal kernels behind lmgpu_trace_closest / lmgpu_trace_any / lmgpu_trace_count.
#include "context.hpp"
#include "traverse.hpp"

#include <algorithm>
#include <type_traits>

namespace lmgpu {

struct RaysSoA {
    const float *ox, *oy, *oz, *dx, *dy, *dz, *tmin, *tmax;
};

__device__ __forceinline__ RayIn load_ray(const RaysSoA& r, uint32_t i) {
    RayIn x;
    x.ox = r.ox[i]; x.oy = r.oy[i]; x.oz = r.oz[i];
    x.dx = r.dx[i]; x.dy = r.dy[i]; x.dz = r.dz[i];
    x.tmin = r.tmin[i]; x.tmax = r.tmax[i];
    return x;
}

struct SoASource {
    RaysSoA rays;
    __device__ __forceinline__ RayIn operator()(uint32_t i) const { return load_ray(rays, i); }
};

// How a closest-hit kernel reports the winner: its FP32 weights, or (kRefine) the winner
// re-evaluated in FP64 at once.
template <bool kRefine, class Tri> struct ClosestSink {
    const Tri* tris;
    float *t_out, *b0_out, *b1_out;
    int32_t* prim_out;
    __device__ __forceinline__ void operator()(uint32_t i, bool found, const HitOut& hit, const RayIn& r) const {
        if (found) {
            HitOut h = hit;
            if constexpr (std::is_same_v<Tri, LeafTri>) h = hit_at(tris, hit.rec, r);
            float t, b0, b1;
            winner_barycentrics(tris, r, h, kRefine, t, b0, b1);
            t_out[i] = t;
            b0_out[i] = b0;
            b1_out[i] = b1;
            prim_out[i] = int32_t(h.prim);
        } else {
            t_out[i] = -1.f;
            b0_out[i] = 0.f;
            b1_out[i] = 0.f;
            prim_out[i] = -1;
        }
    }
};

// The winner's leaf-order record (-1 for a miss) alone, for k_refine_fp64 or k_result_fp32 to
// evaluate: the persistent traversal keeps its registers, and occupancy, free of that arithmetic,
// and stores one word per ray from scattered lanes instead of four.
struct RecordSink {
    int32_t* rec_out;
    __device__ __forceinline__ void operator()(uint32_t i, bool found, const HitOut& h, const RayIn&) const {
        rec_out[i] = found ? int32_t(h.rec) : -1;
    }
};

struct OcclusionSink {
    uint8_t* occluded;
    __device__ __forceinline__ void operator()(uint32_t i, bool found, const HitOut&, const RayIn&) const {
        occluded[i] = found ? 1 : 0;
    }
};

// 5 waves per SIMD, as kBatchBlocks asks for.
__global__ __launch_bounds__(kTraceBlock, 5) void k_trace_record(BvhDev bvh, RaysSoA rays,
                                                              uint32_t n, uint32_t* next,
                                                              int32_t* __restrict__ rec_out) {
    __shared__ TraceShared<true> sm;
    SoASource src{rays};
    RecordSink sink{rec_out};
    TraceCounters cnt{0, 0};
    trace_persistent<false, false>(bvh, n, next, sm, src, sink, cnt);
}

__global__ __launch_bounds__(kTraceBlock, 5) void k_trace_any(BvhDev bvh, RaysSoA rays,
                                                           uint32_t n, uint32_t* next, uint8_t* __restrict__ occluded) {
    __shared__ TraceShared<false> sm;
    SoASource src{rays};
    OcclusionSink sink{occluded};
    TraceCounters cnt{0, 0};
    trace_persistent<true, false>(bvh, n, next, sm, src, sink, cnt);
}

// Scenes of at most kBruteMaxTris triangles: every triangle per ray (trace_brute).
template <bool kRefine>
__global__ __launch_bounds__(kTraceBlock) void k_trace_closest_brute(const TriRecord* __restrict__ tris, uint32_t ntris,
                                                                     RaysSoA rays, uint32_t n, float* __restrict__ t_out,
                                                                     float* __restrict__ b0_out, float* __restrict__ b1_out,
                                                                     int32_t* __restrict__ prim_out) {
    SoASource src{rays};
    ClosestSink<kRefine, TriRecord> sink{tris, t_out, b0_out, b1_out, prim_out};
    trace_brute<false>(tris, ntris, n, src, sink);
}

// Small batches, kLanes lanes per ray (trace_grouped): one launch, the FP64 evaluation included.
template <bool kRefine, int kLanes>
__global__ __launch_bounds__(kTraceBlock, 6) void k_trace_closest_grouped(BvhDev bvh, RaysSoA rays, uint32_t n,
                                                                       float* __restrict__ t_out,
                                                                       float* __restrict__ b0_out,
                                                                       float* __restrict__ b1_out,
                                                                       int32_t* __restrict__ prim_out) {
    __shared__ GroupShared<kLanes> sm;
    SoASource src{rays};
    ClosestSink<kRefine, LeafTri> sink{bvh.tris, t_out, b0_out, b1_out, prim_out};
    TraceCounters cnt{0, 0};
    trace_grouped<false, false, kLanes>(bvh, n, sm, src, sink, cnt);
}

template <int kLanes>
__global__ __launch_bounds__(kTraceBlock) void k_trace_any_grouped(BvhDev bvh, RaysSoA rays, uint32_t n,
                                                                   uint8_t* __restrict__ occluded) {
    __shared__ GroupShared<kLanes> sm;
    SoASource src{rays};
    OcclusionSink sink{occluded};
    TraceCounters cnt{0, 0};
    trace_grouped<true, false, kLanes>(bvh, n, sm, src, sink, cnt);
}

// The hits of k_trace_record as the traversal saw them: the same test of the winner gives the same
// t and weights.  Otherwise as k_refine_fp64.  16M rays against 1M triangles, the traversal storing
// all four results: 3.20 ms, with this pass 3.09; 70k to 1M rays the same either way.
__global__ __launch_bounds__(256) void k_result_fp32(const LeafTri* __restrict__ tris, RaysSoA rays, uint32_t n,
                                                     const int32_t* rec_in, float* t_out, float* b0_out,
                                                     float* b1_out, int32_t* prim_out) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    const int32_t rec = __builtin_nontemporal_load(rec_in + i);
    float t = -1.f, b0 = 0.f, b1 = 0.f;
    int32_t prim = -1;
    if (rec >= 0) {
        RayIn r;
        r.ox = __builtin_nontemporal_load(rays.ox + i); r.oy = __builtin_nontemporal_load(rays.oy + i);
        r.oz = __builtin_nontemporal_load(rays.oz + i);
        r.dx = __builtin_nontemporal_load(rays.dx + i); r.dy = __builtin_nontemporal_load(rays.dy + i);
        r.dz = __builtin_nontemporal_load(rays.dz + i);
        r.tmin = __builtin_nontemporal_load(rays.tmin + i);
        r.tmax = __builtin_nontemporal_load(rays.tmax + i);
        const HitOut h = hit_at(tris, uint32_t(rec), r);
        t = h.t;
        b0 = h.b0;
        b1 = h.b1;
        prim = int32_t(h.prim);
    }
    __builtin_nontemporal_store(t, t_out + i);
    __builtin_nontemporal_store(b0, b0_out + i);
    __builtin_nontemporal_store(b1, b1_out + i);
    __builtin_nontemporal_store(prim, prim_out + i);
}

// The hits of k_trace_record, evaluated in FP64 (refine_fp64): rec_in, one of the results' columns,
// holds the leaf-order record of the winner (-1 for a miss).  Only the origin and
// direction of a hit ray are read.  Where the FP64 determinant is 0 the traversal's FP32
// values are computed again.  The streamed arrays are read and written non-temporally, which
// keeps more of the BVH cached for the next traversal (-1.3 % for the pair of kernels on the
// 16M-ray batch).
__global__ __launch_bounds__(256) void k_refine_fp64(const LeafTri* __restrict__ tris, RaysSoA rays, uint32_t n,
                                                     const int32_t* rec_in, float* t_out, float* b0_out,
                                                     float* b1_out, int32_t* prim_out) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    const int32_t rec = __builtin_nontemporal_load(rec_in + i);
    float t = -1.f, b0 = 0.f, b1 = 0.f;
    int32_t prim = -1;
    if (rec >= 0) {
        const float4* tp = reinterpret_cast<const float4*>(tris + rec);
        const float4 v0 = tp[0], v1 = tp[1], v2 = tp[2];
        RayIn r;
        r.ox = __builtin_nontemporal_load(rays.ox + i); r.oy = __builtin_nontemporal_load(rays.oy + i);
        r.oz = __builtin_nontemporal_load(rays.oz + i);
        r.dx = __builtin_nontemporal_load(rays.dx + i); r.dy = __builtin_nontemporal_load(rays.dy + i);
        r.dz = __builtin_nontemporal_load(rays.dz + i);
        r.tmin = 0.f; r.tmax = 0.f;  // not used by refine_fp64
        if (!refine_fp64(r, v0, v1, v2, t, b0, b1)) {
            HitOut h{};
            float U;
            (void)watertight(make_shear_cyclic(r), v0, v1, v2, -INFINITY, INFINITY, h.t, U, h.b0, h.b1, h.det);
            hit_weights(h);
            t = h.t;
            b0 = h.b0;
            b1 = h.b1;
        }
        prim = __float_as_int(v0.w);
    }
    __builtin_nontemporal_store(t, t_out + i);
    __builtin_nontemporal_store(b0, b0_out + i);
    __builtin_nontemporal_store(b1, b1_out + i);
    if (rec >= 0 || rec_in != prim_out) __builtin_nontemporal_store(prim, prim_out + i);
}

__global__ __launch_bounds__(kTraceBlock) void k_trace_any_brute(const TriRecord* __restrict__ tris, uint32_t ntris,
                                                                 RaysSoA rays, uint32_t n,
                                                                 uint8_t* __restrict__ occluded) {
    SoASource src{rays};
    OcclusionSink sink{occluded};
    trace_brute<true>(tris, ntris, n, src, sink);
}

__global__ void k_zero_next(uint32_t* p) {
    if (threadIdx.x == 0) *p = 0u;
}

struct NullSink {
    __device__ __forceinline__ void operator()(uint32_t, bool, const HitOut&, const RayIn&) const {}
};

// The closest-hit kernel's traversal with counters: node visits and triangle tests.
__global__ __launch_bounds__(kTraceBlock) void k_trace_count(BvhDev bvh, RaysSoA rays,
                                                             uint32_t n, uint32_t* next,
                                                             unsigned long long* __restrict__ counts) {
    __shared__ TraceShared<true> sm;
    SoASource src{rays};
    NullSink sink;
    TraceCounters cnt{0, 0};
    trace_persistent<false, true>(bvh, n, next, sm, src, sink, cnt);
    // Wave-level reduction, one atomic per wave per counter.
    unsigned long long a = cnt.nodes, b = cnt.tris;
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_down(a, off, 64);
        b += __shfl_down(b, off, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&counts[0], a);
        atomicAdd(&counts[1], b);
    }
}

// One built node per thread: its leaves' records go to their place (pad, set by place_leaves)
// with the leaf's box beside them, its leaf references follow, and the packed node is written.
__global__ __launch_bounds__(256) void k_pack_nodes(Node4* __restrict__ nodes, const TriRecord* __restrict__ tris,
                                                    NodeQ* __restrict__ packed, LeafTri* __restrict__ leaf_tris,
                                                    uint32_t n) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    Node4 nd = nodes[i];
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const uint32_t c = nd.child[s];
        if (c == kEmptyChild || !(c & kLeafBit)) continue;
        const uint32_t first = c & kMaxLeafFirst, bits = (c >> 27) & 0xfu;
        for (uint32_t k = 0; k <= bits; k++) {
            const float4* src = reinterpret_cast<const float4*>(tris + first + k);
            float4* dst = reinterpret_cast<float4*>(leaf_tris + nd.pad[s] + k);
            float4 v1 = src[1], v2 = src[2];
            v1.w = nd.lo_x[s];
            v2.w = nd.hi_x[s];
            dst[0] = src[0];
            dst[1] = v1;
            dst[2] = v2;
            dst[3] = make_float4(nd.lo_y[s], nd.hi_y[s], nd.lo_z[s], nd.hi_z[s]);
        }
        nd.child[s] = kLeafBit | (bits << 27) | nd.pad[s];
        nodes[i].child[s] = nd.child[s];
    }
    packed[i] = pack_node(nd);
}

// The rays of a batch beyond its first kMaxBatch: larger batches take two launches.
struct RayTail {
    const float* col[8];
    explicit RayTail(const float* const* r) {
        for (int k = 0; k < 8; k++) col[k] = r[k] + kMaxBatch;
    }
};

static RaysSoA soa_of(const float* const* r) { return RaysSoA{r[0], r[1], r[2], r[3], r[4], r[5], r[6], r[7]}; }

// Blocks per CU of a ray batch: incoherent rays share few lines, so beyond five blocks the lines
// of the rays in flight push each other out of L1 and L2 (16M rays: 6 blocks 3.45 ms, 5: 3.29,
// 4: 3.8; 4M any-hit segments 1.42, 1.31, 1.31).
constexpr int kBatchBlocks = 5;

// Persistent grid: every CU filled to its occupancy limit, never more blocks than the batch needs.
template <class K> static uint32_t persistent_blocks(lmgpu_ctx* ctx, K kernel, uint32_t n) {
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kTraceBlock, 0) != hipSuccess || per_cu < 1)
        per_cu = 1;
    per_cu = std::min(per_cu, kBatchBlocks);
    const uint64_t full = uint64_t(std::max(ctx->num_cus, 1)) * uint64_t(per_cu);
    const uint64_t need = (uint64_t(n) + kTraceBlock - 1) / kTraceBlock;
    return uint32_t(std::max<uint64_t>(1, std::min(full, need)));
}

static dim3 group_blocks(uint32_t n, uint32_t lanes) { return dim3((n + kTraceBlock / lanes - 1) / (kTraceBlock / lanes)); }

// Grid of the brute-force kernels: 16 blocks per CU at most, walking the batch.
static uint32_t brute_blocks(lmgpu_ctx* ctx, uint32_t n) {
    const uint64_t need = (uint64_t(n) + kTraceBlock - 1) / kTraceBlock;
    return uint32_t(std::max<uint64_t>(1, std::min<uint64_t>(need, 16ull * uint64_t(std::max(ctx->num_cus, 1)))));
}

hipError_t launch_pack_nodes(lmgpu_ctx* ctx) {
    const uint32_t n = uint32_t(ctx->nodes.count);
    hipLaunchKernelGGL(k_pack_nodes, dim3((n + 255u) / 256u), dim3(256), 0, ctx->stream, ctx->exact_nodes, ctx->tris.ptr,
                       ctx->nodes.ptr, ctx->leaf_tris.ptr, n);
    return hipGetLastError();
}

// The results' column that carries the records from the traversal to the pass after it, which reads the
// rays again: one that lies in none of the rays' (a caller may have its results written over its rays);
// nullptr if there is none.
static int32_t* record_column(const float* const* rays, uint32_t n, float* t, float* b0, float* b1, int32_t* prim) {
    for (void* c : {static_cast<void*>(prim), static_cast<void*>(t), static_cast<void*>(b0), static_cast<void*>(b1)}) {
        const uintptr_t at = reinterpret_cast<uintptr_t>(c), bytes = uintptr_t(n) * 4u;
        bool apart = true;
        for (int k = 0; k < 8; k++) {
            const uintptr_t r = reinterpret_cast<uintptr_t>(rays[k]);
            apart = apart && (at + bytes <= r || r + bytes <= at);
        }
        if (apart) return static_cast<int32_t*>(c);
    }
    return nullptr;
}

hipError_t launch_trace_closest(lmgpu_ctx* ctx, const float* const* rays, uint32_t n, float* t, float* b0, float* b1,
                                int32_t* prim, bool refine, uint32_t* next) {
    if (n > kMaxBatch) {
        const hipError_t e = launch_trace_closest(ctx, rays, kMaxBatch, t, b0, b1, prim, refine, next);
        if (e != hipSuccess) return e;
        return launch_trace_closest(ctx, RayTail(rays).col, n - kMaxBatch, t + kMaxBatch, b0 + kMaxBatch,
                                    b1 + kMaxBatch, prim + kMaxBatch, refine, next);
    }
    const dim3 block(kTraceBlock);
    const uint32_t ntris = ctx->num_records;
    if (ntris <= kBruteMaxTris)
        return timed(ctx, kKTraceClosest, [&]() {
            if (refine)
                hipLaunchKernelGGL(k_trace_closest_brute<true>, dim3(brute_blocks(ctx, n)), block, 0, ctx->stream,
                                   ctx->tris.ptr, ntris, soa_of(rays), n, t, b0, b1, prim);
            else
                hipLaunchKernelGGL(k_trace_closest_brute<false>, dim3(brute_blocks(ctx, n)), block, 0, ctx->stream,
                                   ctx->tris.ptr, ntris, soa_of(rays), n, t, b0, b1, prim);
        });
    int32_t* const rec = record_column(rays, n, t, b0, b1, prim);
    if (n <= kGroup16Closest || !rec)  // the grouped kernels write a ray's results when they have read it
        return timed(ctx, kKTraceClosest, [&]() {
            const bool whole = n <= kGroup64Rays;
            auto kernel = refine ? (whole ? k_trace_closest_grouped<true, 64> : k_trace_closest_grouped<true, 16>)
                                 : (whole ? k_trace_closest_grouped<false, 64> : k_trace_closest_grouped<false, 16>);
            hipLaunchKernelGGL(kernel, group_blocks(n, whole ? 64 : 16), block, 0, ctx->stream, bvh_of(ctx), soa_of(rays),
                               n, t, b0, b1, prim);
        });
    return timed(ctx, kKTraceClosest, [&]() {
        hipLaunchKernelGGL(k_zero_next, dim3(1), dim3(64), 0, ctx->stream, next);
        hipLaunchKernelGGL(k_trace_record, dim3(persistent_blocks(ctx, k_trace_record, n)), block, 0, ctx->stream,
                           bvh_of(ctx), soa_of(rays), n, next, rec);
        hipLaunchKernelGGL(refine ? k_refine_fp64 : k_result_fp32, dim3((n + 255u) / 256u), dim3(256), 0, ctx->stream,
                           ctx->leaf_tris.ptr, soa_of(rays), n, rec, t, b0, b1, prim);
    });
}

hipError_t launch_trace_any(lmgpu_ctx* ctx, const float* const* rays, uint32_t n, uint8_t* occluded) {
    if (n > kMaxBatch) {
        const hipError_t e = launch_trace_any(ctx, rays, kMaxBatch, occluded);
        if (e != hipSuccess) return e;
        return launch_trace_any(ctx, RayTail(rays).col, n - kMaxBatch, occluded + kMaxBatch);
    }
    uint32_t* next = ctx->next_counter;
    const uint32_t ntris = ctx->num_records;
    if (ntris <= kBruteMaxTris)
        return timed(ctx, kKTraceAny, [&]() {
            hipLaunchKernelGGL(k_trace_any_brute, dim3(brute_blocks(ctx, n)), dim3(kTraceBlock), 0, ctx->stream,
                               ctx->tris.ptr, ntris, soa_of(rays), n, occluded);
        });
    if (n <= kGroup16Any)
        return timed(ctx, kKTraceAny, [&]() {
            const bool whole = n <= kGroup64Rays;
            auto kernel = whole ? k_trace_any_grouped<64> : k_trace_any_grouped<16>;
            hipLaunchKernelGGL(kernel, group_blocks(n, whole ? 64 : 16), dim3(kTraceBlock), 0, ctx->stream, bvh_of(ctx),
                               soa_of(rays), n, occluded);
        });
    return timed(ctx, kKTraceAny, [&]() {
        hipLaunchKernelGGL(k_zero_next, dim3(1), dim3(64), 0, ctx->stream, next);
        hipLaunchKernelGGL(k_trace_any, dim3(persistent_blocks(ctx, k_trace_any, n)), dim3(kTraceBlock), 0,
                           ctx->stream, bvh_of(ctx), soa_of(rays), n, next, occluded);
    });
}

hipError_t launch_trace_count(lmgpu_ctx* ctx, const float* const* rays, uint32_t n, unsigned long long* counts) {
    if (n > kMaxBatch) {
        const hipError_t e = launch_trace_count(ctx, rays, kMaxBatch, counts);
        if (e != hipSuccess) return e;
        return launch_trace_count(ctx, RayTail(rays).col, n - kMaxBatch, counts);
    }
    uint32_t* next = ctx->next_counter;
    hipLaunchKernelGGL(k_zero_next, dim3(1), dim3(64), 0, ctx->stream, next);
    hipLaunchKernelGGL(k_trace_count, dim3(persistent_blocks(ctx, k_trace_count, n)), dim3(kTraceBlock), 0, ctx->stream,
                       bvh_of(ctx), soa_of(rays), n, next, counts);
    return hipGetLastError();
}

}  // namespace lmgpu
