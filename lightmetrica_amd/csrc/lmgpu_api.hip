// C ABI of the MI355X path-tracing hot path (include/lmgpu.h).
#include "context.hpp"
#include "traverse.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <new>
#include <vector>

using namespace lmgpu;

// Scratch of lmgpu_trace_closest_noalloc: word 0 is the persistent traversal's work counter,
// the rest pads the array to 256 B.  Every GPU the library runs on holds its own copy until
// the process ends.  In host code `scratch` names a host-side stand-in, never a device
// address: kernels and copies get this device's address from noalloc_scratch_address().
static __device__ __align__(256) uint32_t scratch[64];

namespace {

// Per-device addresses of `scratch`, resolved once per device with that device current.
std::mutex g_scratch_mutex;
std::vector<uint32_t*> g_scratch_addr;

hipError_t noalloc_scratch_address(int device, uint32_t** out) {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    *out = nullptr;
    if (device < 0) return hipErrorInvalidDevice;
    if (size_t(device) >= g_scratch_addr.size()) g_scratch_addr.resize(size_t(device) + 1, nullptr);
    if (!g_scratch_addr[device]) {
        void* p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        g_scratch_addr[device] = static_cast<uint32_t*>(p);
    }
    *out = g_scratch_addr[device];
    return hipSuccess;
}

}  // namespace

namespace lmgpu {

lmgpu_status fail(lmgpu_ctx* ctx, lmgpu_status s, const std::string& msg) {
    if (ctx) ctx->err = msg;
    return s;
}

lmgpu_status hip_fail(lmgpu_ctx* ctx, hipError_t e, const char* what) {
    return fail(ctx, LMGPU_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
}

lmgpu_status dev_alloc(lmgpu_ctx* ctx, void** p, size_t bytes, const char* what) {
    *p = nullptr;
    if (ctx->inject_alloc_failures > 0) {
        ctx->inject_alloc_failures--;
        return fail(ctx, LMGPU_ERR_INJECTED, std::string("injected allocation failure: ") + what);
    }
    hipError_t e = hipMalloc(p, std::max<size_t>(bytes, 16));
    if (e != hipSuccess) {
        *p = nullptr;
        return fail(ctx, LMGPU_ERR_OUT_OF_MEMORY, std::string("hipMalloc failed for ") + what + ": " + hipGetErrorString(e));
    }
    return LMGPU_OK;
}

void dev_free(void* p) {
    if (p) (void)hipFree(p);
}

static HostIoPool g_host_io_pool;
void host_io_context() { g_host_io_pool.context(); }
HostIo* host_io_acquire() { return g_host_io_pool.acquire(); }
void host_io_release(HostIo* io) {
    HostIo* gone[kIdleIos + 1];
    const size_t n = g_host_io_pool.release(io, gone);
    for (size_t k = 0; k < n; k++) {
        if (gone[k]->pinned) (void)hipHostFree(gone[k]->pinned);
        delete gone[k];
    }
}

bool pinned_pays(lmgpu_ctx* ctx, size_t need, double saved_us, double more_us) {
    if (!ctx->io && !(ctx->io = host_io_acquire())) return false;
    return ctx->io->pays(need, saved_us, more_us);
}

bool ensure_pinned(lmgpu_ctx* ctx, size_t bytes) {
    if (!ctx->io && !(ctx->io = host_io_acquire())) return false;
    HostIo& io = *ctx->io;
    if (bytes <= io.bytes) return true;
    size_t room = size_t(64) << 10;  // small needs in powers of two, to grow seldom
    while (room < bytes && room < (size_t(4) << 20)) room *= 2;
    bytes = std::max(bytes, room);
    if (io.pinned) (void)hipHostFree(io.pinned);
    io.pinned = nullptr;
    io.bytes = 0;
    void* p = nullptr;
    if (hipHostMalloc(&p, bytes, hipHostMallocPortable) != hipSuccess || !p) {
        (void)hipGetLastError();
        return false;
    }
    io.pinned = p;
    io.bytes = bytes;
    return true;
}

bool ensure_io_events(lmgpu_ctx* ctx) {
    for (hipEvent_t& ev : ctx->io_events)
        if (!ev && hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess) {
            ev = nullptr;
            (void)hipGetLastError();
            return false;
        }
    return true;
}

// Results on their way to the caller: a ring of kReadSlots pinned slots of kReadSlot bytes, each
// copied out by the host threads while the next ones are on the link (57 GB/s).  Into pageable
// memory the runtime copies with one thread: the FP64 film of a 1920 x 1080 render (50 MB) took
// 4.8 ms, 1 to 3 so (the caller's pages are made on the way); a raycast of 1280 x 720 (11 MB), its
// kernel included, 0.89 -> 0.51 ms.  Slots of 512 KB: 0.83 ms, a copy has its own cost on the link.
// Fewer bytes than this are left to the runtime, which maps the caller's pages at once: raycasts of
// 133, 537 and 1004 KB take 38, 66 and 91 us so, 45, 83 and 101 through the ring; 1312 KB 121 and
// 108, 1735 KB 139 and 126.
constexpr size_t kRingFrom = size_t(1152) << 10;
bool ring_pays(lmgpu_ctx* ctx, size_t bytes) {
    // 36 us a MiB saved by the raycast above, 90 by the film of 50 MB.
    return bytes >= kRingFrom && pinned_pays(ctx, kPinnedWords + std::min(bytes, kReadSlots * kReadSlot),
                                             double(bytes) * (36.0 / (1 << 20)));
}

hipError_t read_back(lmgpu_ctx* ctx, void* dst, const void* src, size_t bytes, bool ring) {
    const hipStream_t s = ctx->stream;
    const size_t chunks = (bytes + kReadSlot - 1) / kReadSlot;
    if (!ring || !ensure_pinned(ctx, kPinnedWords + std::min(bytes, kReadSlots * kReadSlot)) || !ensure_io_events(ctx)) {
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
        return e == hipSuccess ? hipStreamSynchronize(s) : e;
    }
    char* pin = static_cast<char*>(ctx->io->pinned) + kPinnedWords;
    auto size = [&](size_t c) { return std::min(kReadSlot, bytes - c * kReadSlot); };
    size_t sent = 0;
    hipError_t e = hipSuccess;
    for (size_t c = 0; c < chunks && e == hipSuccess; c++) {
        for (; sent < chunks && sent < c + kReadSlots && e == hipSuccess; sent++) {
            e = hipMemcpyAsync(pin + sent % kReadSlots * kReadSlot, static_cast<const char*>(src) + sent * kReadSlot,
                               size(sent), hipMemcpyDeviceToHost, s);
            if (e == hipSuccess) e = hipEventRecord(ctx->io_events[sent % kReadSlots], s);
        }
        if (e == hipSuccess) e = hipEventSynchronize(ctx->io_events[c % kReadSlots]);
        if (e != hipSuccess) break;
        const CopyJob job{static_cast<char*>(dst) + c * kReadSlot, pin + c % kReadSlots * kReadSlot, size(c)};
        ctx->io->team.run(&job, 1);
    }
    if (e != hipSuccess) (void)hipStreamSynchronize(s);
    return e;
}

}  // namespace lmgpu

namespace {

template <class T> void free_buf(DevBuf<T>& b) {
    dev_free(b.ptr);
    b.ptr = nullptr;
    b.count = 0;
}

template <class T> lmgpu_status upload(lmgpu_ctx* ctx, DevBuf<T>& b, const T* src, size_t count, const char* what) {
    free_buf(b);
    void* p = nullptr;
    lmgpu_status s = dev_alloc(ctx, &p, sizeof(T) * count, what);
    if (s != LMGPU_OK) return s;
    b.ptr = static_cast<T*>(p);
    b.count = count;
    if (count) {
        hipError_t e = hipMemcpyAsync(b.ptr, src, sizeof(T) * count, hipMemcpyHostToDevice, ctx->stream);
        if (e != hipSuccess) return hip_fail(ctx, e, what);
        e = hipStreamSynchronize(ctx->stream);
        if (e != hipSuccess) return hip_fail(ctx, e, what);
    }
    return LMGPU_OK;
}

// 4x4 inverse (column-major) by Gauss-Jordan elimination in double, rounded to float.
bool invert4(const float* m, float* out) {
    double a[4][8];
    for (int r = 0; r < 4; r++) {
        for (int c = 0; c < 4; c++) a[r][c] = m[c * 4 + r];
        for (int c = 0; c < 4; c++) a[r][4 + c] = r == c ? 1.0 : 0.0;
    }
    for (int c = 0; c < 4; c++) {
        int piv = c;
        for (int r = c + 1; r < 4; r++)
            if (std::fabs(a[r][c]) > std::fabs(a[piv][c])) piv = r;
        if (a[piv][c] == 0.0) return false;
        for (int k = 0; k < 8; k++) std::swap(a[c][k], a[piv][k]);
        const double inv = 1.0 / a[c][c];
        for (int k = 0; k < 8; k++) a[c][k] *= inv;
        for (int r = 0; r < 4; r++) {
            if (r == c) continue;
            const double f = a[r][c];
            for (int k = 0; k < 8; k++) a[r][k] -= f * a[c][k];
        }
    }
    for (int r = 0; r < 4; r++)
        for (int c = 0; c < 4; c++) out[c * 4 + r] = float(a[r][4 + c]);
    return true;
}

void mul4h(const float* M, const float v[4], float o[4]) {
    for (int r = 0; r < 4; r++) o[r] = M[r] * v[0] + M[4 + r] * v[1] + M[8 + r] * v[2] + M[12 + r] * v[3];
}

// PerspectiveCamera::Load (perspectivecamera.cpp:97-172) and RegisterPrimitives (:174-184).
bool setup_camera(const lmgpu_camera& in, CameraDev& cam) {
    if (in.width == 0 || in.height == 0) return false;
    std::memcpy(cam.view.m, in.view, sizeof(float) * 16);
    if (!invert4(cam.view.m, cam.inv_view.m)) return false;
    const float aspect = float(in.width) / float(in.height);
    const float rad = in.fovy_deg * 3.14159265358979323846f / 180.f;
    const float t = std::tan(float(rad / 2.f));
    const float zn = 1.f, zf = 1000.f;
    float* P = cam.proj.m;
    std::memset(P, 0, sizeof(float) * 16);
    P[0] = 1.f / (aspect * t);
    P[5] = 1.f / t;
    P[10] = -(zf + zn) / (zf - zn);
    P[11] = -1.f;
    P[14] = -(2.f * zf * zn) / (zf - zn);
    if (!invert4(cam.proj.m, cam.inv_proj.m)) return false;
    const float o[4] = {0.f, 0.f, 0.f, 1.f};
    float pw[4];
    mul4h(cam.inv_view.m, o, pw);
    cam.pos[0] = pw[0];
    cam.pos[1] = pw[1];
    cam.pos[2] = pw[2];
    const float n1[4] = {-1.f, -1.f, 0.f, 1.f}, n2[4] = {1.f, 1.f, 0.f, 1.f};
    float c1[4], c2[4];
    mul4h(cam.inv_proj.m, n1, c1);
    mul4h(cam.inv_proj.m, n2, c2);
    // The reference divides both corners by the first corner's w (perspectivecamera.cpp:162-163).
    float p1[3] = {c1[0] / c1[3], c1[1] / c1[3], c1[2] / c1[3]};
    float p2[3] = {c2[0] / c1[3], c2[1] / c1[3], c2[2] / c1[3]};
    const float z1 = p1[2], z2 = p2[2];
    for (int k = 0; k < 3; k++) { p1[k] /= z1; p2[k] /= z2; }
    const float A = (p2[0] - p1[0]) * (p2[1] - p1[1]);
    cam.inv_A = 1.f / A;
    cam.width = int(in.width);
    cam.height = int(in.height);
    return true;
}

}  // namespace

extern "C" {

int lmgpu_abi_version(void) { return LMGPU_ABI_VERSION; }

lmgpu_status lmgpu_create(int device, lmgpu_ctx** out) {
    if (!out) return LMGPU_ERR_INVALID_ARGUMENT;
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || device < 0 || device >= n) return LMGPU_ERR_INVALID_ARGUMENT;
    lmgpu_ctx* ctx = new (std::nothrow) lmgpu_ctx();
    if (!ctx) return LMGPU_ERR_OUT_OF_MEMORY;
    ctx->device = device;
    hipError_t e = hipSetDevice(device);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&ctx->own_stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreate(&ctx->ev0);
    if (e == hipSuccess) e = hipEventCreate(&ctx->ev1);
    if (e == hipSuccess) e = hipEventCreate(&ctx->run0);
    if (e == hipSuccess) e = hipEventCreate(&ctx->run1);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&ctx->num_cus, hipDeviceAttributeMultiprocessorCount, device);
    if (e != hipSuccess) {
        delete ctx;
        return LMGPU_ERR_HIP;
    }
    host_io_context();
    ctx->stream = ctx->own_stream;
    ctx->env.index = -1;
    void* counters = nullptr;
    if (hipMalloc(&counters, 256) != hipSuccess) {
        lmgpu_destroy(ctx);
        return LMGPU_ERR_OUT_OF_MEMORY;
    }
    // 256 B of counters: [0, 16) lmgpu_trace_count, [64, 96) lmgpu_traversal_counts, [128, 132) the
    // persistent traversal's work counter.
    ctx->count_buf = static_cast<uint64_t*>(counters);
    ctx->trav_counts = reinterpret_cast<unsigned long long*>(static_cast<char*>(counters) + 64);
    ctx->next_counter = reinterpret_cast<uint32_t*>(static_cast<char*>(counters) + 128);
    // The device is current (hipSetDevice above).  A failure only disables
    // lmgpu_trace_closest_noalloc, which reports it.
    uint32_t* sp = nullptr;
    if (noalloc_scratch_address(device, &sp) == hipSuccess) ctx->noalloc_scratch = sp;
    *out = ctx;
    return LMGPU_OK;
}

lmgpu_status lmgpu_destroy(lmgpu_ctx* ctx) {
    if (!ctx) return LMGPU_ERR_INVALID_ARGUMENT;
    (void)hipSetDevice(ctx->device);
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    free_buf(ctx->nodes);
    free_buf(ctx->tris);
    free_buf(ctx->xform);
    free_buf(ctx->shade);
    free_buf(ctx->mats);
    free_buf(ctx->lights);
    free_buf(ctx->light_tris);
    dev_free(ctx->trace_staging);
    for (hipEvent_t ev : ctx->io_events)
        if (ev) (void)hipEventDestroy(ev);
    for (hipStream_t cs : ctx->copy_streams)
        if (cs) (void)hipStreamDestroy(cs);
    dev_free(ctx->count_buf);
    dev_free(ctx->pt_buf);
    dev_free(ctx->film_acc);
    dev_free(ctx->film_out_staging);
    dev_free(ctx->adj_buf);
    dev_free(ctx->splat_buf);
    dev_free(ctx->order_buf);
    if (ctx->ev0) (void)hipEventDestroy(ctx->ev0);
    if (ctx->ev1) (void)hipEventDestroy(ctx->ev1);
    if (ctx->run0) (void)hipEventDestroy(ctx->run0);
    if (ctx->run1) (void)hipEventDestroy(ctx->run1);
    if (ctx->own_stream) (void)hipStreamDestroy(ctx->own_stream);
    host_io_release(ctx->io);
    delete ctx;
    return LMGPU_OK;
}

const char* lmgpu_last_error(const lmgpu_ctx* ctx) { return ctx ? ctx->err.c_str() : "null context"; }

lmgpu_status lmgpu_set_stream(lmgpu_ctx* ctx, void* hip_stream) {
    if (!ctx) return LMGPU_ERR_INVALID_ARGUMENT;
    ctx->stream = hip_stream ? static_cast<hipStream_t>(hip_stream) : ctx->own_stream;
    return LMGPU_OK;
}

lmgpu_status lmgpu_synchronize(lmgpu_ctx* ctx) {
    if (!ctx) return LMGPU_ERR_INVALID_ARGUMENT;
    hipError_t e = hipStreamSynchronize(ctx->stream);
    return e == hipSuccess ? LMGPU_OK : hip_fail(ctx, e, "synchronize");
}

lmgpu_status lmgpu_inject_alloc_failures(lmgpu_ctx* ctx, int n) {
    if (!ctx || n < 0) return LMGPU_ERR_INVALID_ARGUMENT;
    ctx->inject_alloc_failures = n;
    return LMGPU_OK;
}

lmgpu_status lmgpu_scene_upload(lmgpu_ctx* ctx, const lmgpu_scene_desc* d) {
    if (!ctx) return LMGPU_ERR_INVALID_ARGUMENT;
    if (!d || !d->positions || !d->faces || d->num_vertices == 0 || d->num_triangles == 0)
        return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_scene_upload: positions and faces are required");
    (void)hipSetDevice(ctx->device);
    const uint32_t nv = d->num_vertices, nf = d->num_triangles;
    for (size_t k = 0; k < size_t(nf) * 3; k++)
        if (d->faces[k] >= nv) return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_scene_upload: face index out of range");
    const bool shading = d->material_ids != nullptr;
    if (shading) {
        if (!d->normals || !d->materials || d->num_materials == 0)
            return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_scene_upload: materials need normals and a material table");
        for (uint32_t t = 0; t < nf; t++) {
            if (d->material_ids[t] >= d->num_materials)
                return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_scene_upload: material id out of range");
            if (d->light_ids && (d->light_ids[t] < -1 || d->light_ids[t] >= int32_t(d->num_lights)))
                return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_scene_upload: light id out of range");
        }
        for (uint32_t m = 0; m < d->num_materials; m++)
            if (d->materials[m].type > LMGPU_BSDF_DIFFUSEMIRROR)
                return fail(ctx, LMGPU_ERR_UNSUPPORTED, "lmgpu_scene_upload: unsupported BSDF type");
    }
    int env_count = 0;
    for (uint32_t l = 0; l < d->num_lights; l++) {
        if (d->lights[l].type > LMGPU_LIGHT_ENV_CONST)
            return fail(ctx, LMGPU_ERR_UNSUPPORTED, "lmgpu_scene_upload: unsupported light type");
        if (d->lights[l].type == LMGPU_LIGHT_ENV_CONST) env_count++;
    }
    if (env_count > 1) return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_scene_upload: at most one environment light");

    ctx->positions.assign(d->positions, d->positions + size_t(nv) * 3);
    ctx->faces.assign(d->faces, d->faces + size_t(nf) * 3);
    ctx->num_vertices = nv;
    ctx->num_triangles = nf;
    ctx->has_bvh = false;
    ctx->has_shading = false;
    ctx->has_camera = false;
    ctx->has_scene = true;
    free_buf(ctx->nodes);
    free_buf(ctx->tris);
    free_buf(ctx->xform);

    if (d->camera) {
        if (!setup_camera(*d->camera, ctx->cam))
            return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_scene_upload: invalid camera");
        ctx->has_camera = true;
    }
    if (!shading) return LMGPU_OK;

    const float* P = d->positions;
    const float* N = d->normals;
    std::vector<ShadeTri> st(nf);
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (uint32_t t = 0; t < nf; t++) {
        const uint32_t a = d->faces[3 * t], b = d->faces[3 * t + 1], c = d->faces[3 * t + 2];
        const float* p1 = P + 3 * size_t(a);
        const float* p2 = P + 3 * size_t(b);
        const float* p3 = P + 3 * size_t(c);
        for (int k = 0; k < 3; k++) {
            lo[k] = std::min({lo[k], p1[k], p2[k], p3[k]});
            hi[k] = std::max({hi[k], p1[k], p2[k], p3[k]});
        }
        const float e1[3] = {p2[0] - p1[0], p2[1] - p1[1], p2[2] - p1[2]};
        const float e2[3] = {p3[0] - p1[0], p3[1] - p1[1], p3[2] - p1[2]};
        float g[3] = {e1[1] * e2[2] - e1[2] * e2[1], e1[2] * e2[0] - e1[0] * e2[2], e1[0] * e2[1] - e1[1] * e2[0]};
        const float len = std::sqrt(g[0] * g[0] + g[1] * g[1] + g[2] * g[2]);
        ShadeTri& s = st[t];
        for (int k = 0; k < 3; k++) {
            s.gn[k] = len > 0.f ? g[k] / len : 0.f;
            s.n1[k] = N[3 * size_t(a) + k];
            s.n2[k] = N[3 * size_t(b) + k];
            s.n3[k] = N[3 * size_t(c) + k];
        }
        s.mat = d->material_ids[t];
        s.light = d->light_ids ? d->light_ids[t] : -1;
        s.pad0 = s.pad1 = 0.f;
    }
    lmgpu_status s = upload(ctx, ctx->shade, st.data(), st.size(), "shading records");
    if (s != LMGPU_OK) return s;
    std::vector<MaterialDev> mats(d->num_materials);
    for (uint32_t m = 0; m < d->num_materials; m++) {
        mats[m].type = d->materials[m].type;
        for (int k = 0; k < 3; k++) mats[m].R[k] = d->materials[m].R[k];
    }
    s = upload(ctx, ctx->mats, mats.data(), mats.size(), "materials");
    if (s != LMGPU_OK) return s;

    // Lights: area-light CDFs (light.area.cpp:109-144) and the environment sphere
    // (light.env.const.cpp:88-98 over Scene::GetAABB = triangles + camera, scene.cpp:58-65).
    std::vector<LightDev> lights(d->num_lights);
    std::vector<LightTri> ltris;
    ctx->env.index = -1;
    for (uint32_t l = 0; l < d->num_lights; l++) {
        LightDev& L = lights[l];
        std::memset(&L, 0, sizeof(L));
        L.type = d->lights[l].type;
        for (int k = 0; k < 3; k++) L.Le[k] = d->lights[l].Le[k];
        if (L.type == LMGPU_LIGHT_ENV_CONST) {
            ctx->env.index = int(l);
            continue;
        }
        L.tri_begin = uint32_t(ltris.size());
        std::vector<float> cdf(1, 0.f);
        size_t first = ltris.size();
        for (uint32_t t = 0; t < nf; t++) {
            if (!d->light_ids || d->light_ids[t] != int32_t(l)) continue;
            const float* p1 = P + 3 * size_t(d->faces[3 * t]);
            const float* p2 = P + 3 * size_t(d->faces[3 * t + 1]);
            const float* p3 = P + 3 * size_t(d->faces[3 * t + 2]);
            LightTri lt;
            for (int k = 0; k < 3; k++) { lt.p1[k] = p1[k]; lt.p2[k] = p2[k]; lt.p3[k] = p3[k]; }
            lt.p3[3] = 0.f;
            const float e1[3] = {p2[0] - p1[0], p2[1] - p1[1], p2[2] - p1[2]};
            const float e2[3] = {p3[0] - p1[0], p3[1] - p1[1], p3[2] - p1[2]};
            const float cx = e1[1] * e2[2] - e1[2] * e2[1], cy = e1[2] * e2[0] - e1[0] * e2[2],
                        cz = e1[0] * e2[1] - e1[1] * e2[0];
            const float area = std::sqrt(cx * cx + cy * cy + cz * cz) / 2.f;
            cdf.push_back(cdf.back() + area);
            ltris.push_back(lt);
        }
        L.tri_count = uint32_t(ltris.size() - first);
        if (L.tri_count == 0)
            return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_scene_upload: area light without triangles");
        const float total = cdf.back();
        L.inv_area = 1.f / total;
        for (float& v : cdf) v *= L.inv_area;
        for (uint32_t k = 0; k < L.tri_count; k++) {
            ltris[first + k].p1[3] = cdf[k];
            ltris[first + k].p2[3] = cdf[k + 1];
        }
    }
    ctx->num_lights = d->num_lights;
    ctx->num_materials = d->num_materials;
    s = upload(ctx, ctx->lights, lights.data(), lights.size(), "lights");
    if (s != LMGPU_OK) return s;
    s = upload(ctx, ctx->light_tris, ltris.data(), ltris.size(), "light triangles");
    if (s != LMGPU_OK) return s;
    if (ctx->env.index >= 0) {
        if (!ctx->has_camera)
            return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_scene_upload: an environment light needs the camera");
        float blo[3], bhi[3];
        for (int k = 0; k < 3; k++) {
            blo[k] = std::min(lo[k], ctx->cam.pos[k]);
            bhi[k] = std::max(hi[k], ctx->cam.pos[k]);
        }
        float r2 = 0.f;
        for (int k = 0; k < 3; k++) {
            ctx->env.center[k] = (bhi[k] + blo[k]) / 2.f;
            const float dk = ctx->env.center[k] - bhi[k];
            r2 += dk * dk;
        }
        ctx->env.radius = std::sqrt(r2);
        for (int k = 0; k < 3; k++) ctx->env.Le[k] = d->lights[ctx->env.index].Le[k];
        const float area = 4.f * 3.14159265358979323846f * ctx->env.radius * ctx->env.radius;
        ctx->env.inv_area = 1.f / area;
        lights[size_t(ctx->env.index)].inv_area = ctx->env.inv_area;
        s = upload(ctx, ctx->lights, lights.data(), lights.size(), "lights");
        if (s != LMGPU_OK) return s;
    }
    if (!ctx->has_camera) return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_scene_upload: shading scenes need a camera");
    ctx->host_mats = std::move(mats);
    ctx->host_lights = std::move(lights);
    ctx->host_light_tris = std::move(ltris);
    ctx->has_shading = true;
    return LMGPU_OK;
}

lmgpu_status lmgpu_scene_set_params(lmgpu_ctx* ctx, const float* albedo, const float* emission) {
    if (!ctx) return LMGPU_ERR_INVALID_ARGUMENT;
    if (!ctx->has_shading) return fail(ctx, LMGPU_ERR_NO_SCENE, "lmgpu_scene_set_params: no shading scene");
    (void)hipSetDevice(ctx->device);
    for (size_t i = 0; albedo && i < ctx->host_mats.size(); i++)
        for (int k = 0; k < 3; k++) {
            const float v = albedo[3 * i + k];
            if (!(v >= 0.f) || !std::isfinite(v))
                return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_scene_set_params: reflectance must be finite and >= 0");
        }
    for (size_t i = 0; emission && i < ctx->host_lights.size(); i++)
        for (int k = 0; k < 3; k++) {
            const float v = emission[3 * i + k];
            if (!(v >= 0.f) || !std::isfinite(v))
                return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_scene_set_params: emission must be finite and >= 0");
        }
    hipError_t e = hipSuccess;
    if (albedo) {
        for (size_t i = 0; i < ctx->host_mats.size(); i++)
            for (int k = 0; k < 3; k++) ctx->host_mats[i].R[k] = albedo[3 * i + k];
        e = hipMemcpyAsync(ctx->mats.ptr, ctx->host_mats.data(), ctx->host_mats.size() * sizeof(MaterialDev),
                           hipMemcpyHostToDevice, ctx->stream);
    }
    if (e == hipSuccess && emission) {
        for (size_t i = 0; i < ctx->host_lights.size(); i++)
            for (int k = 0; k < 3; k++) ctx->host_lights[i].Le[k] = emission[3 * i + k];
        if (ctx->env.index >= 0)
            for (int k = 0; k < 3; k++) ctx->env.Le[k] = emission[3 * size_t(ctx->env.index) + k];
        e = hipMemcpyAsync(ctx->lights.ptr, ctx->host_lights.data(), ctx->host_lights.size() * sizeof(LightDev),
                           hipMemcpyHostToDevice, ctx->stream);
    }
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) return hip_fail(ctx, e, "lmgpu_scene_set_params");
    return LMGPU_OK;
}

lmgpu_status lmgpu_bvh_build(lmgpu_ctx* ctx, const lmgpu_bvh_params* params, lmgpu_bvh_info* info) {
    if (!ctx) return LMGPU_ERR_INVALID_ARGUMENT;
    if (!ctx->has_scene) return fail(ctx, LMGPU_ERR_NO_SCENE, "lmgpu_bvh_build: upload a scene first");
    (void)hipSetDevice(ctx->device);
    BuildParams bp;
    if (params) {
        bp.max_leaf_size = params->max_leaf_size ? params->max_leaf_size : 4;
        bp.bins = params->sah_bins ? params->sah_bins : 64;
        bp.traversal_cost = params->traversal_cost > 0.f ? params->traversal_cost : 1.2f;
        bp.num_threads = params->num_threads;
    }
    WideBVH w;
    std::string err;
    if (!build_wide_bvh(ctx->positions.data(), ctx->num_vertices, ctx->faces.data(), ctx->num_triangles, bp, w, err))
        return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_bvh_build: " + err);
    if (3u * w.max_depth > 96u)
        return fail(ctx, LMGPU_ERR_BVH_TOO_DEEP, "lmgpu_bvh_build: tree depth " + std::to_string(w.max_depth) +
                                                     " exceeds the traversal stack (max 32)");
    ctx->has_bvh = false;
    // Nodes and records go up as they are built and are packed and placed on the device.
    const size_t nn = w.nodes.size(), nt = place_leaves(w);
    const size_t packed_bytes = sizeof(NodeQ) * nn, exact_bytes = sizeof(Node4) * nn, leaf_bytes = sizeof(LeafTri) * nt;
    free_buf(ctx->nodes);
    free_buf(ctx->tris);
    void* block = nullptr;
    const size_t packed_pad = (packed_bytes + 127) / 128 * 128;
    lmgpu_status s = dev_alloc(ctx, &block, packed_pad + exact_bytes + leaf_bytes, "BVH");
    if (s != LMGPU_OK) return s;
    ctx->nodes.ptr = static_cast<NodeQ*>(block);
    ctx->nodes.count = nn;
    ctx->exact_nodes = reinterpret_cast<Node4*>(static_cast<char*>(block) + packed_pad);
    ctx->leaf_tris = {reinterpret_cast<LeafTri*>(static_cast<char*>(block) + packed_pad + exact_bytes), nt};
    ctx->num_records = uint32_t(w.tris.size());
    hipError_t e = hipMemcpyAsync(ctx->exact_nodes, w.nodes.data(), exact_bytes, hipMemcpyHostToDevice, ctx->stream);
    if (e != hipSuccess) return hip_fail(ctx, e, "BVH nodes");
    s = upload(ctx, ctx->tris, w.tris.data(), w.tris.size(), "triangle records");
    if (s != LMGPU_OK) return s;
    e = launch_pack_nodes(ctx);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) return hip_fail(ctx, e, "k_pack_nodes");
    if (w.tris.size() > kBruteMaxTris) free_buf(ctx->tris);
    ctx->reach = 0.f;
    const Node4& root = w.nodes[0];
    for (int i = 0; i < 4; i++) {
        if (root.child[i] == kEmptyChild) continue;
        for (float v : {root.lo_x[i], root.hi_x[i], root.lo_y[i], root.hi_y[i], root.lo_z[i], root.hi_z[i]})
            ctx->reach = std::max(ctx->reach, std::fabs(v));
    }
    // The path tracer of a scene small enough to test every triangle per ray tests the
    // triangles' transform records.
    free_buf(ctx->xform);
    if (w.tris.size() <= kBruteMaxTrisPt) {
        const std::vector<XformRecord> x = make_xform_records(w.tris);
        s = upload(ctx, ctx->xform, x.data(), x.size(), "triangle transform records");
        if (s != LMGPU_OK) return s;
    }
    ctx->bvh_max_depth = w.max_depth;
    ctx->has_bvh = true;
    if (info) {
        info->num_nodes = uint32_t(w.nodes.size());
        info->num_leaves = w.num_leaves;
        info->max_depth = w.max_depth;
        info->num_tri_records = uint32_t(w.tris.size());
        info->build_seconds = w.build_seconds;
        info->sah_cost = w.sah_cost;
        info->device_bytes = uint64_t(packed_bytes + exact_bytes + leaf_bytes);
    }
    return LMGPU_OK;
}

}  // extern "C"

namespace {

// Host rays are staged into one device allocation: 8 input arrays + 4 output arrays.
lmgpu_status stage(lmgpu_ctx* ctx, size_t bytes) {
    if (bytes <= ctx->trace_staging_bytes) return LMGPU_OK;
    dev_free(ctx->trace_staging);
    ctx->trace_staging = nullptr;
    ctx->trace_staging_bytes = 0;
    lmgpu_status s = dev_alloc(ctx, &ctx->trace_staging, bytes, "ray staging");
    if (s != LMGPU_OK) return s;
    ctx->trace_staging_bytes = bytes;
    return LMGPU_OK;
}

lmgpu_status prepare_rays(lmgpu_ctx* ctx, const lmgpu_rays_soa* rays, uint32_t n, size_t out_bytes,
                          const float* dev[8], char** out_base) {
    const float* src[8] = {rays->ox, rays->oy, rays->oz, rays->dx, rays->dy, rays->dz, rays->tmin, rays->tmax};
    for (int k = 0; k < 8; k++)
        if (!src[k]) return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "ray array is NULL");
    const size_t in_bytes = rays->device ? 0 : size_t(n) * 4 * 8;
    lmgpu_status s = stage(ctx, in_bytes + out_bytes);
    if (s != LMGPU_OK) return s;
    char* base = static_cast<char*>(ctx->trace_staging);
    if (rays->device) {
        for (int k = 0; k < 8; k++) dev[k] = src[k];
        *out_base = base;
        return LMGPU_OK;
    }
    for (int k = 0; k < 8; k++) {
        float* d = reinterpret_cast<float*>(base + size_t(k) * n * 4);
        hipError_t e = hipMemcpyAsync(d, src[k], size_t(n) * 4, hipMemcpyHostToDevice, ctx->stream);
        if (e != hipSuccess) return hip_fail(ctx, e, "ray upload");
        dev[k] = d;
    }
    *out_base = base + in_bytes;
    return LMGPU_OK;
}

// Host rays with host results go through pinned memory.  Up to kDirectRays the kernels read and
// write it themselves: a copy costs more than they wait for the link.  Up to kPipeMinChunk are
// copied to the device and back in one piece each.  More move through the device in chunks of a
// quarter of the batch (between kPipeMinChunk and kPipeChunk rays), two of them at a time in pinned
// memory and in the device staging, on three streams: uploads on one copy stream, the kernels on the
// context's stream, read-backs on the other copy stream, so the two transfer directions and the
// kernels overlap, while the host threads copy chunk c + 1 in from the caller's arrays and chunk
// c - 1 out to them.  A chunk may go to another kernel than the whole batch would (a last one of few
// rays, several lanes to each); a ray's result is the same in every one (hit_order, traverse.hpp).
// 81 rays 210 -> 34 us (eight copies in and four out before); 512 rays direct 36 us, copied 39; 4000
// rays 63 and 61.  65,000 rays 421 -> 240 us, 300,000 rays 900 -> 755 us, 1M rays 2.7 -> 1.6 ms; so
// much is saved a MiB, and once it has paid for the pinned memory and the two streams (3 to 6 ms
// each to make) a batch goes this way (HostIo::pays), from kPipeAlways rays on at once.
constexpr double kPieceUs = 58.0, kChunksUs = 15.0, kStreamsUs = 7000.0;
constexpr uint32_t kPipeAlways = 1u << 20;
constexpr uint32_t kDirectRays = 1024;
constexpr uint32_t kPipeChunk = 1u << 19;
constexpr uint32_t kPipeMinChunk = 1u << 16;

// Pinned host memory of at least `bytes` and what the pipelined path needs besides; false if it
// cannot be had (the caller then takes the plain staged copies).
bool ensure_pipeline(lmgpu_ctx* ctx, size_t bytes) {
    for (hipStream_t& cs : ctx->copy_streams)
        if (!cs && hipStreamCreateWithFlags(&cs, hipStreamNonBlocking) != hipSuccess) {
            cs = nullptr;
            (void)hipGetLastError();
            return false;
        }
    return ensure_pinned(ctx, bytes) && ensure_io_events(ctx);
}

// One result column of the pipelined path: the caller's host array and its element size.
struct HostOut {
    void* dst;
    size_t elem;
};

// Traces n host rays in chunks (see kPipeChunk); `launch(dev_rays, m, dev_out)` enqueues on
// the context's stream the kernels for m rays whose eight columns are dev_rays[0..7] and
// whose result columns start at dev_out[j].  Returns LMGPU_ERR_UNSUPPORTED, having done
// nothing, when the pinned memory or the copy streams cannot be had or do not pay yet.
template <class Launch>
lmgpu_status trace_host_pipelined(lmgpu_ctx* ctx, const lmgpu_rays_soa* rays, uint32_t n, const HostOut* outs,
                                  int nout, Launch&& launch, const char* what) {
    const float* src[8] = {rays->ox, rays->oy, rays->oz, rays->dx, rays->dy, rays->dz, rays->tmin, rays->tmax};
    for (int k = 0; k < 8; k++)
        if (!src[k]) return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "ray array is NULL");
    size_t elems = 0;
    for (int j = 0; j < nout; j++) elems += outs[j].elem;
    if (n <= kPipeMinChunk) {
        const size_t in = size_t(n) * 32, out = size_t(n) * elems;
        if (!pinned_pays(ctx, in + out, double(in + out) * (kPieceUs / (1 << 20))) || !ensure_pinned(ctx, in + out))
            return LMGPU_ERR_UNSUPPORTED;
        char* const pinned = static_cast<char*>(ctx->io->pinned);
        char* dev = pinned;
        CopyJob jobs[8];
        for (int k = 0; k < 8; k++)
            jobs[k] = {pinned + size_t(k) * n * 4, reinterpret_cast<const char*>(src[k]), size_t(n) * 4};
        ctx->io->team.run(jobs, 8);
        hipError_t e = hipSuccess;
        if (n > kDirectRays) {
            const lmgpu_status st = stage(ctx, in + out);
            if (st != LMGPU_OK) return st;
            dev = static_cast<char*>(ctx->trace_staging);
            e = hipMemcpyAsync(dev, pinned, in, hipMemcpyHostToDevice, ctx->stream);
        }
        const float* dr[8];
        for (int k = 0; k < 8; k++) dr[k] = reinterpret_cast<const float*>(dev + size_t(k) * n * 4);
        char* dout[4] = {nullptr, nullptr, nullptr, nullptr};
        size_t off = in;
        for (int j = 0; j < nout; j++) {
            dout[j] = dev + off;
            jobs[j] = {static_cast<char*>(outs[j].dst), pinned + off, size_t(n) * outs[j].elem};
            off += size_t(n) * outs[j].elem;
        }
        if (e == hipSuccess) e = launch(dr, n, dout);
        if (e == hipSuccess && dev != pinned) e = hipMemcpyAsync(pinned + in, dev + in, out, hipMemcpyDeviceToHost, ctx->stream);
        const hipError_t done = hipStreamSynchronize(ctx->stream);
        if (e == hipSuccess) e = done;
        if (e != hipSuccess) return hip_fail(ctx, e, what);
        ctx->io->team.run(jobs, nout);
        return LMGPU_OK;
    }
    const size_t quarter = (size_t(n) + 4 * kPipeMinChunk - 1) / (4 * kPipeMinChunk) * kPipeMinChunk;
    const size_t chunk = std::min<size_t>(kPipeChunk, std::max<size_t>(kPipeMinChunk, quarter));
    const size_t slot = (chunk * (32 + elems) + 255) / 256 * 256;
    if (n < kPipeAlways && !pinned_pays(ctx, 2 * slot, double(n) * double(32 + elems) * (kChunksUs / (1 << 20)),
                                        ctx->copy_streams[1] ? 0.0 : kStreamsUs))
        return LMGPU_ERR_UNSUPPORTED;
    if (!ensure_pipeline(ctx, 2 * slot)) return LMGPU_ERR_UNSUPPORTED;
    lmgpu_status st = stage(ctx, 2 * slot);
    if (st != LMGPU_OK) return st;
    char* pin = static_cast<char*>(ctx->io->pinned);
    char* dev = static_cast<char*>(ctx->trace_staging);
    const hipStream_t sk = ctx->stream, sin = ctx->copy_streams[0], sout = ctx->copy_streams[1];
    // start: the caller's earlier work on the context's stream; up / kdone / down: slot s's
    // upload, kernels and read-back of its latest chunk.
    const hipEvent_t start = ctx->io_events[0], *up = ctx->io_events + 1, *kdone = up + 2, *down = kdone + 2;
    hipError_t e = hipSuccess;
    // The staging buffers may still be in use by work queued earlier on the context's stream.
    if (e == hipSuccess) e = hipEventRecord(start, sk);
    if (e == hipSuccess) e = hipStreamWaitEvent(sin, start, 0);
    if (e == hipSuccess) e = hipStreamWaitEvent(sout, start, 0);
    bool up_pending[2] = {false, false}, used[2] = {false, false}, down_pending[2] = {false, false};
    uint64_t down_first[2] = {0, 0}, down_m[2] = {0, 0};
    // Copies a finished chunk's results from pinned slot s to the caller's arrays.
    auto copy_out = [&](int s) {
        CopyJob jobs[4];
        size_t off = down_m[s] * 32;
        for (int j = 0; j < nout; j++) {
            jobs[j] = {static_cast<char*>(outs[j].dst) + down_first[s] * outs[j].elem, pin + s * slot + off,
                       size_t(down_m[s]) * outs[j].elem};
            off += down_m[s] * outs[j].elem;
        }
        ctx->io->team.run(jobs, nout);
        down_pending[s] = false;
    };
    const uint64_t chunks = (uint64_t(n) + chunk - 1) / chunk;
    for (uint64_t c = 0; c < chunks && e == hipSuccess; c++) {
        const int s = int(c & 1);
        const uint64_t first = c * chunk;
        const uint32_t m = uint32_t(std::min<uint64_t>(chunk, uint64_t(n) - first));
        char* ps = pin + s * slot;
        char* ds = dev + s * slot;
        // The slot's previous upload has finished before its pinned rays are overwritten.
        if (up_pending[s]) {
            e = hipEventSynchronize(up[s]);
            if (e != hipSuccess) break;
            up_pending[s] = false;
        }
        CopyJob in[8];
        for (int k = 0; k < 8; k++)
            in[k] = {ps + size_t(k) * m * 4, reinterpret_cast<const char*>(src[k] + first), size_t(m) * 4};
        ctx->io->team.run(in, 8);
        // Upload once the slot's previous kernels have read its device rays.
        if (used[s]) e = hipStreamWaitEvent(sin, kdone[s], 0);
        if (e == hipSuccess) e = hipMemcpyAsync(ds, ps, size_t(m) * 32, hipMemcpyHostToDevice, sin);
        if (e == hipSuccess) e = hipEventRecord(up[s], sin);
        if (e != hipSuccess) break;
        up_pending[s] = true;
        // Trace once the rays are in and the slot's previous results have been read back.
        e = hipStreamWaitEvent(sk, up[s], 0);
        if (e == hipSuccess && used[s]) e = hipStreamWaitEvent(sk, down[s], 0);
        if (e != hipSuccess) break;
        const float* dr[8];
        for (int k = 0; k < 8; k++) dr[k] = reinterpret_cast<const float*>(ds + size_t(k) * m * 4);
        char* dout[4] = {nullptr, nullptr, nullptr, nullptr};
        size_t off = size_t(m) * 32;
        for (int j = 0; j < nout; j++) {
            dout[j] = ds + off;
            off += size_t(m) * outs[j].elem;
        }
        e = launch(dr, m, dout);
        if (e == hipSuccess) e = hipEventRecord(kdone[s], sk);
        if (e != hipSuccess) break;
        used[s] = true;
        // The previous chunk's results go out to the caller while this one is traced.
        const int t = 1 - s;
        if (down_pending[t]) {
            e = hipEventSynchronize(down[t]);
            if (e != hipSuccess) break;
            copy_out(t);
        }
        e = hipStreamWaitEvent(sout, kdone[s], 0);
        if (e == hipSuccess) e = hipMemcpyAsync(ps + size_t(m) * 32, ds + size_t(m) * 32, m * elems, hipMemcpyDeviceToHost, sout);
        if (e == hipSuccess) e = hipEventRecord(down[s], sout);
        if (e != hipSuccess) break;
        down_pending[s] = true;
        down_first[s] = first;
        down_m[s] = m;
    }
    // The last chunk's results (the one before it went out in the loop).
    for (int s = 0; s < 2 && e == hipSuccess; s++) {
        if (!down_pending[s]) continue;
        e = hipEventSynchronize(down[s]);
        if (e == hipSuccess) copy_out(s);
    }
    if (e != hipSuccess) {
        (void)hipStreamSynchronize(sin);
        (void)hipStreamSynchronize(sk);
        (void)hipStreamSynchronize(sout);
    }
    if (e != hipSuccess) return hip_fail(ctx, e, what);
    return LMGPU_OK;
}

lmgpu_status check_trace(lmgpu_ctx* ctx, const void* rays, const void* out) {
    if (!ctx) return LMGPU_ERR_INVALID_ARGUMENT;
    if (!rays || !out) return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "trace: NULL rays or output");
    if (!ctx->has_bvh) return fail(ctx, LMGPU_ERR_NO_BVH, "trace: build the BVH first");
    (void)hipSetDevice(ctx->device);
    return LMGPU_OK;
}

}  // namespace

extern "C" {

lmgpu_status lmgpu_trace_closest(lmgpu_ctx* ctx, const lmgpu_rays_soa* rays, uint32_t n, lmgpu_hits_soa* hits,
                                 uint32_t flags) {
    lmgpu_status s = check_trace(ctx, rays, hits);
    if (s != LMGPU_OK) return s;
    if (n == 0) return LMGPU_OK;
    if (!hits->t || !hits->b0 || !hits->b1 || !hits->prim)
        return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_trace_closest: NULL hit array");
    const bool refine = (flags & LMGPU_TRACE_REFINE_FP64) != 0;
    if (!rays->device && !hits->device) {
        const HostOut outs[4] = {{hits->t, 4}, {hits->b0, 4}, {hits->b1, 4}, {hits->prim, 4}};
        s = trace_host_pipelined(
            ctx, rays, n, outs, 4,
            [&](const float* const* dr, uint32_t m, char* const* o) {
                return launch_trace_closest(ctx, dr, m, reinterpret_cast<float*>(o[0]), reinterpret_cast<float*>(o[1]),
                                            reinterpret_cast<float*>(o[2]), reinterpret_cast<int32_t*>(o[3]), refine,
                                            ctx->next_counter);
            },
            "closest hit (host buffers)");
        if (s != LMGPU_ERR_UNSUPPORTED) return s;
    }
    const float* dev[8];
    char* out = nullptr;
    s = prepare_rays(ctx, rays, n, hits->device ? 0 : size_t(n) * 16, dev, &out);
    if (s != LMGPU_OK) return s;
    float *t = hits->t, *b0 = hits->b0, *b1 = hits->b1;
    int32_t* prim = hits->prim;
    if (!hits->device) {
        t = reinterpret_cast<float*>(out);
        b0 = t + n;
        b1 = b0 + n;
        prim = reinterpret_cast<int32_t*>(b1 + n);
    }
    hipError_t e = launch_trace_closest(ctx, dev, n, t, b0, b1, prim, refine, ctx->next_counter);
    if (e != hipSuccess) return hip_fail(ctx, e, "closest hit");
    if (!hits->device) {
        const void* srcs[4] = {t, b0, b1, prim};
        void* dsts[4] = {hits->t, hits->b0, hits->b1, hits->prim};
        for (int k = 0; k < 4; k++) {
            e = hipMemcpyAsync(dsts[k], srcs[k], size_t(n) * 4, hipMemcpyDeviceToHost, ctx->stream);
            if (e != hipSuccess) return hip_fail(ctx, e, "hit readback");
        }
        e = hipStreamSynchronize(ctx->stream);
        if (e != hipSuccess) return hip_fail(ctx, e, "trace synchronize");
    }
    return LMGPU_OK;
}

lmgpu_status lmgpu_trace_closest_noalloc(lmgpu_ctx* ctx, const lmgpu_rays_soa* rays, uint32_t n,
                                         lmgpu_hits_soa* hits, uint32_t flags) {
    lmgpu_status s = check_trace(ctx, rays, hits);
    if (s != LMGPU_OK) return s;
    if (!rays->device || !hits->device)
        return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT,
                    "lmgpu_trace_closest_noalloc: rays and hits must be device buffers (host buffers need staging "
                    "memory; use lmgpu_trace_closest)");
    if (n > LMGPU_NOALLOC_MAX_RAYS)
        return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT,
                    "lmgpu_trace_closest_noalloc: more than LMGPU_NOALLOC_MAX_RAYS (2^31) rays in one call");
    const float* dev[8] = {rays->ox, rays->oy, rays->oz, rays->dx, rays->dy, rays->dz, rays->tmin, rays->tmax};
    for (int k = 0; k < 8; k++)
        if (!dev[k]) return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_trace_closest_noalloc: NULL ray array");
    if (!hits->t || !hits->b0 || !hits->b1 || !hits->prim)
        return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_trace_closest_noalloc: NULL hit array");
    if (n == 0) return LMGPU_OK;
    if (!ctx->noalloc_scratch) {
        // Resolution failed when the context was created; the device is current (check_trace).
        uint32_t* sp = nullptr;
        hipError_t e = noalloc_scratch_address(ctx->device, &sp);
        if (e != hipSuccess) return hip_fail(ctx, e, "lmgpu_trace_closest_noalloc: scratch address");
        ctx->noalloc_scratch = sp;
    }
    // The same kernels as lmgpu_trace_closest; the work counter (cleared by a fill kernel
    // before the traversal) is word 0 of this device's static scratch array.
    hipError_t e = launch_trace_closest(ctx, dev, n, hits->t, hits->b0, hits->b1, hits->prim,
                                        (flags & LMGPU_TRACE_REFINE_FP64) != 0, ctx->noalloc_scratch);
    if (e != hipSuccess) return hip_fail(ctx, e, "closest hit");
    return LMGPU_OK;
}

lmgpu_status lmgpu_trace_any(lmgpu_ctx* ctx, const lmgpu_rays_soa* rays, uint32_t n, uint8_t* occluded,
                             int occluded_on_device, uint32_t flags) {
    (void)flags;
    lmgpu_status s = check_trace(ctx, rays, occluded);
    if (s != LMGPU_OK) return s;
    if (n == 0) return LMGPU_OK;
    if (!rays->device && !occluded_on_device) {
        const HostOut outs[1] = {{occluded, 1}};
        s = trace_host_pipelined(
            ctx, rays, n, outs, 1,
            [&](const float* const* dr, uint32_t m, char* const* o) {
                return launch_trace_any(ctx, dr, m, reinterpret_cast<uint8_t*>(o[0]));
            },
            "k_trace_any (host buffers)");
        if (s != LMGPU_ERR_UNSUPPORTED) return s;
    }
    const float* dev[8];
    char* out = nullptr;
    s = prepare_rays(ctx, rays, n, occluded_on_device ? 0 : size_t(n), dev, &out);
    if (s != LMGPU_OK) return s;
    uint8_t* occ = occluded_on_device ? occluded : reinterpret_cast<uint8_t*>(out);
    hipError_t e = launch_trace_any(ctx, dev, n, occ);
    if (e != hipSuccess) return hip_fail(ctx, e, "k_trace_any");
    if (!occluded_on_device) {
        e = hipMemcpyAsync(occluded, occ, n, hipMemcpyDeviceToHost, ctx->stream);
        if (e != hipSuccess) return hip_fail(ctx, e, "occlusion readback");
        e = hipStreamSynchronize(ctx->stream);
        if (e != hipSuccess) return hip_fail(ctx, e, "trace synchronize");
    }
    return LMGPU_OK;
}

lmgpu_status lmgpu_trace_count(lmgpu_ctx* ctx, const lmgpu_rays_soa* rays, uint32_t n, uint64_t* node_visits,
                               uint64_t* tri_tests) {
    lmgpu_status s = check_trace(ctx, rays, node_visits);
    if (s != LMGPU_OK) return s;
    if (!tri_tests) return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_trace_count: NULL output");
    const float* dev[8];
    char* out = nullptr;
    s = prepare_rays(ctx, rays, n, 0, dev, &out);
    if (s != LMGPU_OK) return s;
    hipError_t e = hipMemsetAsync(ctx->count_buf, 0, 16, ctx->stream);
    if (e == hipSuccess) e = launch_trace_count(ctx, dev, n, reinterpret_cast<unsigned long long*>(ctx->count_buf));
    uint64_t h[2] = {0, 0};
    if (e == hipSuccess) e = hipMemcpyAsync(h, ctx->count_buf, 16, hipMemcpyDeviceToHost, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) return hip_fail(ctx, e, "k_trace_count");
    *node_visits = h[0];
    *tri_tests = h[1];
    return LMGPU_OK;
}

lmgpu_status lmgpu_pt_render(lmgpu_ctx* ctx, const lmgpu_pt_params* params, lmgpu_film* film, lmgpu_pt_stats* stats) {
    if (!ctx) return LMGPU_ERR_INVALID_ARGUMENT;
    if (!params) return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_pt_render: NULL params");
    (void)hipSetDevice(ctx->device);
    return run_pt(ctx, params, film, stats);
}

lmgpu_status lmgpu_raycast_render(lmgpu_ctx* ctx, lmgpu_film* film) {
    if (!ctx) return LMGPU_ERR_INVALID_ARGUMENT;
    (void)hipSetDevice(ctx->device);
    return run_raycast(ctx, film);
}

lmgpu_status lmgpu_pt_backward(lmgpu_ctx* ctx, const lmgpu_pt_params* params, lmgpu_adjoint* adjoint,
                               lmgpu_pt_stats* stats) {
    if (!ctx) return LMGPU_ERR_INVALID_ARGUMENT;
    if (!params) return fail(ctx, LMGPU_ERR_INVALID_ARGUMENT, "lmgpu_pt_backward: NULL params");
    (void)hipSetDevice(ctx->device);
    return run_pt_backward(ctx, params, adjoint, stats);
}

lmgpu_status lmgpu_enable_timing(lmgpu_ctx* ctx, int enable) {
    if (!ctx) return LMGPU_ERR_INVALID_ARGUMENT;
    ctx->timing = enable != 0;
    return LMGPU_OK;
}

lmgpu_status lmgpu_kernel_timing(lmgpu_ctx* ctx, int kernel, double* total_ms, uint64_t* launches) {
    if (!ctx || kernel < 0 || kernel >= kKNumClasses || !total_ms || !launches) return LMGPU_ERR_INVALID_ARGUMENT;
    *total_ms = ctx->kernel_ms[kernel];
    *launches = ctx->kernel_launches[kernel];
    return LMGPU_OK;
}

lmgpu_status lmgpu_enable_counting(lmgpu_ctx* ctx, int enable) {
    if (!ctx) return LMGPU_ERR_INVALID_ARGUMENT;
    (void)hipSetDevice(ctx->device);
    ctx->counting = enable != 0;
    const hipError_t e = hipMemsetAsync(ctx->trav_counts, 0, 32, ctx->stream);
    return e == hipSuccess ? LMGPU_OK : hip_fail(ctx, e, "lmgpu_enable_counting");
}

lmgpu_status lmgpu_traversal_counts(lmgpu_ctx* ctx, int kernel, uint64_t* node_visits, uint64_t* tri_tests) {
    if (!ctx || (kernel != kKExtend && kernel != kKShadow) || !node_visits || !tri_tests)
        return LMGPU_ERR_INVALID_ARGUMENT;
    (void)hipSetDevice(ctx->device);
    uint64_t h[4] = {0, 0, 0, 0};
    hipError_t e = hipMemcpyAsync(h, ctx->trav_counts, sizeof(h), hipMemcpyDeviceToHost, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) return hip_fail(ctx, e, "lmgpu_traversal_counts");
    const int k = kernel == kKExtend ? 0 : 2;
    *node_visits = h[k];
    *tri_tests = h[k + 1];
    return LMGPU_OK;
}

lmgpu_status lmgpu_reset_timing(lmgpu_ctx* ctx) {
    if (!ctx) return LMGPU_ERR_INVALID_ARGUMENT;
    for (int k = 0; k < kKNumClasses; k++) {
        ctx->kernel_ms[k] = 0.0;
        ctx->kernel_launches[k] = 0;
    }
    return LMGPU_OK;
}

}  // extern "C"
