#!/usr/bin/env python3
"""Benchmark of the MI355X path-tracing hot path.

Headline line (one JSON object on stdout): closest-hit traversal throughput of the
traversal microbenchmark -- 1M triangles (centroids uniform in the unit cube, vertex
offsets N(0, 0.01)), 16M rays (origins uniform in [-0.5, 1.5]^3, directions uniform on
the sphere), 4-wide SAH BVH, FP32 traversal with the watertight test and the winner
re-evaluated in FP64 (LMGPU_TRACE_REFINE_FP64: t and barycentrics within 1e-5 of the FP64
oracle).  One step = one closest-hit pass over the 16M rays, with rays, BVH and outputs
resident in HBM.  The same pass without the FP64 re-evaluation is reported beside it.

Also reported (key "path_tracing"): the room scene (256 x 256, 16 spp, max depth 8,
RR from depth 3) rendered with the `pt` estimator -- M path-samples/s and Mrays/s -- and
with `pt.direct` / `pt.mis` (key "renderers", closest plus any-hit rays); and (key
"adjoint") the inverse-rendering workload -- the room plus 2,000 boxes (96k triangles),
512 x 512 x 32 spp, max depth 8, L2 loss against a target rendered with hidden box
reflectances -- forward and path-replay backward times, their ratio, and the adjoint
against central differences on 64 parameters.

`roofline` is measured live: HIP events around every traversal launch (the traversal
kernel and the FP64 pass) on the launch stream give the average duration; algorithmic
bytes per launch come from the kernel's own counting run (node visits x 64 B + triangle
tests x 48 B + 32 B ray + 16 B hit per ray) plus the FP64 pass (4 B per ray; ray, FP32
result, triangle record and result per hit).  `cpu_baseline` times the CPU restatement (FP32 4-wide QBVH with SSE,
OpenMP over the host cores) on the same rays.
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

METRIC = "M path-samples/s + Mrays/s on 1 MI355X at fixed RMSE; backward/forward ratio"
HBM_PEAK_GBS = 8000.0
NODE_BYTES = 64   # a packed 4-wide node (origin, steps, 24 8-bit planes, 4 child words)
TRI_BYTES = 48    # the vertices and index of a triangle record
RAY_BYTES = 32    # o, d, tmin, tmax
HIT_BYTES = 16    # t, b0, b1, prim


# Algorithmic bytes of the path tracer's stages (SoA path queues of 16-byte records):
#   extension ray: ray in (origin and direction records) 32 B, hit out 4 B (its record), plus the nodes and
#     triangle records its traversal visits;
#   shadow ray: record in (origin + tmax, direction + pixel, contribution + light) 48 B, one film
#     update 12 B, plus its traversal;
#   pt shading of one path: path in 48 B (3 records), hit 4 B, triangle 48 B, shading record 64 B, material 16 B;
#     a surviving path out 48 B, an ending path one film update 12 B;
#   camera stage: one path out, 48 B.
# A node visit counts as a packed node.  Segments of at most 65,536 rays (98,304 shadow rays) visit
# the nodes as built, 128 B, so the stages' bytes are a lower bound.
EXT_RAY_BYTES = 32 + 4
SHADOW_RAY_BYTES = 48 + 12
SHADE_IN_BYTES = 48 + 4 + 48 + 64 + 16
PATH_BYTES = 48
FILM_ADD_BYTES = 12
CLOCK_GHZ = 2.4  # MI355X peak engine clock
NUM_CUS = 256


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def pt_roofline(dev, renderer, samples, **render_kw):
    """HBM roofline of a path-traced render of a BVH scene, from two extra renders of the same
    work: one with per-kernel HIP-event timing (device time of each stage), one with the
    traversal stages' counting forms (node visits and triangle tests).  Algorithmic bytes per
    stage as EXT_RAY_BYTES ... above; for pt the shading and camera stages are included, so the
    render-level figure covers every kernel of the render."""
    dev.enable_timing(True)
    dev.reset_timing()
    _, st = dev.render(renderer, num_samples=samples, **render_kw)
    t = {k: dev.kernel_timing(k) for k in (2, 3, 4, 5)}
    dev.enable_timing(False)
    dev.enable_counting(True)
    try:
        dev.render(renderer, num_samples=samples, **render_kw)
        ev, et = dev.traversal_counts(5)
        sv, stt = dev.traversal_counts(4)
    finally:
        dev.enable_counting(False)
    ext_bytes = st.closest_rays * EXT_RAY_BYTES + ev * NODE_BYTES + et * TRI_BYTES
    shadow_bytes = st.shadow_rays * SHADOW_RAY_BYTES + sv * NODE_BYTES + stt * TRI_BYTES
    ext_ms, shadow_ms = t[5][0], t[4][0]
    out = {
        "bound": "hbm", "peak": HBM_PEAK_GBS, "unit": "GB/s",
        "extension": {"kernel": "k_extend", "launches": t[5][1], "kernel_ms": round(ext_ms, 4),
                      "node_visits_per_ray": round(ev / max(st.closest_rays, 1), 3),
                      "tri_tests_per_ray": round(et / max(st.closest_rays, 1), 3),
                      "alg_bytes": int(ext_bytes),
                      "achieved": round(ext_bytes / (ext_ms * 1e-3) / 1e9, 1) if ext_ms > 0 else None},
    }
    out["extension"]["frac"] = (round(out["extension"]["achieved"] / HBM_PEAK_GBS, 4)
                                if out["extension"]["achieved"] else None)
    if st.shadow_rays:
        out["shadow"] = {"kernel": "k_shadow", "launches": t[4][1], "kernel_ms": round(shadow_ms, 4),
                         "node_visits_per_ray": round(sv / st.shadow_rays, 3),
                         "tri_tests_per_ray": round(stt / st.shadow_rays, 3), "alg_bytes": int(shadow_bytes),
                         "achieved": round(shadow_bytes / (shadow_ms * 1e-3) / 1e9, 1) if shadow_ms > 0 else None}
        out["shadow"]["frac"] = round(out["shadow"]["achieved"] / HBM_PEAK_GBS, 4) if out["shadow"]["achieved"] else None
    if renderer == "pt":
        shade_bytes = st.closest_rays * SHADE_IN_BYTES + (st.closest_rays - samples) * PATH_BYTES + samples * FILM_ADD_BYTES
        gen_bytes = samples * PATH_BYTES
        total_ms = sum(v[0] for v in t.values())
        total = ext_bytes + shade_bytes + gen_bytes
        out["render"] = {"kernels_ms": round(total_ms, 4), "alg_bytes": int(total),
                         "achieved": round(total / (total_ms * 1e-3) / 1e9, 1),
                         "shade_ms": round(t[2][0], 4), "gen_ms": round(t[3][0], 4)}
        out["render"]["frac"] = round(out["render"]["achieved"] / HBM_PEAK_GBS, 4)
    out["frac"] = out["render"]["frac"] if "render" in out else out["extension"]["frac"]
    if out["frac"] and out["frac"] > 1.0:
        out["note"] = ("algorithmic bytes faster than HBM can deliver: neighbouring rays re-read the same BVH nodes and "
                       "triangle records, which L2 and the 256 MB Infinity Cache serve; the traversal is bound by "
                       "memory latency at its lane occupancy and the per-lane load path, not by HBM bandwidth")
    return out


def cpu_info():
    model = "unknown"
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                model = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    return model


def host_threads() -> int:
    n = len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else (os.cpu_count() or 1)
    env = os.environ.get("OMP_NUM_THREADS")
    if env and env.isdigit():
        n = min(n, int(env))
    return max(1, n)


def traffic_from_profile():
    """HBM bytes per launch from the committed rocprofv3 --pmc summary, if present."""
    p = ROOT / "profiles" / "traversal_closest_1Mtri_16Mray_pmc.json"
    if not p.exists():
        return None
    try:
        d = json.loads(p.read_text())
        return float(d["hbm_bytes_per_launch"])
    except Exception:
        return None


def run_traversal(args, torch, Device, scenes):
    import numpy as np

    t0 = time.time()
    sc = scenes.traversal_scene(args.triangles)
    rays = scenes.traversal_rays(args.rays)
    log(f"[bench] generated {sc.num_triangles} triangles and {len(rays)} rays in {time.time() - t0:.1f}s")
    dev = Device(0)
    dev.upload(sc)
    info = dev.build_bvh(max_leaf_size=args.leaf, sah_bins=args.sah_bins, traversal_cost=args.traversal_cost)
    log(f"[bench] BVH: {info.num_nodes} nodes, depth {info.max_depth}, {info.build_seconds:.2f}s, "
        f"{info.device_bytes / 2**20:.1f} MiB")
    cols = [torch.from_numpy(rays.o[:, k].copy()) for k in range(3)] + \
           [torch.from_numpy(rays.d[:, k].copy()) for k in range(3)] + \
           [torch.from_numpy(rays.tmin), torch.from_numpy(rays.tmax)]
    dcols = [c.to("cuda:0") for c in cols]
    n = len(rays)
    out = [torch.empty(n, dtype=torch.float32, device="cuda:0") for _ in range(3)] + \
          [torch.empty(n, dtype=torch.int32, device="cuda:0")]
    ray_ptrs = [c.data_ptr() for c in dcols]
    out_ptrs = [c.data_ptr() for c in out]
    torch.cuda.synchronize()

    # The library launches on a stream of torch's (default priority), so HIP events recorded
    # on that stream around each launch time the kernels inside the timed region itself.
    stream = torch.cuda.Stream()
    dev.set_stream(stream.cuda_stream)

    def timed_steps(launch, steps):
        """K launches on the host clock, bracketed by device synchronisation, with HIP events
        around each launch: (wall seconds, average event milliseconds per launch)."""
        evs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(steps)]
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for e0, e1 in evs:
            e0.record(stream)
            launch()
            e1.record(stream)
        dev.synchronize()
        torch.cuda.synchronize()
        wall = time.perf_counter() - t0
        return wall, sum(e0.elapsed_time(e1) for e0, e1 in evs) / steps

    # The headline is the closest hit with the winner re-evaluated in FP64
    # (LMGPU_TRACE_REFINE_FP64): FP32 traversal, t and barycentrics within 1e-5 of the FP64
    # oracle, the configuration that meets the precision bar.
    refined = [torch.empty(n, dtype=torch.float32, device="cuda:0") for _ in range(3)] + \
              [torch.empty(n, dtype=torch.int32, device="cuda:0")]
    ref_ptrs = [c.data_ptr() for c in refined]
    for _ in range(args.warmup):
        dev.trace_closest_device(ray_ptrs, ref_ptrs, n, refine_fp64=True)
    dev.synchronize()
    torch.cuda.synchronize()

    # Timed region: K steps.
    wall, avg_ms = timed_steps(lambda: dev.trace_closest_device(ray_ptrs, ref_ptrs, n, refine_fp64=True), args.steps)
    log(f"[bench] traversal: {args.steps} steps in {wall:.3f}s, {avg_ms:.4f} ms per launch (events)")

    # Any hit over the same rays (tmax = FLT_MAX: occluded = hits anything), and the closest hit
    # with the FP32 weights of the watertight test (no FP64 re-evaluation).
    occ = torch.empty(n, dtype=torch.uint8, device="cuda:0")
    extra = {}
    for name, launch in (("any_hit", lambda: dev.trace_any_device(ray_ptrs, occ.data_ptr(), n)),
                         ("closest_fp32", lambda: dev.trace_closest_device(ray_ptrs, out_ptrs, n))):
        for _ in range(args.warmup):
            launch()
        dev.synchronize()
        w, ms = timed_steps(launch, args.steps)
        extra[name] = {"Mrays_per_s": round(n * args.steps / w / 1e6, 1), "ms_per_step": round(w / args.steps * 1e3, 3),
                       "kernel_ms": round(ms, 4)}
        log(f"[bench] {name}: {extra[name]}")

    dev.set_stream(0)
    # Algorithmic bytes per launch from the counting traversal.
    visits, tests = dev.trace_count(rays)
    prim = refined[3].cpu().numpy()
    # The FP64 pass (k_refine_fp64) reads each ray's record index (4 B) and, for a hit, the ray's
    # origin and direction (24 B) and the winner's triangle record, and writes the result.
    hits = int((prim >= 0).sum())
    alg_bytes = n * (RAY_BYTES + HIT_BYTES) + visits * NODE_BYTES + tests * TRI_BYTES + \
        n * 4 + hits * (24 + TRI_BYTES + HIT_BYTES)
    hit_rate = float((prim >= 0).mean())
    occ_h = occ.cpu().numpy()
    extra["any_hit"]["occluded_rate"] = round(float(occ_h.mean()), 4)
    extra["any_hit"]["agrees_with_closest_hit"] = bool(np.array_equal(occ_h != 0, prim >= 0))
    gpu_hits = {"fp32": [c.cpu().numpy() for c in out], "refine_fp64": [c.cpu().numpy() for c in refined]}

    # The same rays from pageable host arrays through lmgpu_trace_closest, the form in which a
    # Scene::Intersect caller hands rays over: staging copies over PCIe in and hits out
    # included (reported beside the value, never as it).
    host_cols = dev.ray_columns(rays)
    dev.trace_closest_columns(host_cols, refine_fp64=False)  # pinned chunks and staging buffers
    t0 = time.perf_counter()
    host_hits = dev.trace_closest_columns(host_cols, refine_fp64=False)
    host_s = time.perf_counter() - t0
    host_same = bool(np.array_equal(host_hits[3], prim))
    dev.close()
    res = {
        "ms_per_step": wall / args.steps * 1e3,
        "value": n * args.steps / wall / 1e6,
        "kernel_ms": avg_ms,
        "alg_bytes": alg_bytes,
        "node_visits_per_ray": visits / n,
        "tri_tests_per_ray": tests / n,
        "hit_rate": hit_rate,
        "bvh": info,
        "host_buffers": {"Mrays_per_s": round(n / host_s / 1e6, 1), "seconds": round(host_s, 4),
                         "same_hits_as_device_buffers": host_same,
                         "note": "lmgpu_trace_closest on pageable host arrays (32 B per ray in, 16 B per hit "
                                 "out over PCIe, in 512k-ray chunks through pinned memory), one call over the "
                                 "same rays"},
        "modes": extra,
        "gpu_hits": gpu_hits,
    }
    return res, sc, rays


def classify_ids(sc, rays, g_prim, g_t, r_prim, r_t, edge_eps=1e-5, tie_rel=1e-6):
    """Primitive ids of every ray, GPU against an oracle, sorted into: identical; near ties
    (both hit, |t_gpu - t_ref| <= 1e-6 t_ref); near edges (the nearer of the two candidate
    triangles -- the only one hit, or the one with the smaller t -- is crossed within 1e-5 of an
    edge in float64 barycentrics, where the GPU's watertight test and the reference's
    Moeller-Trumbore / TriAccel tests may disagree); unexplained (the rest)."""
    import numpy as np

    same = g_prim == r_prim
    d = np.where(~same)[0]
    gp, rp, gt, rt = g_prim[d], r_prim[d], g_t[d], r_t[d]
    both = (gp >= 0) & (rp >= 0)
    tie = both & (np.abs(gt - rt) <= tie_rel * np.abs(rt))
    # the nearer candidate
    use_g = (rp < 0) | (both & (gt < rt))
    cand = np.where(use_g, gp, rp)
    P = sc.positions.astype(np.float64)
    F = sc.faces[cand]
    p0, p1, p2 = P[F[:, 0]], P[F[:, 1]], P[F[:, 2]]
    o = rays.o[d].astype(np.float64)
    dd = rays.d[d].astype(np.float64)
    e1, e2 = p1 - p0, p2 - p0
    s1 = np.cross(dd, e2)
    div = np.einsum("ij,ij->i", s1, e1)
    with np.errstate(divide="ignore", invalid="ignore"):
        inv = 1.0 / div
        q = o - p0
        u = np.einsum("ij,ij->i", q, s1) * inv
        v = np.einsum("ij,ij->i", dd, np.cross(q, e1)) * inv
    edge = np.minimum(np.minimum(np.abs(u), np.abs(v)), np.abs(1.0 - u - v)) <= edge_eps
    near_edge = ~tie & edge
    return {"rays": int(len(g_prim)), "identical": int(same.sum()), "near_tie": int(tie.sum()),
            "near_edge": int(near_edge.sum()), "unexplained": int((~tie & ~edge).sum())}


def id_parity(sc, rays, gpu_hits):
    """Every GPU primitive id against the FP64 oracle (BVH + TriAccel, the reference's double
    build) and the FP32 oracle (the reference's default SSE QBVH), plus t and barycentric errors
    of the FP64-refined closest hit against the FP64 oracle where the ids agree."""
    import numpy as np

    from oracle import lmref

    out = {}
    threads = host_threads()
    ref = {}
    for name, fp64, accel in (("fp64_bvh", True, "bvh"), ("fp32_qbvh", False, "qbvh")):
        t0 = time.time()
        o = lmref.Oracle(sc, fp64=fp64, accel=accel)
        t, b0, b1, tri = o.trace_closest(rays, threads=threads)
        ref[name] = (t, b0, b1, tri)
        for mode, (gt, gb0, gb1, gp) in gpu_hits.items():
            out[f"gpu_{mode}_vs_{name}"] = classify_ids(sc, rays, gp, gt.astype(np.float64), tri, t)
        log(f"[bench] ids vs {name}: {time.time() - t0:.1f}s")
    t, b0, b1, tri = ref["fp64_bvh"]
    gt, gb0, gb1, gp = gpu_hits["refine_fp64"]
    m = (gp == tri) & (tri >= 0)
    out["refine_fp64_errors_vs_fp64_bvh"] = {
        "rays_compared": int(m.sum()),
        "max_rel_t": float(np.max(np.abs(gt[m] - t[m]) / np.abs(t[m]))),
        "max_abs_barycentric": float(max(np.max(np.abs(gb0[m] - b0[m])), np.max(np.abs(gb1[m] - b1[m])))),
    }
    gt, gb0, gb1, gp = gpu_hits["fp32"]
    m = (gp == tri) & (tri >= 0)
    out["fp32_errors_vs_fp64_bvh"] = {
        "rays_compared": int(m.sum()),
        "max_rel_t": float(np.max(np.abs(gt[m] - t[m]) / np.abs(t[m]))),
        "max_abs_barycentric": float(max(np.max(np.abs(gb0[m] - b0[m])), np.max(np.abs(gb1[m] - b1[m])))),
    }
    return out


def run_pt(args, Device, scenes):
    sc = scenes.room_scene(256, 256, 16)
    dev = Device(0)
    dev.upload(sc)
    dev.build_bvh()
    dev.render("pt", film_precision="fp32")  # warm-up at full size (buffers sized, caches warm)
    secs, rays = [], []
    for _ in range(args.pt_steps):
        _, st = dev.render("pt", film_precision="fp32")
        secs.append(st.seconds)
        rays.append(st.closest_rays)
    # The next-event renderers on the same room: closest-hit extension rays plus any-hit
    # shadow rays (one per non-specular vertex, the camera vertex included).
    nee = {}
    for renderer in ("pt.direct", "pt.mis"):
        dev.render(renderer, film_precision="fp32")  # warm-up at full size
        rs, rr = [], []
        for _ in range(args.pt_steps):
            _, st = dev.render(renderer, film_precision="fp32")
            rs.append(st.seconds)
            rr.append(st.closest_rays + st.shadow_rays)
        m = sum(rs) / len(rs)
        nee[renderer] = {"M_path_samples_per_s": round(sc.render.num_samples / m / 1e6, 1),
                         "Mrays_per_s": round(sum(rr) / len(rr) / m / 1e6, 1),
                         "ms_per_render": round(m * 1e3, 3),
                         "rays_per_sample": round(sum(rr) / len(rr) / sc.render.num_samples, 3),
                         "roofline": valu_roofline(renderer, m * 1e3)}
    dev.close()
    s = sum(secs) / len(secs)
    return {
        "workload": "room: 5-quad box room + 2 rotated boxes + 0.25x0.25 light (17,12,4); 256x256, 16 spp "
                    "(1,048,576 samples), max_path_vertices 9, rr_depth 3; renderer pt; FP32 film",
        "M_path_samples_per_s": sc.render.num_samples / s / 1e6,
        "Mrays_per_s": (sum(rays) / len(rays)) / s / 1e6,
        "ms_per_render": s * 1e3,
        "rays_per_sample": (sum(rays) / len(rays)) / sc.render.num_samples,
        "roofline": valu_roofline("pt", s * 1e3),
        "renderers": nee,
    }, sc


def valu_roofline(renderer, ms_per_render):
    """VALU-issue roofline of a room render (triangle by triangle in the shading kernels, no
    memory bound): VALU wave-instructions per render from the committed counter profile
    (profiles/pt_room_valu_pmc.json, rocprofv3 SQ_INSTS_VALU summed over one render's
    dispatches) over the live render time, against one wave-instruction per CU per cycle
    (four SIMDs each issuing a wave64 instruction every four cycles) at the peak clock."""
    p = ROOT / "profiles" / "pt_room_valu_pmc.json"
    if not p.exists():
        return None
    d = json.loads(p.read_text()).get(renderer)
    if not d:
        return None
    inst = float(d["SQ_INSTS_VALU_per_render"])
    achieved = inst / (ms_per_render * 1e-3) / (NUM_CUS * CLOCK_GHZ * 1e9)
    return {"bound": "valu", "achieved": round(achieved, 4), "peak": 1.0,
            "unit": "VALU wave-instructions per CU per cycle", "frac": round(achieved, 4),
            "lane_utilisation": d.get("lane_utilisation"), "valu_instructions_per_render": inst,
            "source": "profiles/pt_room_valu_pmc.json"}


def run_adjoint(args, Device, scenes):
    """Forward render and path-replay backward of the gradient workload (pt, no RR)."""
    import numpy as np

    sc = scenes.gradient_scene(512, 512, 32)
    boxes = np.asarray(sc.meta["box_materials"])
    albedo = np.array([m["R"] for m in sc.materials], np.float64)
    emission = np.array([l["Le"] for l in sc.lights], np.float64)
    hidden = albedo.copy()
    hidden[boxes] = scenes.hidden_box_albedo(len(boxes))
    dev = Device(0)
    dev.upload(sc)
    dev.build_bvh()
    dev.set_params(hidden, emission)
    target, _ = dev.render("pt", film_precision="fp32")
    dev.set_params(albedo, emission)
    import torch

    record = torch.empty((sc.render.num_samples, 4), dtype=torch.float32, device="cuda:0")
    fwd, bwd, bwd2, res = [], [], [], []
    for _ in range(args.pt_steps):
        # forward recording each sample's radiance; backward with one replay
        img, st = dev.render("pt", film_precision="fp32", sample_record_ptr=record.data_ptr())
        fwd.append(st.seconds)
        d = (2.0 * (img - target)).astype(np.float32)
        ga, ge, info = dev.backward("pt", d, sample_record_ptr=record.data_ptr())
        bwd.append(info["seconds"])
        res.append(info["replay_residual"])
        # the same backward without the record: two replays
        _, _, info2 = dev.backward("pt", d)
        bwd2.append(info2["seconds"])
    roof = pt_roofline(dev, "pt", sc.render.num_samples, film_precision="fp32")
    fd = adjoint_fd_check(dev, sc, albedo, emission, hidden, boxes)
    adam = adam_trace(dev, albedo, emission, hidden, boxes)
    # The next-event renderers on the same workload, with their two-slot records.
    from lightmetrica_amd.gpu import record_float4s

    nee = {}
    for renderer in ("pt.direct", "pt.mis"):
        dev.set_params(hidden, emission)
        tgt, _ = dev.render(renderer, film_precision="fp32")
        dev.set_params(albedo, emission)
        rec = torch.empty((record_float4s(renderer, sc.render.num_samples), 4), dtype=torch.float32, device="cuda:0")
        rf, rb, rb2 = [], [], []
        for _ in range(args.pt_steps):
            img, st = dev.render(renderer, film_precision="fp32", sample_record_ptr=rec.data_ptr())
            rf.append(st.seconds)
            d = (2.0 * (img - tgt)).astype(np.float32)
            rb.append(dev.backward(renderer, d, sample_record_ptr=rec.data_ptr())[2]["seconds"])
            rb2.append(dev.backward(renderer, d)[2]["seconds"])
        mf, mb, mb2 = sum(rf) / len(rf), sum(rb) / len(rb), sum(rb2) / len(rb2)
        nee[renderer] = {"forward_ms": round(mf * 1e3, 3), "backward_ms": round(mb * 1e3, 3),
                         "backward_over_forward": round(mb / mf, 3),
                         "backward_without_record_ms": round(mb2 * 1e3, 3),
                         "backward_without_record_over_forward": round(mb2 / mf, 3)}
        del rec
    dev.close()
    f, b, b2 = sum(fwd) / len(fwd), sum(bwd) / len(bwd), sum(bwd2) / len(bwd2)
    return {
        "workload": "gradient: room + 2000 axis-aligned boxes (96,042 triangles), 4 ceiling lights; 512x512, "
                    "32 spp (8,388,608 samples), max_path_vertices 9, no RR; renderer pt; L2 loss vs a target "
                    "with hidden box reflectances U[0.1,0.9]; parameters: 2004 materials x RGB + 4 lights x RGB; "
                    "the forward records each sample's radiance (16 B/sample) for a one-replay backward",
        "forward_ms": round(f * 1e3, 3),
        "backward_ms": round(b * 1e3, 3),
        "backward_over_forward": round(b / f, 3),
        "backward_without_record_ms": round(b2 * 1e3, 3),
        "backward_without_record_over_forward": round(b2 / f, 3),
        "forward_M_path_samples_per_s": round(sc.render.num_samples / f / 1e6, 1),
        "replay_residual": max(res),
        "gradient_norm": float(np.linalg.norm(ga)),
        "fd_check": fd,
        "adam": adam,
        "forward_roofline": roof,
        "parameters": {"materials": len(albedo), "lights": len(emission),
                       "scalar_parameters": 3 * (len(albedo) + len(emission)),
                       "note": "one diffuse reflectance per box (2000) plus the room's 4 materials, RGB each, and "
                               "4 light emissions RGB: 6,024 scalars; the workload's '10k params' is not reached by "
                               "2000 boxes x RGB"},
        "renderers": nee,
    }


def adjoint_fd_check(dev, sc, albedo, emission, hidden, boxes, n_albedo=56, n_light=8, h=1e-3):
    """The adjoint through the torch.autograd.Function (lightmetrica_amd.autograd.render, GPU
    float64 tensors: FP64 film and image, the backward from the forward's sample record)
    against central differences of the same forward on the full gradient workload: h = 1e-3 on
    64 random parameters (56 box reflectance channels, 8 light emission channels), common
    sample streams.  Without Russian roulette every path is a fixed function of its stream, so
    the differences are exact up to rounding."""
    import numpy as np
    import torch

    from lightmetrica_amd.autograd import render as drender

    def t64(x, grad=False):
        return torch.tensor(np.asarray(x, np.float64), device="cuda:0", requires_grad=grad)

    def loss_of(a, e):
        with torch.no_grad():
            d = drender(dev, t64(a), t64(e)) - target
            return float((d * d).sum())

    with torch.no_grad():
        target = drender(dev, t64(hidden), t64(emission))
    a_t, e_t = t64(albedo, True), t64(emission, True)
    loss = ((drender(dev, a_t, e_t) - target) ** 2).sum()
    loss.backward()
    ga, ge = a_t.grad.cpu().numpy(), e_t.grad.cpu().numpy()
    rng = np.random.default_rng(0xC4)
    params = [("albedo", int(rng.choice(boxes)), int(rng.integers(3))) for _ in range(n_albedo)]
    params += [("emission", int(rng.integers(len(sc.lights))), int(rng.integers(3))) for _ in range(n_light)]
    g_fd, g_adj = [], []
    for kind, i, c in params:
        lv = []
        for s in (+1.0, -1.0):
            a, e = albedo.copy(), emission.copy()
            (a if kind == "albedo" else e)[i, c] += s * h
            lv.append(loss_of(a, e))
        g_fd.append((lv[0] - lv[1]) / (2 * h))
        g_adj.append((ga if kind == "albedo" else ge)[i, c])
    dev.set_params(albedo, emission)
    g_fd, g_adj = np.array(g_fd), np.array(g_adj)
    big = np.abs(g_fd) > 1e-2 * np.abs(g_fd).max()
    return {
        "through": "lightmetrica_amd.autograd.render (torch.autograd.Function), loss.backward()",
        "parameters": len(params),
        "h": h,
        "rel_error_norm": float(np.linalg.norm(g_adj - g_fd) / np.linalg.norm(g_fd)),
        "worst_rel_error": float((np.abs(g_adj - g_fd)[big] / np.abs(g_fd[big])).max()),
        "worst_over": int(big.sum()),
    }


def adam_trace(dev, albedo, emission, hidden, boxes, iters=24, lr=0.05):
    """Inverse rendering on the full gradient workload through the torch.autograd.Function:
    the box reflectances start at 0.5 and Adam (lr 0.05, reflectances clamped to [0, 1])
    minimises the L2 image loss against the target rendered with the hidden reflectances.
    Every iteration is one forward (recording each sample's radiance) and one backward."""
    import numpy as np
    import torch

    from lightmetrica_amd.autograd import render as drender

    with torch.no_grad():
        target = drender(dev, torch.tensor(hidden, dtype=torch.float32, device="cuda:0"),
                         torch.tensor(emission, dtype=torch.float32, device="cuda:0"))
    a = torch.tensor(albedo, dtype=torch.float32, device="cuda:0", requires_grad=True)
    e = torch.tensor(emission, dtype=torch.float32, device="cuda:0")
    opt = torch.optim.Adam([a], lr=lr)
    mask = torch.zeros_like(a)
    mask[torch.as_tensor(boxes, device="cuda:0")] = 1.0  # only the box reflectances move
    hid = torch.tensor(hidden, dtype=torch.float32, device="cuda:0")
    losses, prmse = [], []
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(iters):
        opt.zero_grad()
        loss = ((drender(dev, a, e) - target) ** 2).sum()
        loss.backward()
        a.grad *= mask
        losses.append(float(loss))
        prmse.append(float(torch.sqrt(((a.detach() - hid)[mask > 0] ** 2).mean())))
        opt.step()
        with torch.no_grad():
            a.clamp_(0.0, 1.0)
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    dev.set_params(albedo, emission)
    return {"iterations": iters, "optimizer": f"Adam lr {lr}, reflectances clamped to [0, 1]",
            "loss_first": losses[0], "loss_last": losses[-1], "loss_ratio": round(losses[-1] / losses[0], 4),
            "param_rmse_first": round(prmse[0], 4), "param_rmse_last": round(prmse[-1], 4),
            "ms_per_iteration": round(dt / iters * 1e3, 2)}


def rmse(a, b):
    """BitmapImage::EvaluateRMSE (bitmap.cpp:31-52): sqrt(mean over W*H*3 values of (a - b)^2)."""
    import numpy as np

    return float(np.sqrt(np.mean((np.asarray(a, np.float64) - np.asarray(b, np.float64)) ** 2)))


def run_terrain_study(args, Device, scenes):
    """Film precision study on the terrain: the same 132,710,400 path samples accumulated in
    FP32, compensated FP32 and FP64 films, each compared with the FP64 film of the same
    contributions and with the FP64 CPU restatement tracing the same sample streams."""
    import numpy as np

    from oracle import lmref

    t0 = time.time()
    spp = args.spp or 64
    sc = scenes.terrain_scene(1920, 1080, spp)
    log(f"[terrain] {sc.num_triangles} triangles, {len(sc.materials)} materials, generated in {time.time() - t0:.1f}s")
    dev = Device(0)
    dev.upload(sc)
    info = dev.build_bvh()
    log(f"[terrain] BVH {info.num_nodes} nodes, depth {info.max_depth}, {info.build_seconds:.1f}s")
    dev.render("pt", num_samples=1 << 22)  # warm-up
    films, out = {}, {}
    for mode in ("fp32", "fp32c", "fp64"):
        img, st = dev.render("pt", film_precision=mode, out_precision="fp64")
        films[mode] = img
        out[mode] = {"seconds": round(st.seconds, 4), "M_path_samples_per_s": round(st.samples / st.seconds / 1e6, 1),
                     "Mrays_per_s": round((st.closest_rays + st.shadow_rays) / st.seconds / 1e6, 1)}
        log(f"[terrain] {mode}: {st.seconds:.3f}s")
    roof = pt_roofline(dev, "pt", sc.render.num_samples, film_precision="fp32")
    ref = films["fp64"]
    scale = float(np.sqrt(np.mean(ref ** 2)))
    for mode in ("fp32", "fp32c"):
        out[mode]["rmse_vs_gpu_fp64_film"] = rmse(films[mode], ref)
        out[mode]["max_rel_vs_gpu_fp64_film"] = float(np.max(np.abs(films[mode] - ref)) / np.max(np.abs(ref)))
    # The FP64 oracle traces the same streams; compared over the whole image.
    threads = host_threads()
    t0 = time.time()
    o = lmref.Oracle(sc, fp64=True, accel="bvh")
    log(f"[terrain] oracle BVH built in {time.time() - t0:.1f}s")
    t0 = time.time()
    oimg, ost = o.render("pt", threads=threads)
    log(f"[terrain] oracle rendered {ost['samples']} samples in {time.time() - t0:.1f}s on {threads} threads")
    for mode in ("fp32", "fp32c", "fp64"):
        d = films[mode] - oimg
        out[mode]["rmse_vs_fp64_oracle"] = rmse(films[mode], oimg)
        out[mode]["rel_rmse_vs_fp64_oracle"] = rmse(films[mode], oimg) / scale
        out[mode]["pixels_within_1e-3"] = float(np.mean(np.abs(d) <= 1e-3 * np.maximum(np.abs(oimg), 1e-2 * scale)))
    # Control: the oracle's FP32 build (the reference's FP32 QBVH, exact normalize) on the same
    # streams against the FP64 oracle -- what FP32 path arithmetic alone does to this image.
    t0 = time.time()
    o32 = lmref.Oracle(sc, fp64=False, accel="qbvh")
    cimg, cst = o32.render("pt", threads=threads)
    log(f"[terrain] FP32 oracle control in {time.time() - t0:.1f}s")
    d = cimg - oimg
    control = {"rmse_vs_fp64_oracle": rmse(cimg, oimg), "rel_rmse_vs_fp64_oracle": rmse(cimg, oimg) / scale,
               "pixels_within_1e-3": float(np.mean(np.abs(d) <= 1e-3 * np.maximum(np.abs(oimg), 1e-2 * scale))),
               "seconds": round(cst["seconds"], 2)}
    dev.close()
    return {"workload": "terrain: 1024x1024-cell heightfield (2,097,152 triangles), 6-octave fBm x 0.2, 40% mirror "
                        "triangles, 60% diffuse U[0.1,0.9]; 1x1 quad light (Le 10) + constant environment (0.5); "
                        f"1920x1080, {spp} spp ({sc.render.num_samples} samples), max_path_vertices 17, rr_depth 3; "
                        "renderer pt",
            "image_rms": scale, "films": out, "roofline": roof,
            "M_path_samples_per_s": out["fp32"]["M_path_samples_per_s"],
            "cpu_fp32_oracle_control": control,
            "oracle": {"seconds": round(ost["seconds"], 2), "threads": threads, "cpu": cpu_info(),
                       "M_path_samples_per_s": round(ost["samples"] / ost["seconds"] / 1e6, 3)}}


def run_city(args, torch, Device, scenes):
    """The 16M-triangle city: FP32 forward, path-replay backward (FP64 gradient reduction), HBM use."""
    import numpy as np

    t0 = time.time()
    spp = args.spp or 256
    sc = scenes.city_scene(3840, 2160, spp)
    log(f"[city] {sc.num_triangles} triangles generated in {time.time() - t0:.1f}s")
    free0, total = torch.cuda.mem_get_info(0)
    dev = Device(0)
    dev.upload(sc)
    info = dev.build_bvh()
    log(f"[city] BVH {info.num_nodes} nodes, depth {info.max_depth}, {info.build_seconds:.1f}s, "
        f"{info.device_bytes / 2**30:.2f} GiB")
    dev.render("pt", num_samples=1 << 22)  # warm-up
    img, st = dev.render("pt", film_precision="fp32", out_precision="fp32")
    log(f"[city] forward {st.samples} samples in {st.seconds:.2f}s")
    free1, _ = torch.cuda.mem_get_info(0)
    roof = pt_roofline(dev, "pt", sc.render.num_samples, film_precision="fp32", out_precision="fp32")
    # Backward of L = 0.5 * sum(I^2): dL/dI = I.
    ga, ge, binfo = dev.backward("pt", img.astype(np.float32))
    log(f"[city] backward in {binfo['seconds']:.2f}s, replay residual {binfo['replay_residual']:.1e}")
    free2, _ = torch.cuda.mem_get_info(0)
    # The same with the forward's per-sample record (16 B per sample, resident in HBM): one replay.
    record = torch.empty((sc.render.num_samples, 4), dtype=torch.float32, device="cuda:0")
    img_r, st_r = dev.render("pt", film_precision="fp32", out_precision="fp32", sample_record_ptr=record.data_ptr())
    ga_r, ge_r, rinfo = dev.backward("pt", img_r.astype(np.float32), sample_record_ptr=record.data_ptr())
    free3, _ = torch.cuda.mem_get_info(0)
    log(f"[city] forward with record {st_r.seconds:.2f}s, backward from the record {rinfo['seconds']:.2f}s")
    rec_agree = float(np.abs(ga_r - ga).max() / max(np.abs(ga).max(), 1e-30))
    del record
    dev.close()
    res = {"workload": f"city: 1000x1000 boxes (16,000,034 triangles), log-normal heights, 10k albedo groups, "
                       f"16 quad lights; 3840x2160, {spp} spp ({sc.render.num_samples} samples), max_path_vertices 13, "
                       f"rr_depth 3; renderer pt",
           "forward_s": round(st.seconds, 3),
           "M_path_samples_per_s": round(st.samples / st.seconds / 1e6, 1),
           "Mrays_per_s": round((st.closest_rays + st.shadow_rays) / st.seconds / 1e6, 1),
           "rays_per_sample": round((st.closest_rays + st.shadow_rays) / st.samples, 3),
           "roofline": roof,
           "backward_s": round(binfo["seconds"], 3),
           "backward_over_forward": round(binfo["seconds"] / st.seconds, 3),
           "replay_residual": binfo["replay_residual"],
           "forward_with_record_s": round(st_r.seconds, 3),
           "backward_from_record_s": round(rinfo["seconds"], 3),
           "backward_from_record_over_forward": round(rinfo["seconds"] / st_r.seconds, 3),
           "record_GiB": round(sc.render.num_samples * 16 / 2**30, 2),
           "gradient_rel_diff_record_vs_replays": rec_agree,
           "bvh_build_s": round(info.build_seconds, 2),
           "bvh_device_GiB": round(info.device_bytes / 2**30, 3),
           "hbm_used_forward_GiB": round((free0 - free1) / 2**30, 3),
           "hbm_used_peak_GiB": round((free0 - min(free1, free2)) / 2**30, 3),
           "hbm_used_peak_with_record_GiB": round((free0 - free3) / 2**30, 3),
           "hbm_total_GiB": round(total / 2**30, 1)}
    if not args.no_cpu_baseline:
        from oracle import lmref

        threads = host_threads()
        n = sc.render.num_samples // 64
        t0 = time.time()
        o = lmref.Oracle(sc, fp64=False, accel="qbvh", approx_rsqrt=True)
        log(f"[city] CPU QBVH built in {time.time() - t0:.1f}s")
        _, cst = o.render("pt", num_samples=n, rng="mt", threads=threads)
        res["cpu_baseline"] = {"value": cst["samples"] / cst["seconds"] / 1e6, "unit": "M path-samples/s",
                               "cores": threads, "kind": "port",
                               "sample": f"1/64 of the samples ({n}), FP32 SSE QBVH, mt scheduler, {threads} threads "
                                         f"of {cpu_info()}; the full render extrapolates linearly to "
                                         f"{sc.render.num_samples / (cst['samples'] / cst['seconds']):.0f} s"}
    return res


def cpu_baseline_traversal(sc, rays, sample_rays):
    from oracle import lmref

    threads = host_threads()
    o = lmref.Oracle(sc, fp64=False, accel="qbvh", approx_rsqrt=True)
    sub = rays.slice(0, min(sample_rays, len(rays)))
    t0 = time.perf_counter()
    o.trace_closest(sub, threads=threads)
    dt = time.perf_counter() - t0
    return {"value": len(sub) / dt / 1e6, "unit": "Mrays/s", "cores": threads, "kind": "port",
            "sample": f"first {len(sub)} of the 16M rays, closest hit, FP32 SSE 4-wide QBVH (the reference's "
                      f"default scene), OpenMP over {threads} threads of {cpu_info()}; BVH build excluded"}


def cpu_baseline_pt(sc, samples, renderer="pt"):
    from oracle import lmref

    threads = host_threads()
    o = lmref.Oracle(sc, fp64=False, accel="qbvh", approx_rsqrt=True)
    _, st = o.render(renderer, num_samples=samples, rng="mt", threads=threads)
    return {"value": st["samples"] / st["seconds"] / 1e6, "unit": "M path-samples/s", "cores": threads,
            "kind": "port", "Mrays_per_s": st["rays"] / st["seconds"] / 1e6,
            "sample": f"{samples} path samples of the room scene ({renderer}, mt scheduler, 100 samples per block, "
                      f"std::mt19937 streams), {threads} threads of {cpu_info()}"}


def equal_rmse_check(sc, Device, samples=1 << 20):
    """The room at equal sample counts: the GPU image against the FP64 oracle drawing the same
    Philox streams (arithmetic difference), next to the Monte-Carlo RMSE of one image (from two
    independent GPU renders).  With the estimator identical on both sides, equal sample counts
    give equal RMSE when the first is far below the second."""
    import numpy as np

    from oracle import lmref

    dev = Device(0)
    dev.upload(sc)
    dev.build_bvh()
    g1, _ = dev.render("pt", num_samples=samples, seed=1, film_precision="fp64")
    g2, _ = dev.render("pt", num_samples=samples, seed=2, film_precision="fp64")
    dev.close()
    o1, _ = lmref.Oracle(sc, fp64=True, accel="bvh").render("pt", num_samples=samples, seed=1, threads=host_threads())
    c1, _ = lmref.Oracle(sc, fp64=False, accel="qbvh", approx_rsqrt=True).render(
        "pt", num_samples=samples, seed=1, threads=host_threads())
    mc = rmse(g1, g2) / np.sqrt(2.0)
    return {"samples": samples,
            "rmse_gpu_vs_fp64_oracle_same_streams": rmse(g1, o1),
            "rmse_cpu_fp32_vs_fp64_oracle_same_streams": rmse(c1, o1),
            "monte_carlo_rmse_per_image": mc,
            "gpu_deviation_over_mc_rmse": rmse(g1, o1) / mc}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--triangles", type=int, default=1_000_000)
    ap.add_argument("--rays", type=int, default=16_000_000)
    ap.add_argument("--leaf", type=int, default=4)
    ap.add_argument("--sah-bins", type=int, default=64)
    ap.add_argument("--traversal-cost", type=float, default=1.2)
    ap.add_argument("--pt-steps", type=int, default=5)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-pt", action="store_true")
    ap.add_argument("--no-adjoint", action="store_true")
    ap.add_argument("--no-terrain", action="store_true", help="skip the 2M-triangle terrain leg")
    ap.add_argument("--no-city", action="store_true", help="skip the 16M-triangle city leg")
    ap.add_argument("--cpu-sample-rays", type=int, default=16_000_000)
    ap.add_argument("--cpu-sample-paths", type=int, default=32 * 1_048_576)
    ap.add_argument("--workload", choices=["traversal", "room", "terrain", "city"], default="traversal",
                    help="traversal: the headline line (with every other workload); room: the room renders only; "
                         "terrain: the film-precision study only; city: the 16M-triangle forward + backward only")
    ap.add_argument("--spp", type=int, default=0, help="terrain / city: samples per pixel (0 = the workload's)")
    ap.add_argument("--copy-calibration", type=int, default=0, metavar="MIB",
                    help="only run a plain device-to-device copy of MIB MiB (profiler byte-counter calibration)")
    args = ap.parse_args()
    if args.copy_calibration:
        import torch

        n = args.copy_calibration * (1 << 20) // 4
        a = torch.ones(n, dtype=torch.float32, device="cuda:0")
        b = torch.empty_like(a)
        for _ in range(3):
            b.copy_(a)
        torch.cuda.synchronize()
        print(json.dumps({"copy_bytes_read": n * 4, "copy_bytes_written": n * 4, "launches": 3}), flush=True)
        return 0
    if args.gpus != 1:
        print(f"bench.py measures one GPU; --gpus {args.gpus} is not supported: the path shards by global "
              f"sample index with one film reduction, and only the one-GPU share is measured here.",
              file=sys.stderr)
        return 2
    rank = int(os.environ.get("RANK", "0"))

    import torch

    from lightmetrica_amd import scenes
    from lightmetrica_amd.gpu import Device

    if not torch.cuda.is_available():
        print("bench.py needs a GPU", file=sys.stderr)
        return 1
    if args.workload == "room":
        print(json.dumps(run_pt(args, Device, scenes)[0]), flush=True)
        return 0
    if args.workload == "terrain":
        print(json.dumps(run_terrain_study(args, Device, scenes)), flush=True)
        return 0
    if args.workload == "city":
        print(json.dumps(run_city(args, torch, Device, scenes)), flush=True)
        return 0
    res, sc, rays = run_traversal(args, torch, Device, scenes)
    achieved = res["alg_bytes"] / (res["kernel_ms"] * 1e-3) / 1e9
    traffic = traffic_from_profile()
    line = {
        "metric": METRIC,
        "value": round(res["value"], 2),
        "unit": "Mrays/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(res["ms_per_step"], 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "fp32",
        "data": "synthetic",
        "config": {
            "workload": f"traversal microbench: {args.triangles} triangles (centroids U[0,1]^3, vertices + "
                        f"N(0,0.01)), {args.rays} rays (origins U[-0.5,1.5]^3, directions uniform on the sphere), "
                        f"closest hit, 4-wide SAH BVH (max leaf {args.leaf}), FP32 traversal with the watertight "
                        f"test, the winner re-evaluated in FP64 (t and barycentrics within 1e-5 of the FP64 "
                        f"oracle)",
            "triangles": args.triangles,
            "rays": args.rays,
            "hit_rate": round(res["hit_rate"], 4),
            "node_visits_per_ray": round(res["node_visits_per_ray"], 2),
            "tri_tests_per_ray": round(res["tri_tests_per_ray"], 2),
            "bvh_nodes": res["bvh"].num_nodes,
            "bvh_depth": res["bvh"].max_depth,
            "bvh_build_s": round(res["bvh"].build_seconds, 2),
        },
        "host_buffers": res["host_buffers"],
        "traversal_modes": res["modes"],
        "roofline": {
            "bound": "hbm",
            "achieved": round(achieved, 1),
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": round(achieved / HBM_PEAK_GBS, 4),
            "traffic": traffic,
            "kernel": "k_trace_record + k_refine_fp64",
            "kernel_ms": round(res["kernel_ms"], 4),
            "alg_bytes_per_launch": int(res["alg_bytes"]),
        },
    }
    if not args.no_pt:
        pt, room = run_pt(args, Device, scenes)
        line["path_tracing"] = pt
    if not args.no_adjoint:
        line["adjoint"] = run_adjoint(args, Device, scenes)
    # The large-scene workloads, each on its own context; a failure is reported in the line.
    for key, skip, fn in (("terrain", args.no_terrain, lambda: run_terrain_study(args, Device, scenes)),
                          ("city", args.no_city, lambda: run_city(args, torch, Device, scenes))):
        if skip:
            continue
        try:
            line[key] = fn()
        except Exception as e:  # noqa: BLE001 -- reported, never hidden
            log(f"[bench] {key} failed: {e!r}")
            line[key] = {"error": repr(e)}
        torch.cuda.empty_cache()
    if not args.no_cpu_baseline and rank == 0:
        line["id_parity"] = id_parity(sc, rays, res.pop("gpu_hits"))
        line["cpu_baseline"] = cpu_baseline_traversal(sc, rays, args.cpu_sample_rays)
        if not args.no_pt:
            line["path_tracing"]["cpu_baseline"] = cpu_baseline_pt(room, args.cpu_sample_paths)
            line["path_tracing"]["equal_rmse"] = equal_rmse_check(room, Device)
            line["path_tracing"]["speedup_vs_cpu"] = round(
                line["path_tracing"]["M_path_samples_per_s"] / line["path_tracing"]["cpu_baseline"]["value"], 1)
            for renderer, r in line["path_tracing"]["renderers"].items():
                r["cpu_baseline"] = cpu_baseline_pt(room, args.cpu_sample_paths // 4, renderer)
                r["speedup_vs_cpu"] = round(r["M_path_samples_per_s"] / r["cpu_baseline"]["value"], 1)
        line["speedup_vs_cpu"] = round(line["value"] / line["cpu_baseline"]["value"], 1)
    if rank == 0:
        print(json.dumps(line), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
