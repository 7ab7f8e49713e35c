"""A ray's result does not depend on the batch it is traced in: 64, 16 or one lane per ray, on device
arrays or in chunks from the host, whatever rays share its wave.  On geometry where the FP32
triangle test and the boxes disagree most: rays along edges and in the planes of triangles that are
slivers, lie on their boxes' faces, or are large against the origin's coordinates.

No difference is admissible: every kernel evaluates a record by the same operations, accepts it if
its leaf's box as built accepts the ray, and orders what it accepts by one distance."""
import numpy as np
import pytest

from lightmetrica_amd import scenes

pytestmark = pytest.mark.gpu

NRAYS = 8000
FRAMES = 40  # a multiple of the rays, each time in another order


def make(kind):
    r = np.random.default_rng({"slivers": 1, "walls": 2, "large": 3, "edge-on": 4}[kind])
    if kind == "slivers":      # edges of 1 and 1e-2 ... 1e-6
        a = r.uniform(0, 1, (600, 3))
        b = a + r.normal(size=(600, 3)) * 0.5
        c = a + (b - a) * r.uniform(0, 1, (600, 1)) + r.normal(size=(600, 3)) * 10.0 ** r.uniform(-6, -2, (600, 1))
        v = np.stack([a, b, c], 1)
    elif kind == "walls":      # sides of boxes on a grid: edges in box faces, shared by triangles
        lo = r.integers(0, 12, (60, 3)) / 3.0
        hi = lo + r.integers(1, 6, (60, 3)) / 3.0
        corner = np.array([[i & 1, i >> 1 & 1, i >> 2 & 1] for i in range(8)], float)
        p = lo[:, None] + corner[None] * (hi - lo)[:, None]
        quads = [(0, 1, 3, 2), (4, 5, 7, 6), (0, 1, 5, 4), (2, 3, 7, 6), (0, 2, 6, 4), (1, 3, 7, 5)]
        v = np.concatenate([np.concatenate([p[:, [q[0], q[1], q[2]]], p[:, [q[0], q[2], q[3]]]]) for q in quads])
    elif kind == "large":      # sides of 100 and 10,000 past points near the origin, in planes of
        # constant x, y or z, each with an edge along its box's
        n, ax = 600, np.arange(600) % 3
        ay, az, row = (ax + 1) % 3, (ax + 2) % 3, np.arange(600)
        near = r.normal(size=(n, 3)).astype(np.float32).astype(np.float64)
        side = np.where(row % 2 == 0, 100.0, 1e4)
        v = np.repeat(near[:, None], 3, 1)
        v[row, 0, az] -= r.uniform(0, 1, n) * side
        v[row, 1, az] += r.uniform(0, 1, n) * side
        v[row, 2, ay] += r.normal(size=n) * side
        v[row, 2, az] += r.normal(size=n) * side
    else:                      # a fan of almost parallel layers, seen along them
        v = r.uniform(-1, 1, (600, 3, 3)) * np.array([30.0, 30.0, 1e-4]) + np.array([0, 0, 1.0]) * np.arange(600)[:, None, None] * 1e-5
    v = v.astype(np.float32)
    k = r.integers(0, len(v), NRAYS)
    T = v[k].astype(np.float64)
    s, u = r.uniform(0, 1, (2, NRAYS, 1))
    on_edge = T[:, 0] + s * (T[:, 1] - T[:, 0])
    inside = on_edge + u * (T[:, 2] - on_edge)
    target = np.where(np.arange(NRAYS)[:, None] % 4 == 0, inside, np.where(np.arange(NRAYS)[:, None] % 4 == 1, T[:, 2], on_edge))
    if kind == "large":  # past the edge's near point, by less than the FP32 test can tell
        target = near[k] + 10.0 ** r.uniform(-7.5, -3.5, (NRAYS, 1)) * r.normal(size=(NRAYS, 3))
    o = r.normal(size=(NRAYS, 3))
    # every other origin in the target triangle's plane (or near it, rounded)
    w = r.normal(size=(NRAYS, 2, 1)) * 3.0
    plane = T[:, 0] + w[:, 0] * (T[:, 1] - T[:, 0]) + w[:, 1] * (T[:, 2] - T[:, 0])
    if kind != "large":
        o = np.where(np.arange(NRAYS)[:, None] % 2 == 1, plane, o)
    d = target - o
    n = np.linalg.norm(d, axis=1, keepdims=True)
    d = np.where(n > 0, d / np.where(n > 0, n, 1), [0.0, 0.0, 1.0])
    tmax = np.full(NRAYS, scenes.FLT_MAX, np.float32)
    tmax[::3] = n[::3, 0]  # a third of them end at the target
    tmin = np.zeros(NRAYS, np.float32)
    if kind == "large":  # little else around the target
        tmin, tmax = 0.8 * n[:, 0], 1.2 * n[:, 0]
    rays = scenes.Rays(o.astype(np.float32), d.astype(np.float32), tmin.astype(np.float32), tmax.astype(np.float32))
    P = v.reshape(-1, 3)
    return scenes.Scene(kind, P, np.zeros_like(P), np.arange(len(P), dtype=np.uint32).reshape(-1, 3)), rays


@pytest.mark.parametrize("leaf", [1, 4, 16])
@pytest.mark.parametrize("kind", ["slivers", "walls", "large", "edge-on"])
def test_results_do_not_depend_on_the_batch(gpu, kind, leaf):
    sc, rays = make(kind)
    gpu.upload(sc)
    gpu.build_bvh(max_leaf_size=leaf)
    r = np.random.default_rng(7)
    pick = np.concatenate([r.permutation(NRAYS) for _ in range(FRAMES)])
    want = {f: [np.asarray(x).copy() for x in gpu.trace_closest(rays, refine_fp64=f)] for f in (False, True)}
    any_want = gpu.trace_any(rays)
    hit = want[True][3] >= 0
    assert 0.2 < hit.mean() < 1.0
    np.testing.assert_array_equal(any_want, hit)
    for n in (100, 40_000, 65_537, 98_305, 320_000):  # 64, 16, 1 (any hit 16), 1 lanes; host chunks
        part = pick[:n]
        many = scenes.Rays(rays.o[part], rays.d[part], rays.tmin[part], rays.tmax[part])
        for fp64 in (False, True):
            got = gpu.trace_closest(many, refine_fp64=fp64)
            for name, a, b in zip(("prim", "t", "b0", "b1"), (got[3], *got[:3]), (want[fp64][3], *want[fp64][:3])):
                bad = np.flatnonzero(~((a == b[part]) | (np.isnan(a) & np.isnan(b[part]))))
                assert len(bad) == 0, f"n {n} fp64 {fp64} {name}: {len(bad)} rays differ, first {bad[:3]}"
        np.testing.assert_array_equal(gpu.trace_any(many), any_want[part], err_msg=f"n {n}")


@pytest.mark.parametrize("n", [100, 40_000, 120_000])
def test_hits_behind_the_origin(gpu, n):
    """Intervals of negative distances, among boxes without extent: whether -d hits in (-T, 0) is
    whether d does in (0, T), as the triangle test is the same but for the sign of t."""
    r = np.random.default_rng(11)
    v = r.uniform(0, 1, (600, 1, 3)) + r.normal(size=(600, 3, 3)) * 0.1
    flat = np.arange(600)
    v[flat, :, flat % 3] = v[flat, :1, flat % 3]
    P = v.reshape(-1, 3).astype(np.float32)
    gpu.upload(scenes.Scene("flat", P, np.zeros_like(P), np.arange(len(P), dtype=np.uint32).reshape(-1, 3)))
    gpu.build_bvh()
    o = r.uniform(-0.5, 1.5, (n, 3)).astype(np.float32)
    d = r.normal(size=(n, 3))
    d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    T, zero = r.uniform(0.1, 3.0, n).astype(np.float32), np.zeros(n, np.float32)
    ahead = gpu.trace_any(scenes.Rays(o, d, zero, T))
    back = scenes.Rays(o, -d, -T, zero)
    assert 0.1 < ahead.mean() < 0.9
    np.testing.assert_array_equal(gpu.trace_any(back), ahead)
    np.testing.assert_array_equal(gpu.trace_closest(back)[3] >= 0, ahead)
