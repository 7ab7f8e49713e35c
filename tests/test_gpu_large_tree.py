"""The nodes as they were built beyond 2 GiB (2^24 nodes of 128 bytes): the kernels of small batches
and the second tracing of ties read them there.  The packed nodes, 64 bytes each and at most 2^25,
end at 2 GiB."""
import numpy as np
import pytest

from lightmetrica_amd import scenes

pytestmark = pytest.mark.gpu


def test_built_nodes_beyond_2gib(gpu):
    """A flat grid of 35M triangles in single-triangle leaves; vertical rays through centroids, each of
    which hits its own triangle at t = 1, and through the middles of diagonals, which tie between two."""
    n = 4200
    g = (np.arange(n + 1, dtype=np.float64) / n).astype(np.float32)
    P = np.zeros(((n + 1) * (n + 1), 3), dtype=np.float32)
    P[:, 0] = np.tile(g, n + 1)
    P[:, 1] = np.repeat(g, n + 1)
    v00 = (np.arange(n, dtype=np.uint32)[:, None] * (n + 1) + np.arange(n, dtype=np.uint32)[None, :]).ravel()
    F = np.empty((2 * n * n, 3), dtype=np.uint32)
    F[0::2, 0], F[0::2, 1], F[0::2, 2] = v00, v00 + 1, v00 + n + 2
    F[1::2, 0], F[1::2, 1], F[1::2, 2] = v00, v00 + n + 2, v00 + n + 1
    gpu.upload(scenes.Scene("grid", P, np.zeros_like(P), F))
    info = gpu.build_bvh(max_leaf_size=1)
    assert info.num_nodes * 128 > 1 << 31
    nt = F.shape[0]
    rng = np.random.default_rng(5)

    def down(xy):
        m = len(xy)
        o = np.concatenate([xy, np.ones((m, 1))], axis=1).astype(np.float32)
        return scenes.Rays(o, np.tile(np.array([0, 0, -1], np.float32), (m, 1)), np.zeros(m, np.float32),
                           np.full(m, scenes.FLT_MAX, np.float32))

    for m in (8192, 65_536):
        k = np.concatenate([rng.integers(0, nt, m - 4000), np.arange(2000), np.arange(nt - 2000, nt)])
        rays = down(P[F[k]].astype(np.float64).mean(axis=1)[:, :2])
        t, b0, b1, prim = gpu.trace_closest(rays)
        np.testing.assert_array_equal(prim, k)
        np.testing.assert_allclose(t, 1.0, rtol=0, atol=1e-6)
        assert gpu.trace_any(rays).all()

    cell = rng.integers(0, n * n, 140_000)
    rays = down((P[v00[cell]].astype(np.float64) + P[v00[cell] + n + 2])[:, :2] / 2)
    many = gpu.trace_closest(rays)
    assert (many[3] // 2 == cell).mean() > 0.99  # some middles round into the neighbours
    for a in range(0, 140_000, 8000):
        part = scenes.Rays(rays.o[a:a + 8000], rays.d[a:a + 8000], rays.tmin[a:a + 8000], rays.tmax[a:a + 8000])
        for x, y in zip(gpu.trace_closest(part), many):
            np.testing.assert_array_equal(x, y[a:a + 8000])
