"""Host rays and films on their way through pinned memory, at the sizes where the way changes."""
import numpy as np
import pytest

from lightmetrica_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 1024, 1025, 65_536, 65_537, 300_003])
def test_host_rays_of_any_number(gpu, n):
    """Read and written in place, copied in one piece, in chunks: the results of device arrays."""
    torch = pytest.importorskip("torch")
    r = np.random.default_rng(n)
    v = (r.uniform(0.0, 1.0, (300, 1, 3)) + r.normal(0.0, 0.1, (300, 3, 3))).reshape(-1, 3).astype(np.float32)
    gpu.upload(scenes.Scene("soup", v, np.zeros_like(v), np.arange(900, dtype=np.uint32).reshape(-1, 3)))
    gpu.build_bvh()
    d = r.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    rays = scenes.Rays(r.uniform(-0.5, 1.5, (n, 3)).astype(np.float32), d.astype(np.float32),
                       np.zeros(n, np.float32), np.full(n, scenes.FLT_MAX, np.float32))
    cols = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (*rays.o.T, *rays.d.T, rays.tmin, rays.tmax)]
    out = [torch.empty(n, device="cuda") for _ in range(3)] + [torch.empty(n, dtype=torch.int32, device="cuda")]
    occ = torch.empty(n, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    gpu.trace_closest_device([c.data_ptr() for c in cols], [c.data_ptr() for c in out], n, refine_fp64=True)
    gpu.trace_any_device([c.data_ptr() for c in cols], occ.data_ptr(), n)
    gpu.synchronize()
    for host, dev in zip(gpu.trace_closest(rays, refine_fp64=True), out):
        np.testing.assert_array_equal(host, dev.cpu().numpy())
    np.testing.assert_array_equal(gpu.trace_any(rays), occ.cpu().numpy().astype(bool))


@pytest.mark.parametrize("width,height", [(1, 1), (208, 210), (209, 209), (512, 171), (800, 600)])
def test_host_films_of_any_size(gpu, width, height):
    """Resolved in place (208 x 210 is the largest), in one slot, in a ring that wraps: the film of a
    device buffer.  FP64 sums of some dozen terms a pixel in any order: within 1e-14."""
    torch = pytest.importorskip("torch")
    gpu.upload(scenes.room_scene(width, height, 2))
    gpu.build_bvh()
    film, _ = gpu.render("pt", film_precision="fp64")
    dev = torch.full((height, width, 3), -1.0, dtype=torch.float64, device="cuda")
    gpu.render("pt", film_precision="fp64", device_out_ptr=dev.data_ptr())
    np.testing.assert_allclose(film, dev.cpu().numpy(), rtol=1e-14, atol=0)
