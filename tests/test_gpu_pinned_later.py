"""Host rays and films of a program that goes on calling: the results of the first calls, by the
runtime's copies, and of the later ones, through pinned memory, are those of device arrays."""
import numpy as np
import pytest

from lightmetrica_amd import scenes
from lightmetrica_amd.gpu import Device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,calls", [(20_000, 9), (65_536, 9), (65_537, 250), (300_003, 70)])
def test_host_rays_before_and_after(n, calls):
    torch = pytest.importorskip("torch")
    r = np.random.default_rng(n)
    with Device(0) as gpu:
        gpu.upload(scenes.traversal_scene(2000, sigma=0.05))
        gpu.build_bvh()
        rays = scenes.traversal_rays(n)
        cols = [torch.from_numpy(c).cuda() for c in gpu.ray_columns(rays)]
        out = [torch.empty(n, device="cuda") for _ in range(3)] + [torch.empty(n, dtype=torch.int32, device="cuda")]
        torch.cuda.synchronize()
        for k in range(calls):
            fp64, turn = bool(k & 1), int(r.integers(n))
            if k < 2:
                gpu.trace_closest_device([c.data_ptr() for c in cols], [c.data_ptr() for c in out], n, refine_fp64=fp64)
                gpu.synchronize()
                want = [o.cpu().numpy() for o in out]
                first = want if k == 0 else first
                second = want if k == 1 else None
            want = first if not fp64 else second
            host = [np.roll(c, turn) for c in gpu.ray_columns(rays)]  # other arrays each time
            for a, b in zip(gpu.trace_closest_columns(host, fp64), want):
                np.testing.assert_array_equal(np.roll(a, -turn), b)


@pytest.mark.parametrize("width,height,calls", [(200, 150, 4), (209, 200, 9), (700, 500, 9), (1280, 720, 12)])
def test_host_films_before_and_after(width, height, calls):
    """FP64 sums of some dozen terms a pixel in any order: within 1e-14."""
    torch = pytest.importorskip("torch")
    with Device(0) as gpu:
        gpu.upload(scenes.room_scene(width, height, 2))
        gpu.build_bvh()
        dev = torch.full((height, width, 3), -1.0, dtype=torch.float64, device="cuda")
        gpu.render("pt", film_precision="fp64", device_out_ptr=dev.data_ptr())
        want, first = dev.cpu().numpy(), gpu.raycast()
        for _ in range(calls):
            film, _ = gpu.render("pt", film_precision="fp64")
            np.testing.assert_allclose(film, want, rtol=1e-14, atol=0)
            np.testing.assert_array_equal(gpu.raycast(), first)
