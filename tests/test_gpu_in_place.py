"""Results written over the rays' own columns, element by element: every ray is read before its result
is written, whatever the size of the batch."""
import numpy as np
import pytest

from lightmetrica_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("over", [(7, 6, 0, 3), (0, 1, 2, 7), (None, 6, 7, 0), (None, None, None, 4)],
                         ids=["prim-dx", "prim-tmax", "prim-ox", "prim-dy"])
@pytest.mark.parametrize("n", [1000, 50_000, 200_001])
def test_results_over_rays(gpu, n, over):
    torch = pytest.importorskip("torch")
    gpu.upload(scenes.traversal_scene(3000, sigma=0.05))
    gpu.build_bvh()
    host = gpu.ray_columns(scenes.traversal_rays(n))
    for fp64 in (False, True):
        cols = [torch.from_numpy(c).cuda() for c in host]
        out = [torch.full((n,), -7, dtype=torch.int32, device="cuda") for _ in range(4)]
        torch.cuda.synchronize()
        gpu.trace_closest_device([c.data_ptr() for c in cols], [o.data_ptr() for o in out], n, refine_fp64=fp64)
        gpu.synchronize()
        placed = [out[k] if o is None else cols[o] for k, o in enumerate(over)]
        want = [o.cpu().numpy().copy() for o in out]
        gpu.trace_closest_device([c.data_ptr() for c in cols], [p.data_ptr() for p in placed], n, refine_fp64=fp64)
        gpu.synchronize()
        for p, w in zip(placed, want):
            np.testing.assert_array_equal(p.view(torch.int32).cpu().numpy(), w)
