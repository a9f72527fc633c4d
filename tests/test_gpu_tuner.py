"""What the tuners return: a default grid, so that the launch's rules by batch
size apply to a tuned caller, and no option that the chosen kernel does not
read."""
import numpy as np
import pytest

import hiprt
from parity import uniform_sphere_rays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("any_hit", [False, True])
def test_tuned_options_keep_the_default_grid(torch_cuda, hip_ctx, any_hit):
    torch = torch_cuda
    print(f"case: autotune 3,000 triangles, 5,001 rays, any-hit {any_hit}", flush=True)
    sc = hiprt.HostScene.random(3000, 0.05, 5)
    bvh = hiprt.Bvh(sc)
    n = 5001
    rays = torch.from_numpy(np.ascontiguousarray(uniform_sphere_rays(n, 3))).cuda()
    res, tuned = hiprt.autotune(hip_ctx, sc, bvh, rays, any=any_hit)
    print(res)
    assert res["blocks"] == 0 and res["mrays_per_s"] > 0
    if res["bvh_format"] == "bvh2":
        assert res["stack_config"] == 0
    ds = hiprt.DeviceScene(hip_ctx, sc, bvh)
    kw = dict(tracer=res["tracer"], refill_threshold=res["refill_threshold"], blocks=res["blocks"],
              stack_config=res["stack_config"], work_chunks=res["work_chunks"])
    got, want = hiprt.new_hits(n), hiprt.new_hits(n)
    hiprt.trace_closest(tuned, rays, got, park_leaves=res["park_leaves"], **kw)
    hiprt.trace_closest(ds, rays, want)
    occ, occ_want = (torch.full((n,), 7, dtype=torch.uint8, device="cuda") for _ in range(2))
    hiprt.trace_any(tuned, rays, occ, **kw)
    hiprt.trace_any(ds, rays, occ_want)
    torch.cuda.synchronize()
    assert torch.equal(got["t"], want["t"]) and torch.equal(occ, occ_want)
    tuned.close()
    ds.close()
