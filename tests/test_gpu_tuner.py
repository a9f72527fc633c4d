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


@pytest.mark.parametrize("wide", [False, True])
def test_frame_tuner_leaves_out_equal_candidates(torch_cuda, hip_ctx, wide):
    """Two samples at most: one candidate per tracer on the binary tree, two per
    tracer on the 4-wide one, two with two samples in flight, three limits of
    parked leaves."""
    sc = hiprt.HostScene.generate(2)
    cam = sc.cam.copy()
    cam[10], cam[11] = 96, 54
    bvh = hiprt.Bvh(sc)
    ds = hiprt.DeviceScene(hip_ctx, sc, bvh)
    ds4 = hiprt.DeviceScene(hip_ctx, sc, bvh, hiprt.BVH4) if wide else None
    print(f"case: frame tuner, 96 x 54, 4-wide tree {wide}", flush=True)
    kw, info = hiprt.pt_autotune(ds, ds4, cam, max_samples=2)
    assert info["candidates"] == (2 + 4 * wide) + 2 + 3
    if info["layout"] == "bvh2":
        assert kw["stack_config"] == 0
    for x in (ds, ds4):
        if x is not None:
            x.close()
