"""Closest and any hits of the postponing kernel on both sides of the sizes at
which its default grid changes, trees on both sides of each depth: every ray is
traced once, whatever the grid.  Checked against the plain kernel, which has no
work counters."""
import numpy as np
import pytest

import hiprt
from parity import uniform_sphere_rays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_tris", [40, 2000, 9000, 40000])   # stack needs about 6, 12, 14, 17
@pytest.mark.parametrize("n", [(1 << 20), (1 << 20) + 1, (1 << 21), (1 << 21) + 1])
def test_every_ray_once(torch_cuda, hip_ctx, n_tris, n):
    torch = torch_cuda
    sc = hiprt.HostScene.random(n_tris, 0.02 * (8192.0 / n_tris) ** (1.0 / 3.0), 3)
    ds = hiprt.DeviceScene(hip_ctx, sc, hiprt.Bvh(sc))
    print(f"case: {n_tris} triangles, stack need {ds.stack_need}, {n} rays", flush=True)
    dev = torch.from_numpy(np.ascontiguousarray(uniform_sphere_rays(n, 4))).cuda()
    want, got = hiprt.new_hits(n), hiprt.new_hits(n)
    occ, occ_want = (torch.full((n,), 7, dtype=torch.uint8, device="cuda") for _ in range(2))
    hiprt.trace_closest(ds, dev, want)
    hiprt.trace_any(ds, dev, occ_want)
    for tracer in ("persistent-speculative-while-while", "dynamic-while-while"):
        for x in got.values():
            x.fill_(-5)
        occ.fill_(7)
        hiprt.trace_closest(ds, dev, got, tracer=tracer)
        hiprt.trace_any(ds, dev, occ, tracer=tracer)
        torch.cuda.synchronize()
        assert torch.equal(got["t"], want["t"])       # (an equal-t tie may name the other triangle)
        assert float((got["id"] != want["id"]).float().mean()) <= 1e-4
        assert torch.equal(occ, occ_want)
    ds.close()
