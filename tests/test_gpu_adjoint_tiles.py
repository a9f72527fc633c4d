"""Vertex gradients on both sides of the switch of the sort's tile: the sums
over the rays of each triangle against the caller's per-ray corner gradients
added in float64."""
import numpy as np
import pytest

import hiprt
from parity import uniform_sphere_rays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1023, 1024, 1025, 9 * 1024 + 5, 100_003, 1 << 20, (1 << 20) + 1])
def test_vertex_gradients(torch_cuda, hip_ctx, n):
    print(f"case: {n} rays", flush=True)
    torch = torch_cuda
    sc = hiprt.HostScene.random(70_000, 0.02, 3)
    _, idx, _ = sc.arrays()
    ds = hiprt.DeviceScene(hip_ctx, sc, hiprt.Bvh(sc))
    rays = torch.from_numpy(uniform_sphere_rays(n, 2)).cuda()
    hits = hiprt.new_hits(n)
    hiprt.trace_closest(ds, rays, hits)
    g = [torch.randn(n, device="cuda", generator=torch.Generator(device="cuda").manual_seed(k)) for k in range(3)]
    nv = int(idx.max()) + 1
    gv = torch.zeros((nv, 3), device="cuda")
    corners = torch.zeros((n, 9), device="cuda")
    hiprt.adjoint_closest(ds, rays, hits, *g, grad_vertices=gv)
    hiprt.adjoint_closest(ds, rays, hits, *g, grad_corners=corners)
    torch.cuda.synchronize()
    hit = hits["t"] < 3e38
    assert float(hit.float().mean()) > 0.1
    tri = torch.from_numpy(idx.astype(np.int64)).cuda()[hits["id"].long().clamp(min=0)]
    c = torch.where(hit[:, None], corners, torch.zeros_like(corners)).double().reshape(n, 3, 3)
    want = torch.zeros((nv, 3), dtype=torch.float64, device="cuda")
    size = torch.zeros((nv, 3), dtype=torch.float64, device="cuda")
    rays_of = torch.zeros(nv, dtype=torch.float64, device="cuda")
    for k in range(3):
        want.index_add_(0, tri[:, k], c[:, k])
        size.index_add_(0, tri[:, k], c[:, k].abs())
        rays_of.index_add_(0, tri[:, k], hit.double())
    # float32 sums of m terms in any order: at most m ulps of the terms' magnitudes
    bound = (rays_of[:, None] + 1) * 2.0 ** -23 * size + 1e-30
    assert bool(((gv.double() - want).abs() <= bound).all())
    ds.close()
