"""Batches around the size up to which several lanes trace one ray, which
depends on the tree: trees of one leaf, of a few and of many nodes, a closed
hall, trees built on the device and an upload whose boxes say nothing about
its rays.  The hits are those of the counting kernel, bit for bit, at every
size; occlusion agrees with them."""
import numpy as np
import pytest

import hiprt
from parity import uniform_sphere_rays
from test_gpu_refit import ctypes_upload

pytestmark = pytest.mark.gpu


def _same(torch, ds, dev):
    n = dev.shape[1]
    got, want = hiprt.new_hits(n), hiprt.new_hits(n)
    stats = torch.zeros(2, dtype=torch.int64, device="cuda")
    hiprt.trace_closest(ds, dev, got)
    hiprt.trace_closest(ds, dev, want, fetch_stats=stats)
    occ = torch.full((n,), 7, dtype=torch.uint8, device="cuda")
    hiprt.trace_any(ds, dev, occ)
    torch.cuda.synchronize()
    for k in got:
        assert torch.equal(got[k].view(torch.int32), want[k].view(torch.int32)), (n, k)
    assert torch.equal(occ.bool(), want["t"] < 3e38), n


@pytest.mark.parametrize("scene", [1, 30, 500, 3000, "hall", "built 500", "built 3", "huge boxes"])
def test_sizes(torch_cuda, hip_ctx, scene):
    torch = torch_cuda
    built = isinstance(scene, str) and scene.startswith("built")
    n_tris = int(scene.split()[1]) if built else 500 if scene == "huge boxes" else scene
    sc = hiprt.HostScene.generate(2) if scene == "hall" else hiprt.HostScene.random(n_tris, 0.05, 5)
    if built:
        pos, idx, _ = sc.arrays()
        ds, _ = hiprt.build_device_scene(hip_ctx, torch.from_numpy(pos).cuda(),
                                         torch.from_numpy(idx.view(np.int32)).cuda())
    else:
        ds = hiprt.DeviceScene(hip_ctx, sc, hiprt.Bvh(sc))
    if scene == "huge boxes":
        nodes, recs, ids = ds.download()
        f = np.ascontiguousarray(nodes).view(np.float32).reshape(-1, 16)
        f[:, 0:12:2], f[:, 1:12:2] = -3.4e38, 3.4e38   # their surface overflows
        ds.close()
        like, ds = ds, ctypes_upload(hip_ctx, f, recs, ids, ds)
    rays = uniform_sphere_rays(700_001, 3)
    if scene == "hall":
        rays[0:3] = rays[0:3] * 2 + np.float32([[19], [6], [6]])
    dev = torch.from_numpy(np.ascontiguousarray(rays)).cuda()
    for n in (1, 65536, 65537, 150_000, 300_000, 390_000, 585_000, 700_001):
        print(f"case: {scene}, {n} rays", flush=True)
        _same(torch, ds, dev[:, :n].contiguous())
    ds.close()
