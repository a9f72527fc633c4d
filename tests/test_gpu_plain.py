"""The plain kernel's postponed leaves, which batches above the group trace's
take, against its counting variant, which postpones nothing and visits nodes
in the reference's order: the hits must agree to the bit.  Scenes of exact and
near ties in flat boxes, one-triangle and large leaves, trees refitted and
built on the device, a deep tree, rays with non-finite components, both
triangle formats, opacity, and an uploaded tree whose boxes are not nested."""
import numpy as np
import pytest

import hiprt
from test_gpu_dynamic import _rays
from test_gpu_group import _stacked_quads
from test_gpu_refit import ctypes_upload
from test_gpu_spill import nested_rays, nested_scene

pytestmark = pytest.mark.gpu
N = (1 << 20) + 77   # the smallest batches of this kernel, with a partial wavefront


def _check(torch, ds, rays, tracer="while-while", hits=0.02):
    dev = torch.from_numpy(rays).cuda()
    n = rays.shape[1]
    got, want = hiprt.new_hits(n), hiprt.new_hits(n)
    for x in (*got.values(), *want.values()):
        x.fill_(-5)
    stats = torch.zeros(2, dtype=torch.int64, device="cuda")
    hiprt.trace_closest(ds, dev, got, tracer=tracer)
    hiprt.trace_closest(ds, dev, want, tracer=tracer, fetch_stats=stats)
    occ = torch.full((n,), 7, dtype=torch.uint8, device="cuda")
    hiprt.trace_any(ds, dev, occ, tracer=tracer)
    torch.cuda.synchronize()
    for k in got:
        assert torch.equal(got[k].view(torch.int32), want[k].view(torch.int32)), k
    found = want["t"] < 3e38
    assert float(found.float().mean()) > hits
    finite = torch.from_numpy(np.isfinite(rays).all(0) & (rays[4:7] != 0).all(0)).cuda()
    assert torch.equal(occ[finite], found[finite].to(torch.uint8))


@pytest.mark.parametrize("max_tris", [1, 4, 32])
@pytest.mark.parametrize("tri", [hiprt.TRI_EXACT, hiprt.TRI_WOOP])
def test_soup(torch_cuda, hip_ctx, max_tris, tri):
    print(f"case: soup, leaves of up to {max_tris} triangles, format {tri}", flush=True)
    sc = hiprt.HostScene.random(3000, 0.06, 5)
    ds = hiprt.DeviceScene(hip_ctx, sc, hiprt.Bvh(sc, max_tris=max_tris, esc=max_tris == 4), hiprt.BVH2, tri)
    _check(torch_cuda, ds, _rays(N, 6))
    ds.close()


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("max_tris", [1, 4])
def test_ties_in_flat_boxes(torch_cuda, hip_ctx, axis, max_tris):
    print(f"case: stacked quads, axis {axis}", flush=True)
    sc = _stacked_quads(2 + axis, axis)
    ds = hiprt.DeviceScene(hip_ctx, sc, hiprt.Bvh(sc, max_tris=max_tris, esc=False))
    _check(torch_cuda, ds, _rays(N, 8))
    ds.close()


def test_deep_tree(torch_cuda, hip_ctx):
    pos, idx = nested_scene()
    sc = hiprt.HostScene.from_arrays(pos, idx)
    ds = hiprt.DeviceScene(hip_ctx, sc, hiprt.Bvh(sc, max_tris=1))
    _check(torch_cuda, ds, nested_rays(N, 3), hits=0.001)
    ds.close()


def test_refitted_and_built_trees(torch_cuda, hip_ctx):
    torch = torch_cuda
    sc = hiprt.HostScene.random(3000, 0.06, 15)
    pos, idx, mat = sc.arrays()
    moved = torch.from_numpy((pos + np.random.default_rng(2).normal(0, 0.05, pos.shape)).astype(np.float32)).cuda()
    ds = hiprt.DeviceScene(hip_ctx, sc, hiprt.Bvh(sc))
    ds.refit(moved)
    _check(torch, ds, _rays(N, 16))
    ds.close()
    ds, _ = hiprt.build_device_scene(hip_ctx, moved, torch.from_numpy(idx.view(np.int32)).cuda())
    _check(torch, ds, _rays(N, 17))
    ds.close()


@pytest.mark.parametrize("change", ["shrink", "invert"])
def test_boxes_that_are_not_nested(torch_cuda, hip_ctx, change):
    """An uploaded tree may hold any boxes: children reach out of shrunken or
    inverted parents, and the reference's order and culling still decide."""
    sc = hiprt.HostScene.random(3000, 0.06, 25)
    ds = hiprt.DeviceScene(hip_ctx, sc, hiprt.Bvh(sc))
    nodes, recs, ids = ds.download()
    f = np.ascontiguousarray(nodes).view(np.float32).reshape(-1, 16)
    rng = np.random.default_rng(4)
    for lo, hi in ((0, 1), (2, 3), (4, 5), (6, 7), (8, 9), (10, 11)):
        some = rng.random(len(f)) < 0.2
        if change == "shrink":
            size = f[some, hi] - f[some, lo]
            f[some, lo] += 0.2 * size
            f[some, hi] -= 0.2 * size
        else:
            f[some, lo], f[some, hi] = f[some, hi].copy(), f[some, lo].copy()
    up = ctypes_upload(hip_ctx, f, recs, ids, ds)
    dev, n = torch_cuda.from_numpy(_rays(N, 26)).cuda(), N
    got, want = hiprt.new_hits(n), hiprt.new_hits(n)
    stats = torch_cuda.zeros(2, dtype=torch_cuda.int64, device="cuda")
    hiprt.trace_closest(up, dev, got)
    hiprt.trace_closest(up, dev, want, fetch_stats=stats)
    torch_cuda.cuda.synchronize()
    for k in got:
        assert torch_cuda.equal(got[k].view(torch_cuda.int32), want[k].view(torch_cuda.int32)), k
    up.close()
    ds.close()


def test_opacity(torch_cuda, hip_ctx):
    base = hiprt.HostScene.random(2000, 0.08, 30)
    pos, idx, _ = base.arrays()
    sc = hiprt.HostScene.from_arrays(pos, idx, np.zeros(len(idx), np.uint32))
    sc.set_texcoords(np.random.default_rng(1).uniform(-1, 2, (len(pos), 2)).astype(np.float32))
    tex = np.ones((8, 8, 4), np.float32)
    tex[::2, :, 3] = 0.1
    sc.set_texture(0, tex)
    ds = hiprt.DeviceScene(hip_ctx, sc, hiprt.Bvh(sc))
    _check(torch_cuda, ds, _rays(N, 31), tracer="while-while-alpha")
    ds.close()


@pytest.mark.parametrize("tri", [hiprt.TRI_EXACT, hiprt.TRI_WOOP])
def test_persistent_while_while_is_this_kernel(torch_cuda, hip_ctx, tri):
    """Its own kernel, which a caller's grid selects, returns the same bits;
    so does the allocation-free entry, in a tree that fits its stack and in
    one that spills."""
    torch = torch_cuda
    pos, idx = nested_scene()
    soup = hiprt.HostScene.random(3000, 0.06, 35)
    deep = hiprt.HostScene.from_arrays(pos, idx)
    for sc, max_tris, rays in ((soup, 4, _rays(N, 36)), (deep, 1, nested_rays(N, 37))):
        ds = hiprt.DeviceScene(hip_ctx, sc, hiprt.Bvh(sc, max_tris=max_tris), hiprt.BVH2, tri)
        dev = torch.from_numpy(rays).cuda()
        want, got, free = (hiprt.new_hits(N) for _ in range(3))
        hiprt.trace_closest(ds, dev, want, tracer="persistent-while-while", blocks=512)
        hiprt.trace_closest(ds, dev, got, tracer="persistent-while-while")
        hiprt.trace_closest_noalloc(ds, dev, free, blocks=512)
        occ, occ2 = (torch.full((N,), 7, dtype=torch.uint8, device="cuda") for _ in range(2))
        hiprt.trace_any(ds, dev, occ, tracer="persistent-while-while", blocks=512)
        hiprt.trace_any(ds, dev, occ2, tracer="persistent-while-while")
        torch.cuda.synchronize()
        for k in got:
            assert torch.equal(got[k].view(torch.int32), want[k].view(torch.int32)), k
            assert torch.equal(free[k].view(torch.int32), want[k].view(torch.int32)), k
        assert torch.equal(occ, occ2)
        ds.close()
