"""The group trace (several lanes per ray, the kernel of small batches) against
the oracle, bit for bit: batch sizes around a block's rays and around the
switches between 16 lanes, 8 lanes and the one-ray-per-lane kernels; leaves of
up to 32 triangles (larger than a step's four, than 8 and than 16 lanes);
scenes made of exact and near ties in flat boxes, where the rays that meet a
hit in a possibly culled leaf start over; both triangle formats; opacity.  The
persistent kernels, which a caller's own grid selects at any size, are held
to the same hits."""
import numpy as np
import pytest

import hiprt
import oracle_py as orc
from parity import bit_exact, classify, uniform_sphere_rays
from test_gpu_spill import nested_rays, nested_scene

pytestmark = pytest.mark.gpu


def _closest(torch, ds, rays, tracer="while-while", **kw):
    h = hiprt.new_hits(rays.shape[1])
    for x in h.values():
        x.fill_(-5)
    hiprt.trace_closest(ds, torch.from_numpy(rays).cuda(), h, tracer=tracer, **kw)
    torch.cuda.synchronize()
    return tuple(h[k].cpu().numpy() for k in ("t", "u", "v")) + (h["id"].cpu().numpy().view(np.uint32),)


def _any(torch, ds, rays, tracer="while-while", **kw):
    occ = torch.full((rays.shape[1],), 7, dtype=torch.uint8, device="cuda")
    hiprt.trace_any(ds, torch.from_numpy(rays).cuda(), occ, tracer=tracer, **kw)
    torch.cuda.synchronize()
    return occ.cpu().numpy()


def _check(torch, ctx, sc, bvh, rays, tracers=("while-while", "dynamic-while-while")):
    pos, idx, _ = sc.arrays()
    want = orc.trace_closest(pos, idx, bvh.nodes, bvh.root, bvh.index, rays)
    want_any = orc.trace_any(pos, idx, bvh.nodes, bvh.root, bvh.index, rays)
    ds = hiprt.DeviceScene(ctx, sc, bvh)
    for tracer in tracers:
        assert bit_exact(_closest(torch, ds, rays, tracer), want), tracer
        assert np.array_equal(_any(torch, ds, rays, tracer), want_any), tracer
    ds.close()
    return want


@pytest.fixture(scope="module")
def soup():
    sc = hiprt.HostScene.random(3000, 0.03, 5)
    return sc, hiprt.Bvh(sc)


@pytest.mark.parametrize("n", [1, 3, 4, 15, 16, 17, 33, 4095, 65535, 65536, 65537, 65569, 200003])
def test_batch_sizes(torch_cuda, hip_ctx, soup, n):
    print(f"case: {n} rays", flush=True)
    _check(torch_cuda, hip_ctx, *soup, uniform_sphere_rays(n, n))


@pytest.mark.parametrize("n", [655360, 655361, 1048576, 1048577])
def test_switch_to_one_ray_per_lane(torch_cuda, hip_ctx, soup, n):
    print(f"case: {n} rays, the largest group batch", flush=True)
    _check(torch_cuda, hip_ctx, *soup, uniform_sphere_rays(n, 3), tracers=("while-while", "persistent-while-while"))


@pytest.mark.parametrize("max_tris", [1, 4, 5, 9, 17, 32])
@pytest.mark.parametrize("n", [5000, 70000])
def test_large_leaves(torch_cuda, hip_ctx, max_tris, n):
    print(f"case: leaves of up to {max_tris} triangles, {n} rays", flush=True)
    sc = hiprt.HostScene.random(1500, 0.08, 6)
    _check(torch_cuda, hip_ctx, sc, hiprt.Bvh(sc, max_tris=max_tris, esc=False), uniform_sphere_rays(n, 11))


def _stacked_quads(seed, axis):
    """Axis-aligned quads, many in one plane and many a few ulps apart, split
    into triangles both ways: flat boxes whose entry distances and hit
    distances differ by rounding only."""
    rng = np.random.default_rng(seed)
    pos, idx = [], []
    for k in range(400):
        z = np.float32(0.5) + np.float32(rng.integers(0, 4)) * np.float32(6e-8)
        c = rng.uniform(0.2, 0.8, 2)
        s = rng.uniform(0.05, 0.4, 2)
        q = np.array([[c[0] - s[0], c[1] - s[1], z], [c[0] + s[0], c[1] - s[1], z],
                      [c[0] + s[0], c[1] + s[1], z], [c[0] - s[0], c[1] + s[1], z]], np.float32)
        b = len(pos)
        pos.extend(np.roll(q, axis, axis=1))
        idx.extend(([b, b + 1, b + 2], [b, b + 2, b + 3]) if k & 1 else ([b, b + 1, b + 3], [b + 1, b + 2, b + 3]))
    return hiprt.HostScene.from_arrays(np.array(pos, np.float32), np.array(idx, np.uint32))


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("n", [20000, 100000])
def test_ties_in_flat_boxes(torch_cuda, hip_ctx, axis, n):
    print(f"case: stacked quads, axis {axis}, {n} rays", flush=True)
    sc = _stacked_quads(2 + axis, axis)
    want = _check(torch_cuda, hip_ctx, sc, hiprt.Bvh(sc, max_tris=1, esc=False), uniform_sphere_rays(n, 8))
    assert (want[0] < 3e38).mean() > 0.1
    _check(torch_cuda, hip_ctx, sc, hiprt.Bvh(sc), uniform_sphere_rays(n, 9))


def test_woop_records(torch_cuda, hip_ctx, soup):
    torch = torch_cuda
    sc, bvh = soup
    ds = hiprt.DeviceScene(hip_ctx, sc, bvh, hiprt.BVH2, hiprt.TRI_WOOP)
    for n in (3000, 80000):
        rays = uniform_sphere_rays(n, 4)
        # the counting variant is the plain one-ray-per-lane kernel
        stats = torch.zeros(2, dtype=torch.int64, device="cuda")
        assert bit_exact(_closest(torch, ds, rays), _closest(torch, ds, rays, fetch_stats=stats))
    ds.close()


@pytest.mark.parametrize("tracer", hiprt.TRACERS[1:])
@pytest.mark.parametrize("stack", [0, 1, 2, 3, 4])
def test_own_grid_selects_the_persistent_kernel(torch_cuda, hip_ctx, soup, tracer, stack):
    torch = torch_cuda
    sc, bvh = soup
    pos, idx, _ = sc.arrays()
    rays = uniform_sphere_rays(30000, 12)
    want = orc.trace_closest(pos, idx, bvh.nodes, bvh.root, bvh.index, rays)
    ds = hiprt.DeviceScene(hip_ctx, sc, bvh)
    got = _closest(torch, ds, rays, tracer, stack_config=stack, blocks=64)
    if tracer == "persistent-while-while":
        assert bit_exact(got, want)
    else:
        assert classify(orc, pos, idx, rays, got, want)["unexplained"] == 0
    ds.close()


def test_alpha_and_batch(torch_cuda, hip_ctx):
    """Opacity decides hits inside a group, and a descriptor table's small
    scenes trace like single launches."""
    torch = torch_cuda
    scenes = []
    for k in range(3):
        base = hiprt.HostScene.random(1000 + 700 * k, 0.05, 30 + k)
        pos, idx, _ = base.arrays()
        sc = hiprt.HostScene.from_arrays(pos, idx, np.zeros(len(idx), np.uint32))
        tc = np.random.default_rng(k).uniform(-1, 2, (len(pos), 2)).astype(np.float32)
        sc.set_texcoords(tc)
        tex = np.ones((8, 8, 4), np.float32)
        tex[::2, :, 3] = 0.1
        sc.set_texture(0, tex)
        bvh = hiprt.Bvh(sc)
        rays = uniform_sphere_rays(4000 + 999 * k, 50 + k)
        alpha = orc.Alpha(tc, np.zeros(len(idx), np.uint32), {0: tex}, 1)
        want = orc.trace_closest_alpha(pos, idx, bvh.nodes, bvh.root, bvh.index, rays, alpha)
        ds = hiprt.DeviceScene(hip_ctx, sc, bvh)
        assert bit_exact(_closest(torch, ds, rays, "while-while-alpha"), want)
        scenes.append((ds, torch.from_numpy(rays).cuda(), hiprt.new_hits(rays.shape[1]), want))
    hiprt.trace_batch([s[:3] + (None,) for s in scenes], tracer="dynamic-while-while-alpha")
    torch.cuda.synchronize()
    for ds, _, h, want in scenes:
        got = tuple(h[k].cpu().numpy() for k in ("t", "u", "v")) + (h["id"].cpu().numpy().view(np.uint32),)
        assert bit_exact(got, want)
        ds.close()


def test_deep_tree(torch_cuda, hip_ctx):
    """The nested triangles' 38-level tree: the group kernel's list, and the
    plain kernel's LDS stack (its counting variant)."""
    torch = torch_cuda
    pos, idx = nested_scene()
    sc = hiprt.HostScene.from_arrays(pos, idx)
    bvh = hiprt.Bvh(sc, max_tris=1)
    ds = hiprt.DeviceScene(hip_ctx, sc, bvh)
    assert 24 < ds.stack_need < 64, ds.stack_need
    for n in (4000, 70000):
        rays = nested_rays(n, n)
        want = orc.trace_closest(pos, idx, bvh.nodes, bvh.root, bvh.index, rays)
        assert bit_exact(_closest(torch, ds, rays), want)
        stats = torch.zeros(2, dtype=torch.int64, device="cuda")
        assert bit_exact(_closest(torch, ds, rays, fetch_stats=stats), want)
    ds.close()
