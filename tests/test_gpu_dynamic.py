"""The postponing kernel with its stack in LDS (one scene, and descriptor
tables) against the oracle: wavefront remainders, refill thresholds, work
counters, parked leaves, triangle formats, opacity, rays with non-finite
components, trees just inside and outside of its stack, a scene that is one
leaf.  A caller's grid selects the kernel at any size; occlusion is compared
exactly, closest hits up to ties."""
import numpy as np
import pytest

import hiprt
import oracle_py as orc
from parity import classify, uniform_sphere_rays
from test_gpu_edge import INF, NAN
from test_gpu_spill import nested_rays, nested_scene

pytestmark = pytest.mark.gpu
SPEC = ("persistent-speculative-while-while", "dynamic-while-while")


@pytest.fixture(scope="module")
def soup():
    sc = hiprt.HostScene.random(3000, 0.03, 5)
    return sc, hiprt.Bvh(sc)


def _rays(n, seed):
    """Short and long rays; some of every hundred with a component that is not finite or a zero direction."""
    rays = uniform_sphere_rays(n, seed)
    rng = np.random.default_rng(seed)
    rays[7] = np.where(rng.random(n) < 0.5, rng.uniform(0.01, 0.5, n), rays[7])
    for k, (row, value) in enumerate(((4, 0.0), (5, INF), (0, NAN), (6, -0.0), (7, NAN))):
        rays[row, 31 + 7 * k::101] = value
    return np.ascontiguousarray(rays, np.float32)


def _any(torch, ds, rays, **kw):
    occ = torch.full((rays.shape[1],), 7, dtype=torch.uint8, device="cuda")
    hiprt.trace_any(ds, torch.from_numpy(rays).cuda(), occ, **kw)
    torch.cuda.synchronize()
    return occ.cpu().numpy()


@pytest.mark.parametrize("tracer", SPEC)
@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 30001])
@pytest.mark.parametrize("blocks,refill,chunks", [(1, 1, 8), (3, 40, 8), (3, 64, 1), (200, 0, 0)])
def test_any_hit(torch_cuda, hip_ctx, soup, tracer, n, blocks, refill, chunks):
    print(f"case: any-hit, {n} rays, {tracer}, {blocks} blocks", flush=True)
    sc, bvh = soup
    pos, idx, _ = sc.arrays()
    rays = _rays(n, n)
    want = orc.trace_any(pos, idx, bvh.nodes, bvh.root, bvh.index, rays)
    ds = hiprt.DeviceScene(hip_ctx, sc, bvh)
    assert np.array_equal(_any(torch_cuda, ds, rays, tracer=tracer, blocks=blocks, refill_threshold=refill,
                               work_chunks=chunks), want)
    ds.close()


@pytest.mark.parametrize("tracer", SPEC)
def test_any_hit_above_the_group_batches(torch_cuda, hip_ctx, soup, tracer):
    sc, bvh = soup
    pos, idx, _ = sc.arrays()
    rays = _rays((1 << 20) + 1, 3)
    want = orc.trace_any(pos, idx, bvh.nodes, bvh.root, bvh.index, rays)
    ds = hiprt.DeviceScene(hip_ctx, sc, bvh)
    assert np.array_equal(_any(torch_cuda, ds, rays, tracer=tracer), want)
    ds.close()


@pytest.mark.parametrize("limit", [0, 1000])
def test_stack_of_the_tree(torch_cuda, hip_ctx, limit):
    """Nested triangles: trees that fill more and more of the LDS column,
    trees beyond it, and a bounded spill column, which keeps the spilling
    kernel."""
    needs = set()
    for n_tris in (12, 60, 90, 95, 100, 105, 110, 120):
        pos, idx = nested_scene()
        idx = np.ascontiguousarray(idx[:n_tris])
        pos = np.ascontiguousarray(pos[:3 * n_tris])
        sc = hiprt.HostScene.from_arrays(pos, idx)
        bvh = hiprt.Bvh(sc, max_tris=1)
        rays = nested_rays(4000, n_tris)
        want = orc.trace_any(pos, idx, bvh.nodes, bvh.root, bvh.index, rays)
        ds = hiprt.DeviceScene(hip_ctx, sc, bvh)
        print(f"case: {n_tris} nested triangles, stack need {ds.stack_need}", flush=True)
        needs.add(ds.stack_need)
        for tracer in SPEC:
            for stack in (0, 4):
                assert np.array_equal(_any(torch_cuda, ds, rays, tracer=tracer, blocks=5, stack_config=stack,
                                           spill_limit=limit), want)
        ds.close()
    assert min(needs) < 32 < max(needs), needs


def _closest(torch, ds, rays, **kw):
    h = hiprt.new_hits(rays.shape[1])
    for x in h.values():
        x.fill_(-5)
    hiprt.trace_closest(ds, torch.from_numpy(rays).cuda(), h, **kw)
    torch.cuda.synchronize()
    return tuple(h[k].cpu().numpy() for k in ("t", "u", "v")) + (h["id"].cpu().numpy().view(np.uint32),)


@pytest.mark.parametrize("tracer", SPEC)
@pytest.mark.parametrize("n", [1, 64, 257, 30001])
@pytest.mark.parametrize("blocks,refill,chunks,park", [(1, 1, 8, 1), (3, 40, 8, 2), (3, 64, 1, 3), (200, 0, 0, 4)])
def test_closest_hit(torch_cuda, hip_ctx, soup, tracer, n, blocks, refill, chunks, park):
    print(f"case: closest hit, {n} rays, {tracer}, {blocks} blocks, {park} parked leaves", flush=True)
    sc, bvh = soup
    pos, idx, _ = sc.arrays()
    rays = _rays(n, n)
    want = orc.trace_closest(pos, idx, bvh.nodes, bvh.root, bvh.index, rays)
    ds = hiprt.DeviceScene(hip_ctx, sc, bvh)
    got = _closest(torch_cuda, ds, rays, tracer=tracer, blocks=blocks, refill_threshold=refill, work_chunks=chunks,
                   park_leaves=park)
    assert classify(orc, pos, idx, rays, got, want)["unexplained"] == 0
    ds.close()


@pytest.mark.parametrize("tri", [hiprt.TRI_EXACT, hiprt.TRI_WOOP])
def test_closest_hit_columns(torch_cuda, hip_ctx, tri):
    """Trees whose stack fits the LDS words and trees that spill one group of
    entries and more: the counting kernel, with a stack of its own, finds the
    same hits."""
    torch = torch_cuda
    needs = set()
    for n_tris in (12, 55, 60, 65, 75, 90, 105, 120):
        pos, idx = nested_scene()
        pos, idx = np.ascontiguousarray(pos[:3 * n_tris]), np.ascontiguousarray(idx[:n_tris])
        sc = hiprt.HostScene.from_arrays(pos, idx)
        ds = hiprt.DeviceScene(hip_ctx, sc, hiprt.Bvh(sc, max_tris=1), hiprt.BVH2, tri)
        print(f"case: {n_tris} nested triangles, stack need {ds.stack_need}", flush=True)
        needs.add(ds.stack_need)
        rays = nested_rays(20000, n_tris)
        stats = torch.zeros(2, dtype=torch.int64, device="cuda")
        want = _closest(torch, ds, rays, fetch_stats=stats)
        for tracer in SPEC:
            for blocks in (2, 300):
                got = _closest(torch, ds, rays, tracer=tracer, blocks=blocks)
                assert classify(orc, pos, idx, rays, got, want)["unexplained"] == 0, (tracer, blocks)
        ds.close()
    assert min(needs) < 18 < max(needs), needs


def _scenes(hip_ctx, tri):
    """A single leaf, small and larger soups, the nested triangles; the second without rays."""
    out = []
    pos, idx = nested_scene()
    for k, (sc, n) in enumerate(((hiprt.HostScene.random(1, 0.3, 1), 70), (hiprt.HostScene.random(50, 0.2, 2), 0),
                                 (hiprt.HostScene.random(700, 0.08, 3), 1), (hiprt.HostScene.random(4000, 0.03, 4), 9001),
                                 (hiprt.HostScene.from_arrays(pos[:180], idx[:60]), 3000))):
        bvh = hiprt.Bvh(sc, max_tris=1 if k == 4 else 4)
        rays = nested_rays(n, 9) if k == 4 else _rays(n, 20 + k)
        out.append((sc, bvh, rays, hiprt.DeviceScene(hip_ctx, sc, bvh, hiprt.BVH2, tri)))
    return out


@pytest.mark.parametrize("tracer", SPEC)
@pytest.mark.parametrize("blocks", [2, 100])
def test_table(torch_cuda, hip_ctx, tracer, blocks):
    torch = torch_cuda
    scenes = _scenes(hip_ctx, hiprt.TRI_EXACT)
    dev = [torch.from_numpy(s[2]).cuda() for s in scenes]
    hits = [hiprt.new_hits(s[2].shape[1]) for s in scenes]
    occ = [torch.full((s[2].shape[1],), 7, dtype=torch.uint8, device="cuda") for s in scenes]
    hiprt.trace_batch([(s[3], d, h, None) for s, d, h in zip(scenes, dev, hits)], tracer=tracer, blocks=blocks)
    hiprt.trace_batch([(s[3], d, None, o) for s, d, o in zip(scenes, dev, occ)], any=True, tracer=tracer,
                      blocks=blocks)
    torch.cuda.synchronize()
    for k, (sc, bvh, rays, ds) in enumerate(scenes):
        pos, idx, _ = sc.arrays()
        args = (pos, idx, bvh.nodes, bvh.root, bvh.index, rays)
        if rays.shape[1]:
            want = orc.trace_closest(*args)
            got = tuple(hits[k][p].cpu().numpy() for p in ("t", "u", "v")) + (hits[k]["id"].cpu().numpy().view(np.uint32),)
            assert classify(orc, pos, idx, rays, got, want)["unexplained"] == 0, k
            assert np.array_equal(occ[k].cpu().numpy(), orc.trace_any(*args)), k
        ds.close()


@pytest.mark.parametrize("any_hit", [False, True])
def test_table_of_woop_records(torch_cuda, hip_ctx, any_hit):
    """Against the plain kernel on the same records, scene by scene."""
    torch = torch_cuda
    scenes = [s for s in _scenes(hip_ctx, hiprt.TRI_WOOP) if s[2].shape[1]]
    for tracer in SPEC:
        entries = []
        for _, _, rays, ds in scenes:
            n = rays.shape[1]
            entries.append((ds, torch.from_numpy(rays).cuda(), None if any_hit else hiprt.new_hits(n),
                            torch.full((n,), 7, dtype=torch.uint8, device="cuda") if any_hit else None))
        hiprt.trace_batch(entries, any=any_hit, tracer=tracer, blocks=7)
        for (sc, _, rays, ds), (_, dr, h, o) in zip(scenes, entries):
            if any_hit:
                want = torch.empty_like(o)
                hiprt.trace_any(ds, dr, want)
                torch.cuda.synchronize()
                assert torch.equal(o, want)
            else:
                ref = hiprt.new_hits(rays.shape[1])
                hiprt.trace_closest(ds, dr, ref)
                torch.cuda.synchronize()
                pos, idx, _ = sc.arrays()
                planes = [tuple(x[p].cpu().numpy() for p in ("t", "u", "v")) + (x["id"].cpu().numpy().view(np.uint32),)
                          for x in (h, ref)]
                assert classify(orc, pos, idx, rays, *planes)["unexplained"] == 0
    for s in scenes:
        s[3].close()


def test_opacity(torch_cuda, hip_ctx):
    torch = torch_cuda
    base = hiprt.HostScene.random(2000, 0.05, 30)
    pos, idx, _ = base.arrays()
    sc = hiprt.HostScene.from_arrays(pos, idx, np.zeros(len(idx), np.uint32))
    sc.set_texcoords(np.random.default_rng(1).uniform(-1, 2, (len(pos), 2)).astype(np.float32))
    tex = np.ones((8, 8, 4), np.float32)
    tex[::2, :, 3] = 0.1
    sc.set_texture(0, tex)
    bvh = hiprt.Bvh(sc)
    ds = hiprt.DeviceScene(hip_ctx, sc, bvh)
    rays = _rays(20001, 8)
    want, plain = _any(torch, ds, rays, tracer="while-while-alpha"), _any(torch, ds, rays)
    assert not np.array_equal(want, plain)
    for tracer in SPEC:
        assert np.array_equal(_any(torch, ds, rays, tracer=tracer + "-alpha", blocks=9), want)
        assert np.array_equal(_any(torch, ds, rays, tracer=tracer, blocks=9), plain)
    ds.close()
