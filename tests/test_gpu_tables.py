"""Descriptor tables of binary trees on the persistent kernels, which a caller's
grid selects at any size, against the oracle: the tracer that keeps the
reference's order, over shallow trees (no vote in its node loop) and with the
38-entry nested tree (vote, spill column), and the postponing tracers with that
tree, which is too deep for the kernel that holds its whole stack in LDS."""
import numpy as np
import pytest

import hiprt
import oracle_py as orc
from parity import bit_exact, classify, uniform_sphere_rays
from test_gpu_spill import nested_rays, nested_scene

pytestmark = pytest.mark.gpu
PERSISTENT = [t for t in hiprt.TRACERS if t != "while-while"]


def _scenes(hip_ctx, deep):
    """One leaf, none without rays, small soups; the nested triangles when `deep`."""
    made = [(hiprt.HostScene.random(1, 0.3, 1), 4, 70), (hiprt.HostScene.random(50, 0.2, 2), 4, 0),
            (hiprt.HostScene.random(700, 0.08, 3), 4, 1),
            (hiprt.HostScene.random(4000 if deep else 1000, 0.03, 4), 4, 9001)]
    if deep:
        made.append((hiprt.HostScene.from_arrays(*nested_scene()), 1, 5000))
    out = []
    for k, (sc, max_tris, n) in enumerate(made):
        bvh = hiprt.Bvh(sc, max_tris=max_tris)
        rays = nested_rays(n, 9) if max_tris == 1 else np.ascontiguousarray(uniform_sphere_rays(n, 20 + k))
        ds = hiprt.DeviceScene(hip_ctx, sc, bvh)
        pos, idx, _ = sc.arrays()
        args = (pos, idx, bvh.nodes, bvh.root, bvh.index, rays)
        want = (orc.trace_closest(*args), orc.trace_any(*args)) if n else None
        out.append((ds, rays, pos, idx, want))
    return out


@pytest.mark.parametrize("deep", [False, True])
@pytest.mark.parametrize("tracer", PERSISTENT)
def test_tables_match_the_oracle(torch_cuda, hip_ctx, tracer, deep):
    torch = torch_cuda
    scenes = _scenes(hip_ctx, deep)
    assert max(s[0].stack_need for s in scenes) > 32 if deep else max(s[0].stack_need for s in scenes) <= 12
    dev = [torch.from_numpy(s[1]).cuda() for s in scenes]
    for stack in (0, 1, 3, 4):
        for chunks, blocks in ((1, 3), (8, 3), (8, 100)):
            print(f"case: table, {tracer}, deep {deep}, stack {stack}, {chunks} chunks, {blocks} blocks", flush=True)
            hits = [hiprt.new_hits(s[1].shape[1]) for s in scenes]
            occ = [torch.full((s[1].shape[1],), 7, dtype=torch.uint8, device="cuda") for s in scenes]
            for h in hits:
                for x in h.values():
                    x.fill_(-5)
            kw = dict(tracer=tracer, blocks=blocks, stack_config=stack, work_chunks=chunks)
            hiprt.trace_batch([(s[0], d, h, None) for s, d, h in zip(scenes, dev, hits)], **kw)
            hiprt.trace_batch([(s[0], d, None, o) for s, d, o in zip(scenes, dev, occ)], any=True, **kw)
            torch.cuda.synchronize()
            for (ds, rays, pos, idx, want), h, o in zip(scenes, hits, occ):
                if want is None:
                    continue
                got = tuple(h[p].cpu().numpy() for p in ("t", "u", "v")) + (h["id"].cpu().numpy().view(np.uint32),)
                if tracer == "persistent-while-while":
                    assert bit_exact(got, want[0])
                assert classify(orc, pos, idx, rays, got, want[0])["unexplained"] == 0
                assert np.array_equal(o.cpu().numpy(), want[1])
    for s in scenes:
        s[0].close()


def test_large_table_without_a_grid(torch_cuda, hip_ctx):
    """Above the group trace's sizes the default grid runs the same kernels."""
    torch = torch_cuda
    sc = hiprt.HostScene.random(700, 0.08, 3)
    bvh = hiprt.Bvh(sc)
    pos, idx, _ = sc.arrays()
    ds = hiprt.DeviceScene(hip_ctx, sc, bvh)
    sizes = (700_001, 400_000)
    rays = [np.ascontiguousarray(uniform_sphere_rays(n, 40 + k)) for k, n in enumerate(sizes)]
    dev = [torch.from_numpy(r).cuda() for r in rays]
    hits = [hiprt.new_hits(n) for n in sizes]
    occ = [torch.full((n,), 7, dtype=torch.uint8, device="cuda") for n in sizes]
    print(f"case: table of {sum(sizes)} rays, persistent-while-while", flush=True)
    hiprt.trace_batch([(ds, d, h, None) for d, h in zip(dev, hits)], tracer="persistent-while-while")
    hiprt.trace_batch([(ds, d, None, o) for d, o in zip(dev, occ)], any=True, tracer="persistent-while-while")
    torch.cuda.synchronize()
    for r, h, o in zip(rays, hits, occ):
        args = (pos, idx, bvh.nodes, bvh.root, bvh.index, r)
        got = tuple(h[p].cpu().numpy() for p in ("t", "u", "v")) + (h["id"].cpu().numpy().view(np.uint32),)
        assert bit_exact(got, orc.trace_closest(*args))
        assert np.array_equal(o.cpu().numpy(), orc.trace_any(*args))
    ds.close()
