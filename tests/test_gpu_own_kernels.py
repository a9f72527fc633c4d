"""Binary-tree batches on the kernel of the tracer that was asked for, which a
caller's grid selects at sizes the group trace would serve: every stack
configuration, both work counters, a tree that fits the stack and one that
spills, against the oracle."""
import numpy as np
import pytest

import hiprt
import oracle_py as orc
from parity import bit_exact, classify, uniform_sphere_rays
from test_gpu_spill import PERSISTENT, _any, _closest, nested_rays, nested_scene

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=["soup", "nested"])
def scene(request, torch_cuda, hip_ctx):
    deep = request.param == "nested"
    sc = hiprt.HostScene.from_arrays(*nested_scene()) if deep else hiprt.HostScene.generate(1)
    bvh = hiprt.Bvh(sc, max_tris=1 if deep else 4)
    pos, idx, _ = sc.arrays()
    rays = nested_rays(20_000, 11) if deep else np.ascontiguousarray(uniform_sphere_rays(20_001, 12))
    args = (pos, idx, bvh.nodes, bvh.root, bvh.index, rays)
    ds = hiprt.DeviceScene(hip_ctx, sc, bvh)
    yield ds, pos, idx, rays, orc.trace_closest(*args), orc.trace_any(*args)
    ds.close()


@pytest.mark.parametrize("tracer", PERSISTENT)
@pytest.mark.parametrize("chunks,blocks", [(1, 3), (8, 3), (8, 300)])
def test_every_stack_configuration(torch_cuda, scene, tracer, chunks, blocks):
    ds, pos, idx, rays, want, want_any = scene
    for stack in range(5):
        print(f"case: stack need {ds.stack_need}, {tracer}, stack {stack}, {chunks} chunks, {blocks} blocks", flush=True)
        kw = dict(stack_config=stack, work_chunks=chunks, blocks=blocks)
        got = _closest(torch_cuda, ds, rays, tracer, **kw)
        if tracer == "persistent-while-while":
            assert bit_exact(got, want)
        assert classify(orc, pos, idx, rays, got, want)["unexplained"] == 0
        assert np.array_equal(_any(torch_cuda, ds, rays, tracer, **kw), want_any)


@pytest.mark.parametrize("tracer", PERSISTENT)
@pytest.mark.parametrize("chunks", [1, 8])
def test_default_grid_of_large_batches(torch_cuda, hip_ctx, tracer, chunks):
    n = (1 << 20) + 65
    sc = hiprt.HostScene.random(3000, 0.05, 5)
    bvh = hiprt.Bvh(sc)
    pos, idx, _ = sc.arrays()
    ds = hiprt.DeviceScene(hip_ctx, sc, bvh)
    rays = np.ascontiguousarray(uniform_sphere_rays(n, 7))
    print(f"case: {n} rays, {tracer}, {chunks} chunks, default grid", flush=True)
    args = (pos, idx, bvh.nodes, bvh.root, bvh.index, rays)
    got, want = _closest(torch_cuda, ds, rays, tracer, work_chunks=chunks), orc.trace_closest(*args)
    assert classify(orc, pos, idx, rays, got, want)["unexplained"] == 0
    assert np.array_equal(_any(torch_cuda, ds, rays, tracer, work_chunks=chunks), orc.trace_any(*args))
    ds.close()
