"""Calls bounded by scratch memory, at batch sizes that other kernels serve."""
import numpy as np
import pytest

import hiprt
from test_gpu_spill import nested_rays, nested_scene

pytestmark = pytest.mark.gpu
SPEC = ("persistent-speculative-while-while", "dynamic-while-while")


def _nested(hip_ctx, n_tris):
    pos, idx = nested_scene()
    sc = hiprt.HostScene.from_arrays(np.ascontiguousarray(pos[:3 * n_tris]), np.ascontiguousarray(idx[:n_tris]))
    return hiprt.DeviceScene(hip_ctx, sc, hiprt.Bvh(sc, max_tris=1))


@pytest.mark.parametrize("tracer", ("persistent-while-while",) + SPEC)
def test_allocation_free_refusal_at_every_batch_size(torch_cuda, hip_ctx, tracer):
    """The deep tree with stack configuration 4 needs at least ten spill
    entries per lane: 10 x 2048 blocks x 1 KiB = 20 MiB, more than the scratch
    holds.  One ray is refused as a large batch is; fewer blocks and the plain
    tracer, which has no column, are served."""
    torch = torch_cuda
    ds = _nested(hip_ctx, 120)
    assert ds.stack_need - 20 >= 10
    rays = torch.from_numpy(nested_rays(300, 1)).cuda()
    hits, want = hiprt.new_hits(300), hiprt.new_hits(300)
    for n in (1, 300):
        with pytest.raises(hiprt.HiprtError, match="spill column"):
            hiprt.trace_closest_noalloc(ds, rays[:, :n].contiguous(), hits, tracer=tracer, stack_config=4)
    hiprt.trace_closest(ds, rays, want)
    for kw in (dict(tracer=tracer, stack_config=4, blocks=8), dict(tracer="while-while", stack_config=4)):
        hiprt.trace_closest_noalloc(ds, rays, hits, **kw)
        torch.cuda.synchronize()
        assert torch.equal(hits["t"], want["t"])
    ds.close()


@pytest.mark.parametrize("tracer", SPEC)
def test_captured_launch_keeps_no_column(torch_cuda, hip_ctx, tracer):
    """A tree of 19 to 32 stack entries, captured on a stream that has only
    traced another scene: no allocation and no wait under capture, and replays
    on new rays give the eager results before and after a deeper tree has made
    the stream's column grow."""
    torch = torch_cuda
    ds, deep = _nested(hip_ctx, 60), _nested(hip_ctx, 120)
    assert 18 < ds.stack_need <= 32 < deep.stack_need
    other = hiprt.HostScene.random(50, 0.2, 2)
    warm = hiprt.DeviceScene(hip_ctx, other, hiprt.Bvh(other))
    n = 20001
    kw = dict(tracer=tracer, blocks=64)   # this tracer's own kernel at any size
    rays = torch.from_numpy(nested_rays(n, 1)).cuda()
    hits, scratch = hiprt.new_hits(n), hiprt.new_hits(n)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    hiprt.trace_closest(warm, rays, hits, stream=s.cuda_stream, **kw)
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        hiprt.trace_closest(ds, rays, hits, stream=s.cuda_stream, **kw)
    for k in range(4):
        rays.copy_(torch.from_numpy(nested_rays(n, 10 + k)))
        for x in hits.values():
            x.fill_(-5)
        if k == 2:   # a larger column, in the place of any before
            hiprt.trace_closest(deep, rays, scratch, stream=s.cuda_stream, tracer=tracer, blocks=2048)
            assert torch.ones(1 << 20, device="cuda").sum().item() == 1 << 20
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        want = hiprt.new_hits(n)
        hiprt.trace_closest(ds, rays, want)
        torch.cuda.synchronize()
        assert torch.equal(hits["t"], want["t"]), k
        assert float((want["t"] < 3e38).float().mean()) > 0.2
    for x in (ds, deep, warm):
        x.close()
