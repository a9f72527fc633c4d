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
