"""A binary tree whose node array passes 4 GiB, uploaded with leaves that share
slots: the nodes beyond 2^26 are reached by 64-bit addresses in every kernel a
trace can take.  The only path to two of the three triangles leads through the
last node, whose index keeps just its lowest bit when cut to 26 bits."""
import ctypes

import numpy as np
import pytest

import hiprt

pytestmark = pytest.mark.gpu
LAST = (1 << 26) + 1


def _leaf(slot):
    return ~(slot << 5)   # one triangle


def _node(box_l, box_r, ref_l, ref_r):
    n = np.zeros(16, np.float32)
    for at, (lo, hi) in ((0, box_l), (4, box_r)):
        n[at:at + 4] = lo[0], hi[0], lo[1], hi[1]
    n[8:12] = box_l[0][2], box_l[1][2], box_r[0][2], box_r[1][2]
    n[12:14].view(np.int32)[:] = ref_l, ref_r
    return n.view(np.int32)


@pytest.fixture(scope="module")
def large(torch_cuda, hip_ctx):
    base = np.array([[-1, -1, 5], [1, -1, 5], [0, 1, 5]], np.float32)
    pos = np.concatenate([base + np.float32([10 * k, 0, 0]) for k in range(3)]).astype(np.float32)
    sc = hiprt.HostScene.from_arrays(pos, np.arange(9, dtype=np.uint32).reshape(3, 3))
    small = hiprt.DeviceScene(hip_ctx, sc, hiprt.Bvh(sc, esc=False))
    _, recs, ids = small.download()
    small.close()
    slot = [int(np.nonzero(ids == k)[0][0]) for k in range(3)]
    box = [(pos[3 * k:3 * k + 3].min(0), pos[3 * k:3 * k + 3].max(0)) for k in range(3)]
    nodes = np.zeros((LAST + 1, 16), np.int32)   # between the two: empty boxes at the origin
    nodes[:, 12:14] = _leaf(slot[0])
    both = (np.minimum(box[1][0], box[2][0]), np.maximum(box[1][1], box[2][1]))
    nodes[0] = _node(box[0], both, _leaf(slot[0]), LAST)
    nodes[LAST] = _node(box[1], box[2], _leaf(slot[1]), _leaf(slot[2]))
    out = ctypes.c_void_p()
    hiprt.check(hiprt.lib().hiprt_scene_upload(hip_ctx.h, nodes.ctypes.data, LAST + 1, hiprt.BVH2, recs.ctypes.data,
                                               np.ascontiguousarray(ids).ctypes.data, len(ids), hiprt.TRI_EXACT, 0,
                                               ctypes.byref(out)))
    ds = hiprt.DeviceScene(hip_ctx, None, None, handle=out)
    yield ds
    ds.close()


@pytest.mark.parametrize("tracer", hiprt.TRACERS)
@pytest.mark.parametrize("blocks", [0, 3])
def test_every_tracer_reaches_the_last_node(torch_cuda, large, tracer, blocks):
    torch = torch_cuda
    print(f"case: {LAST + 1} nodes, {tracer}, blocks {blocks}", flush=True)
    n = 300
    rays = torch.zeros((8, n), device="cuda")
    rays[0] = 10.0 * (torch.arange(n, device="cuda") % 4)   # the fourth misses
    rays[6], rays[7] = 1.0, 3.4028234663852886e38
    want = torch.arange(n, device="cuda") % 4
    hits, occ = hiprt.new_hits(n), torch.full((n,), 7, dtype=torch.uint8, device="cuda")
    hiprt.trace_closest(large, rays, hits, tracer=tracer, blocks=blocks)
    hiprt.trace_any(large, rays, occ, tracer=tracer, blocks=blocks)
    tables = []
    if tracer != "while-while":
        th, to = hiprt.new_hits(n), torch.full((n,), 7, dtype=torch.uint8, device="cuda")
        hiprt.trace_batch([(large, rays, th, None)], tracer=tracer, blocks=blocks)
        hiprt.trace_batch([(large, rays, None, to)], any=True, tracer=tracer, blocks=blocks)
        tables = [(th, to)]
    torch.cuda.synchronize()
    for h, o in [(hits, occ)] + tables:
        hit = want < 3
        assert torch.equal(h["t"], torch.where(hit, 5.0, 3.4028234663852886e38).to(h["t"].dtype))
        assert torch.equal(h["id"][hit].long(), want[hit])
        assert torch.equal(o.bool(), hit)
