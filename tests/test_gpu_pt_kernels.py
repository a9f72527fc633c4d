"""The path tracer on the kernels that trace large frames.  A caller's grid
selects them at any frame size (without one, frames of up to 1.3 M paths take
the group trace): persistent kernels that read their queue's length on the
device, ray records gathered through the sorted permutation, a spill column
held by the captured graph (the hall's tree outgrows the LDS words), refill
thresholds, work counters, stack configurations, path regeneration.

The tracer that keeps the reference's order gives the plain schedule's bits;
the postponing ones may take the other triangle of an equal-t tie, so their
images are held to the oracle with the bars of test_gpu_pt_oracle.py."""
import numpy as np
import pytest

import hiprt
from test_gpu_pt_oracle import COUNT_REL, MAX_DIFF_PATHS, PIXEL_REL, SUM_REL, _oracle, hall  # noqa: F401
from test_gpu_spill import nested_scene

pytestmark = pytest.mark.gpu
SPEC = ("persistent-speculative-while-while", "dynamic-while-while")


def _frames(ds, cam, calls, profile=False, **kw):
    pt = hiprt.PathTracer(ds, cam, **kw)
    for f in range(calls):
        pt.render(f)
    if profile:   # the counting pass runs between two renders of the graph
        pt.profile(calls)
        pt.reset()
        for f in range(calls):
            pt.render(f)
    out = pt.image(), pt.ray_counts(), pt.ray_totals()
    pt.close()
    return out


@pytest.mark.parametrize("res,blocks,kw", [
    ((333, 97), 7, {}), ((320, 180), 300, dict(stack_config=4)), ((320, 180), 64, dict(stack_config=3, work_chunks=1)),
    ((61, 33), 3, dict(sort_rays=False)), ((97, 61), 1792, dict(sort_rays=False, work_chunks=1, stack_config=1)),
    ((13, 7), 2, dict(max_depth=1)), ((64, 40), 2, dict(max_depth=0))])
def test_reference_order_equals_the_plain_schedule(torch_cuda, hall, res, blocks, kw):  # noqa: F811
    print(f"case: hall {res}, persistent-while-while, {blocks} blocks, {kw}", flush=True)
    cam = hall["cam"].copy()
    cam[10], cam[11] = res
    depth = dict(max_depth=kw["max_depth"]) if "max_depth" in kw else {}
    want = _frames(hall["ds"], cam, 3, batched=False, seed=5, **depth)
    got = _frames(hall["ds"], cam, 3, profile=True, seed=5, tracer="persistent-while-while", blocks=blocks, **kw)
    assert want[1].tolist() == got[1].tolist()
    assert np.array_equal(want[0].view(np.uint32), got[0].view(np.uint32))


@pytest.mark.parametrize("tracer", SPEC)
@pytest.mark.parametrize("res,samples,blocks,kw", [
    ((320, 180), 1, 200, {}), ((333, 97), 1, 5, dict(sort_rays=False)), ((160, 90), 1, 1792, dict(work_chunks=1)),
    ((80, 45), 64, 300, dict(stack_config=4)), ((160, 90), 16, 100, dict(stack_config=4, refill_coherent=60)),
    ((160, 90), 8, 100, dict(refill_threshold=64, refill_coherent=1, park_leaves=2))])
def test_postponing_tracers_match_the_oracle(torch_cuda, hall, tracer, res, samples, blocks, kw):  # noqa: F811
    print(f"case: hall {res}, {samples} samples, {tracer}, {blocks} blocks, {kw}", flush=True)
    cam = hall["cam"].copy()
    cam[10], cam[11] = res
    calls = 2 if samples == 1 else 1
    got, _, got_levels = _frames(hall["ds"], cam, calls, seed=7, tracer=tracer, samples=samples, blocks=blocks, **kw)
    want, want_levels = _oracle(hall, cam, 7, samples * calls)
    n_paths = res[0] * res[1] * samples * calls
    differ = (got.view(np.uint32) != want.view(np.uint32)).any(-1)
    total = float(want.sum(dtype=np.float64))
    assert want.sum() > 0 and got_levels[0] == n_paths
    assert differ.sum() <= MAX_DIFF_PATHS * n_paths + 1
    assert abs(float(got.sum(dtype=np.float64)) - total) <= SUM_REL * total
    assert (np.abs(got_levels.astype(np.int64) - want_levels.astype(np.int64)) <= COUNT_REL * want_levels + 1).all()


@pytest.mark.parametrize("tracer", ("persistent-while-while",) + SPEC)
@pytest.mark.parametrize("pool,sort", [(1, True), (3, True), (2, False)])
def test_regeneration_matches_the_oracle(torch_cuda, hall, tracer, pool, sort):  # noqa: F811
    print(f"case: hall regeneration, {pool} slots per pixel, sorted {sort}, {tracer}", flush=True)
    cam = hall["cam"].copy()
    cam[10], cam[11] = 97, 61
    samples = 6
    got, _, got_levels = _frames(hall["ds"], cam, 1, seed=7, tracer=tracer, samples=samples, regen_pool=pool,
                                 sort_rays=sort, blocks=50, stack_config=4)
    want, want_levels = _oracle(hall, cam, 7, samples)
    n_paths = 97 * 61 * samples
    far = np.abs(got - want).max(-1) > PIXEL_REL * np.maximum(np.abs(want).max(-1), 1e-30)
    assert far.sum() <= MAX_DIFF_PATHS * n_paths + 1
    assert (np.abs(got_levels.astype(np.int64) - want_levels.astype(np.int64)) <= COUNT_REL * want_levels + 1).all()


@pytest.mark.parametrize("stack", [0, 3, 4])
def test_deep_tree(torch_cuda, hip_ctx, stack):
    """38 stack entries: the graph's column holds several groups of four."""
    pos, idx = nested_scene()
    sc = hiprt.HostScene.from_arrays(pos, idx)
    ds = hiprt.DeviceScene(hip_ctx, sc, hiprt.Bvh(sc, max_tris=1))
    cam = np.array([0.02, 0.02, 0.02, -1, -1, -1, 0, 1, 0, 60, 160, 120], np.float32)
    print(f"case: nested scene path tracer, stack {stack}", flush=True)
    want = _frames(ds, cam, 2, batched=False, seed=5)
    for tracer in ("persistent-while-while",) + SPEC:
        for sort in (True, False):
            got = _frames(ds, cam, 2, seed=5, tracer=tracer, stack_config=stack, sort_rays=sort, blocks=40)
            same = (got[0].view(np.uint32) == want[0].view(np.uint32)).all(-1)
            if tracer == "persistent-while-while":
                assert same.all()
            assert (~same).sum() <= MAX_DIFF_PATHS * 2 * same.size + 1
    ds.close()


@pytest.mark.parametrize("samples,res", [(1, (1487, 883)), (9, (409, 357))])
def test_frames_above_the_group_trace(torch_cuda, hall, samples, res):  # noqa: F811
    """1,313,021 and 1,314,117 paths on the default grid, with the tracer the
    path tracer picks itself, against the plain schedule."""
    print(f"case: hall {res}, {samples} samples in flight, default dispatch", flush=True)
    cam = hall["cam"].copy()
    cam[10], cam[11] = res
    assert res[0] * res[1] * samples > 5 << 18
    got, got_counts, got_levels = _frames(hall["ds"], cam, 1, seed=3, samples=samples)
    want, _, want_levels = _frames(hall["ds"], cam, samples, seed=3, batched=False)
    n_paths = res[0] * res[1] * samples
    differ = (got.view(np.uint32) != want.view(np.uint32)).any(-1)
    assert got.sum() > 0 and differ.sum() <= MAX_DIFF_PATHS * n_paths
    assert (np.abs(got_levels.astype(np.int64) - want_levels.astype(np.int64)) <= COUNT_REL * want_levels + 1).all()
