"""Small frames trace their bounce queues in the order the shading step
appends them: image and ray counts equal the form that never sorts, on both
sides of the limit, with samples in flight, with path regeneration, and after
a counting pass, which sorts."""
import numpy as np
import pytest

import hiprt

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene(hip_ctx):
    sc = hiprt.HostScene.generate(3)
    ds = hiprt.DeviceScene(hip_ctx, sc, hiprt.Bvh(sc))
    yield ds, sc.cam
    ds.close()


@pytest.mark.parametrize("res,kw", [((61, 47), {}), ((1280, 716), {}), ((1280, 717), {}), ((320, 179), {"samples": 16}),
                                    ((97, 61), {"samples": 6, "regen_pool": 2}), ((33, 9), {"max_depth": 1})])
def test_equals_the_unsorted_form(torch_cuda, scene, res, kw):
    print(f"case: {res}, {kw}", flush=True)
    ds, cam = scene
    cam = cam.copy()
    cam[10], cam[11] = res
    out = []
    for sort in (True, False):
        pt = hiprt.PathTracer(ds, cam, seed=5, tracer="persistent-while-while", sort_rays=sort, **kw)
        pt.render(0)
        if sort and "regen_pool" not in kw:
            pt.profile(1)
            pt.reset()
            pt.render(0)
        pt.render(1)
        pt.render(2)
        out.append((pt.image(), pt.ray_counts()))
        pt.close()
    assert out[0][1].tolist() == out[1][1].tolist() and out[0][1][1] > 0
    assert out[0][0].sum() > 0
    assert np.array_equal(out[0][0].view(np.uint32), out[1][0].view(np.uint32))
