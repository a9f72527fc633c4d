"""Scratch of device builds: one per context however many streams build, and
builds from several threads at once give the trees that builds one after the
other give."""
import threading

import numpy as np
import pytest

import hiprt

pytestmark = pytest.mark.gpu


def _tris(torch, n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    pos = torch.rand((n, 1, 3), device="cuda", generator=g) + 0.02 * torch.randn((n, 3, 3), device="cuda", generator=g)
    return pos.reshape(-1, 3).contiguous(), torch.arange(3 * n, dtype=torch.int32, device="cuda").view(-1, 3)


def test_streams_share_the_kept_scratch(torch_cuda, hip_ctx):
    torch = torch_cuda
    n = 400_000   # about 70 MB of scratch
    pos, idx = _tris(torch, n, 1)
    streams = [torch.cuda.Stream() for _ in range(6)]
    free = []
    for s in [streams[0]] + streams:
        s.wait_stream(torch.cuda.current_stream())
        ds, _ = hiprt.build_device_scene(hip_ctx, pos, idx, stream=s.cuda_stream)
        ds.close()
        torch.cuda.synchronize()
        free.append(torch.cuda.mem_get_info()[0])
    print("case: free bytes after each build", free, flush=True)
    assert free[0] - free[-1] < 64 << 20


def test_threads_build_at_once(torch_cuda, hip_ctx):
    torch = torch_cuda
    sizes = (1, 3000, 20_001, 90_000, 150_000)
    made = [_tris(torch, n, n) for n in sizes]
    want = []
    for pos, idx in made:
        ds, _ = hiprt.build_device_scene(hip_ctx, pos, idx)
        want.append(ds.download())
        ds.close()
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in sizes]
    errors = []

    def build(k):
        try:
            for _ in range(4):
                ds, _ = hiprt.build_device_scene(hip_ctx, *made[k], stream=streams[k].cuda_stream)
                got = ds.download()
                ds.close()
                for a, b in zip(got, want[k]):
                    assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), sizes[k]
        except BaseException as e:   # noqa: BLE001  (reported by the test's thread)
            errors.append(e)

    print("case: five threads build at once", flush=True)
    threads = [threading.Thread(target=build, args=(k,)) for k in range(len(sizes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
