"""The box tree behind the device build and the refit at the sizes where its
levels change: one slot, odd counts, around the 1,024 slots of a block and the
1,048,576 that two launches cover.  Node boxes of the build and of a refit
equal the exact bounds of the slots below each child, the nodes are numbered
in pre-order, and the depth the device reports is the tree's."""
import numpy as np
import pytest

import hiprt

pytestmark = pytest.mark.gpu


def _walk(nodes):
    """Per node: the slot range of each child, and the depth, from the references alone."""
    n = len(nodes)
    refs = nodes[:, 12:14].view(np.int32)
    lo, hi, depth = np.zeros((n, 2), np.int64), np.zeros((n, 2), np.int64), np.ones(n, np.int64)
    for i in range(n - 1, -1, -1):
        for c in range(2):
            r = int(refs[i, c])
            if r < 0:
                slot, cnt = (~r) >> 5, ((~r) & 31) + 1
                lo[i, c], hi[i, c] = slot, slot + cnt
            else:
                assert r > i
                lo[i, c], hi[i, c] = lo[r, 0], hi[r, 1]
                depth[i] = max(depth[i], depth[r] + 1)
        # pre-order: the left child follows its parent, the right one the left subtree
        if refs[i, 0] >= 0:
            assert refs[i, 0] == i + 1
    return lo, hi, depth


def _check(ds, pos, idx):
    nodes, _, slots = ds.download()
    nodes = nodes.reshape(-1, 16).view(np.float32)
    lo, hi, depth = _walk(nodes)
    assert (lo[:, 1] == hi[:, 0]).all()
    if len(nodes):
        assert (lo[0, 0], hi[0, 1]) == (0, len(idx)) and depth[0] == ds.depth
    tri = pos[idx[slots]]
    tlo, thi = tri.min(1), tri.max(1)
    # node rows: (l.x lo hi, l.y lo hi | r.x, r.y | l.z lo hi, r.z lo hi)
    cols = ((0, 2, 8), (4, 6, 10))
    pick = np.random.default_rng(1).permutation(len(nodes))[:1500]
    for i in np.union1d(pick, np.arange(min(len(nodes), 200))):
        for c in range(2):
            want_lo, want_hi = tlo[lo[i, c]:hi[i, c]].min(0), thi[lo[i, c]:hi[i, c]].max(0)
            assert np.array_equal(nodes[i, list(cols[c])], want_lo)
            assert np.array_equal(nodes[i, [k + 1 for k in cols[c]]], want_hi)


@pytest.mark.parametrize("n", [1, 2, 3, 5, 6, 63, 64, 65, 1023, 1024, 1025, 2049, 5000, 1048575, 1048577])
def test_build_and_refit(torch_cuda, hip_ctx, n):
    torch = torch_cuda
    print(f"case: {n} triangles", flush=True)
    rng = np.random.default_rng(n)
    pos = (rng.random((n, 1, 3)) + 0.02 * rng.normal(size=(n, 3, 3))).reshape(-1, 3).astype(np.float32)
    idx = np.arange(3 * n, dtype=np.uint32).reshape(-1, 3)
    d_idx = torch.from_numpy(idx.view(np.int32)).cuda()
    for max_leaf in ((4,) if n > 100000 else (1, 4, 32)):
        ds, _ = hiprt.build_device_scene(hip_ctx, torch.from_numpy(pos).cuda(), d_idx, max_leaf=max_leaf)
        _check(ds, pos, idx)
        moved = (pos * np.float32(1.5) + 0.01 * rng.normal(size=pos.shape).astype(np.float32)).astype(np.float32)
        ds.refit(torch.from_numpy(moved).cuda())
        _check(ds, moved, idx)
        ds.close()


def test_build_reports_bad_materials_and_vertices(torch_cuda, hip_ctx):
    torch = torch_cuda
    pos = torch.rand((30, 3), device="cuda")
    idx = torch.arange(30, dtype=torch.int32, device="cuda").view(-1, 3)
    mat = torch.zeros(10, dtype=torch.int32, device="cuda")
    table = np.zeros((2, 8), np.float32)
    mat[7] = 2
    with pytest.raises(hiprt.HiprtError, match="material"):
        hiprt.build_device_scene(hip_ctx, pos, idx, mat, table)
    bad = idx.clone()
    bad[3, 1] = 30
    with pytest.raises(hiprt.HiprtError, match="vertex"):
        hiprt.build_device_scene(hip_ctx, pos, bad)
