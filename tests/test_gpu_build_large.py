"""GPU: builds on both sides of the length (3072 tiles of 1024 points) above which
a scan gives the partition's tile offsets: every point is in the tree once, each
node's box holds its subtree, and searches find the nearest points."""
import importlib

import numpy as np
import pytest

from common import grid_cloud, in_box, uniform_cloud

pytestmark = pytest.mark.gpu
LAST = 3072 * 1024


@pytest.mark.parametrize("n,kind", [(LAST, "uniform"), (LAST + 1, "uniform"), (LAST + 1025, "grid")])
def test_build_around_the_scanned_length(n, kind):
    import torch

    ikd = importlib.import_module("ikd-tree_amd")
    rng = np.random.default_rng(n)
    p = uniform_cloud(rng, n) if kind == "uniform" else grid_cloud(rng, n)
    t = ikd.KD_TREE(0.5, 0.6, 0.5)
    t.Build(p)
    assert t.size() == n and t.validnum() == n
    assert np.array_equal(np.asarray(t.tree_range(), np.float32).reshape(2, 3), np.stack([p.min(0), p.max(0)]))
    xyz, ids = t.flatten()
    assert np.array_equal(np.sort(ids), np.arange(n, dtype=np.uint32)) and np.array_equal(xyz, p[ids])
    boxes = np.array([[-20, -20, -20, -11, -13, -14], [3, 3, 3, 3.5, 9, 4]], np.float32)
    off, _, got = t.box_search_batch(boxes)
    for i in range(2):
        assert np.array_equal(np.sort(got[off[i]:off[i + 1]]), np.nonzero(in_box(p, boxes[i]))[0])
    q = uniform_cloud(rng, 200, -55, 55)
    _, d2, _, cnt = t.knn(q, 5)
    dp = torch.from_numpy(p).to("cuda:0")
    for i in range(len(q)):
        x, y, z = (dp - torch.from_numpy(q[i]).to("cuda:0")).square_().unbind(1)
        want = torch.topk((x + y) + z, 5, largest=False).values.sort().values.cpu().numpy()
        assert cnt[i] == 5 and np.array_equal(d2[i].view(np.uint32), want.view(np.uint32)), f"query {i}"
