"""GPU: range searches around the number of queries above which one lane walks
each query instead of a wavefront (32768).  Both ways give the same points in the
same order, also for queries with more items than the first walk keeps, queries
that find nothing, and queries of a launch over several trees."""
import importlib

import numpy as np
import pytest

from common import brute_radius, grid_cloud, in_box, random_boxes, uniform_cloud

pytestmark = pytest.mark.gpu
LAST = 32768  # queries of the largest launch that wavefronts walk


def _tree(ikd, rng, n, kind="uniform"):
    t = ikd.KD_TREE(0.5, 0.6, 0.5)
    p = grid_cloud(rng, n) if kind == "grid" else uniform_cloud(rng, n)
    t.Build(p)
    if n > 60:
        t.Delete_Point_Boxes(random_boxes(rng, 3))
        t.Delete_Points(p[::9])
    return t


@pytest.mark.parametrize("n,kind", [(1, "uniform"), (33, "grid"), (129, "uniform"), (20000, "grid"),
                                    (20000, "uniform")])
def test_lanes_and_wavefronts_find_the_same(n, kind):
    ikd = importlib.import_module("ikd-tree_amd")
    rng = np.random.default_rng(n)
    t = _tree(ikd, rng, n, kind)
    nq = LAST + 65
    boxes = random_boxes(rng, nq, smin=0.2, smax=2.0)
    c = uniform_cloud(rng, nq)
    r = (0.1 + rng.random(nq)).astype(np.float32)
    for i in (0, 7, LAST, nq - 1):  # many items
        boxes[i], r[i] = [-1e9] * 3 + [1e9] * 3, 200.0
    boxes[5], r[5] = [5, 5, 5, 4, 4, 4], 0.0
    for search, args in ((t.box_search_batch, (boxes,)), (t.radius_search_batch, (c, r))):
        parts = [search(*(a[i:i + 8000] for a in args)) for i in range(0, nq, 8000)]
        counts = np.concatenate([np.diff(p[0]) for p in parts])
        ids = np.concatenate([p[2] for p in parts])
        xyz = np.concatenate([p[1] for p in parts])
        for m in (LAST, LAST + 1, nq):
            off, gx, gi = search(*(a[:m] for a in args))
            assert np.array_equal(np.diff(off), counts[:m])
            assert np.array_equal(gi, ids[:off[-1]]) and np.array_equal(gx, xyz[:off[-1]])
    live, lid = t.flatten()
    off, _, gi = t.box_search_batch(boxes)
    for i in list(range(0, nq, 4001)) + [5, LAST]:
        assert np.array_equal(gi[off[i]:off[i + 1]], lid[in_box(live, boxes[i])]), f"box {i}"


def test_many_balls_over_several_trees():
    import torch

    ikd = importlib.import_module("ikd-tree_amd")
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    rng = np.random.default_rng(3)
    trees = [_tree(ikd, rng, n) for n in (9000, 40, 3000)]
    nq = LAST + 300
    c = uniform_cloud(rng, nq)
    r = (0.1 + 2 * rng.random(nq)).astype(np.float32)
    qt = rng.integers(-1, 4, nq).astype(np.int32)  # -1 and 3 name no tree
    args = [torch.from_numpy(a).to(dev) for a in (qt, c, r)]
    off = torch.zeros(nq + 1, dtype=torch.int64, device=dev)
    b = ikd.Batch()
    total = b.radius_search_device(trees, *args, off)
    xyz = torch.zeros((total, 3), device=dev)
    ids = torch.zeros(total, dtype=torch.int32, device=dev)
    if dev.type == "cuda":
        torch.cuda.synchronize()  # the batch has a stream of its own
    assert b.radius_search_device(trees, *args, off, xyz, ids) == total
    b.synchronize()
    off, ids = off.cpu().numpy(), ids.cpu().numpy()
    assert off[-1] == total and np.all(np.diff(off)[(qt < 0) | (qt > 2)] == 0)
    flat = [t.flatten() for t in trees]
    for i in range(0, nq, 257):
        if 0 <= qt[i] < 3:
            live, lid = flat[qt[i]]
            inside, band = brute_radius(live, c[i], float(r[i]))
            differ = np.setxor1d(ids[off[i]:off[i + 1]], lid[inside])
            assert np.isin(differ, lid[band]).all(), f"ball {i}"
