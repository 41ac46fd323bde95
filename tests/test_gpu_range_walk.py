"""GPU: the wavefront-per-query range walk where it can go wrong: trees around
the item size (32 nodes), one query and many (both stack sizes), frontiers far
wider than 64 nodes, a chain-like tree (one point a call), and a query with more
items than the first walk keeps.  Box results are the half-open filter of
flatten()'s pre-order; ball results the same with the sqrt rounding band."""
import importlib

import numpy as np
import pytest

from common import brute_radius, grid_cloud, in_box, random_boxes, uniform_cloud

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nq,kind", [(1, 1, "uniform"), (31, 3, "grid"), (32, 3, "grid"), (33, 3, "uniform"),
                                       (65, 5, "uniform"), (5000, 2049, "grid"), (60000, 40, "uniform"),
                                       (60000, 4200, "uniform"), (300, 20, "chain")])
def test_range_walk(n, nq, kind):
    ikd = importlib.import_module("ikd-tree_amd")
    rng = np.random.default_rng(n + nq)
    t = ikd.KD_TREE(0.5, 0.6, 0.5)
    if kind == "chain":
        p = np.zeros((n, 3), np.float32)
        p[:, 0] = np.arange(n)
        t.set_tuning(ikd.IKD_TUNE_DEFER_REBUILD, 1)  # no rebalancing: the tree stays as it grew
        t.Build(p[:1])
        for i in range(1, min(n, 50)):
            t.Add_Points(p[i:i + 1], False)
        if n > 50:
            t.Add_Points(p[50:], False)
    else:
        p = grid_cloud(rng, n) if kind == "grid" else uniform_cloud(rng, n)
        t.Build(p)
        if n > 60:
            t.Delete_Point_Boxes(random_boxes(rng, 3))
            t.Delete_Points(p[::9])
    xyz, ids = t.flatten()
    boxes = random_boxes(rng, nq, smin=0.5, smax=4.0)
    boxes[0] = [-1e9] * 3 + [1e9] * 3
    if nq > 2:
        boxes[1] = [5, 5, 5, 4, 4, 4]
        boxes[2] = [-30, -30, -30, 30, 30, 30]
    off, bx, bi = t.box_search_batch(boxes)
    check = range(nq) if nq < 50 else list(range(3)) + list(range(3, nq, nq // 40)) + [nq - 1]
    for i in check:
        want = in_box(xyz, boxes[i])
        assert np.array_equal(bi[off[i]:off[i + 1]], ids[want]), f"box {i}"
        assert np.array_equal(bx[off[i]:off[i + 1]], xyz[want])
    c = uniform_cloud(rng, nq)
    r = (0.5 + 3 * rng.random(nq)).astype(np.float32)
    r[0] = 200.0
    off, bx, bi = t.radius_search_batch(c, r)
    place = np.full(int(ids.max()) + 1, -1, np.int64)
    place[ids] = np.arange(len(ids))
    for i in check:
        got = place[bi[off[i]:off[i + 1]]]
        assert np.all(np.diff(got) > 0), f"ball {i}: pre-order"
        inside, band = brute_radius(xyz, c[i], float(r[i]))
        differ = np.setxor1d(got, np.nonzero(inside)[0])
        assert np.isin(differ, np.nonzero(band)[0]).all(), f"ball {i}"
