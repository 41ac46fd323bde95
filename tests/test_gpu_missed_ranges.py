"""GPU: after Add_Point_Boxes stored ranges can miss restored points, and what a
walk then finds depends on its order.  Nearest_Search walks in the reference's
order there: every entry point, at any number of lanes asked for, gives the
answer of one lane per query."""
import importlib

import numpy as np
import pytest
import torch

from common import brute_knn, knn_equivalent, random_boxes, uniform_cloud

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lanes", [-1, 4, 16])
@pytest.mark.parametrize("seed", range(4))
def test_knn_where_ranges_miss_points(seed, lanes):
    ikd = importlib.import_module("ikd-tree_amd")
    rng = np.random.default_rng(40 + seed)
    base = uniform_cloud(rng, 6000, -8, 8)
    g = ikd.KD_TREE(1.0, 1.0, 0.5)
    g.Build(base)
    g.set_tuning(ikd.IKD_TUNE_LANES_PER_QUERY, lanes)
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    n, k = 600, 5
    q = uniform_cloud(rng, n, -9, 9)
    dq, qt = torch.from_numpy(q).to(dev), torch.zeros(n, dtype=torch.int32, device=dev)

    def room():
        return (torch.zeros((n, k, 3), device=dev), torch.zeros((n, k), device=dev),
                torch.zeros((n, k), dtype=torch.int32, device=dev), torch.zeros(n, dtype=torch.int32, device=dev))

    b = ikd.Batch()
    b.set_tuning(ikd.IKD_TUNE_LANES_PER_QUERY, lanes)
    for x in (g, b):  # one stack form: a recording always takes this one
        x.set_tuning(ikd.IKD_TUNE_KNN_COMPACT, 0)
    rec = room()
    graph = b.knn_graph([g], qt, dq, k, *rec)  # recorded before any range misses a point
    for _ in range(3):
        box = random_boxes(rng, 1, -8, 8, 3, 8)
        g.Delete_Point_Boxes(box)
        add = random_boxes(rng, 2, -8, 8, 3, 10)
        g.Add_Point_Boxes(add)
        _, d2, ids, cnt = g.knn(q, k)
        g.set_tuning(ikd.IKD_TUNE_LANES_PER_QUERY, 1)
        _, one_d2, one_ids, one_cnt = g.knn(q, k)
        g.set_tuning(ikd.IKD_TUNE_LANES_PER_QUERY, lanes)
        assert np.array_equal(d2.view(np.uint32), one_d2.view(np.uint32)), "tree"
        assert np.array_equal(ids, one_ids) and np.array_equal(cnt, one_cnt), "tree"
        out, noalloc = room(), room()
        b.nearest_search_device([g], qt, dq, k, *out)
        b.nearest_search_noalloc([g], qt, dq, k, *noalloc)
        graph.launch()
        b.synchronize()
        for what, res in (("batch", out), ("no-alloc", noalloc), ("recorded", rec)):
            assert np.array_equal(res[1].cpu().numpy().view(np.uint32), one_d2.view(np.uint32)), what
            assert np.array_equal(res[2].cpu().numpy().view(np.uint32), one_ids), what
            assert np.array_equal(res[3].cpu().numpy(), one_cnt), what
    graph.close()
    # a tree built anew has ranges that miss nothing
    live, lid = g.flatten()
    g.Build(live)
    _, d2, ids, cnt = g.knn(q, k)
    assert len(knn_equivalent(d2, ids, cnt, *brute_knn(live, np.arange(len(live), dtype=np.uint32), q, k))) == 0
