"""GPU: after Add_Point_Boxes stored ranges can miss restored points, and what a
walk then finds depends on its pruning decisions.  With the default tuning every
entry point makes the reference's: the same answer from all of them, also beside
trees whose ranges miss nothing, and, where both trees have grown alike (without
rebuilds, whose splits may differ), for every query the squared distances of the
oracle's walk or else those of a search through all live points."""
import importlib

import numpy as np
import pytest

from common import brute_knn, random_boxes, uniform_cloud

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", range(12))
def test_default_tuning_against_the_oracle(seed):
    import torch

    from oracle import OracleTree

    ikd = importlib.import_module("ikd-tree_amd")
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    rng = np.random.default_rng(400 + seed)
    prm = (1.0, 1.0, 0.5) if seed % 2 == 0 else (0.5, 0.6, 0.5)  # without and with rebuilds
    base = uniform_cloud(rng, 4000, -8, 8)
    g, other, o = ikd.KD_TREE(*prm), ikd.KD_TREE(*prm), OracleTree(*prm)
    for t in (g, o):
        t.Build(base)
    other.Build(uniform_cloud(rng, 3000, -8, 8))
    b = ikd.Batch()
    nq, kmax, next_id = 500, 10, 4000

    def room():
        return (torch.zeros((nq, kmax, 3), device=dev), torch.zeros((nq, kmax), device=dev),
                torch.zeros((nq, kmax), dtype=torch.int32, device=dev),
                torch.zeros(nq, dtype=torch.int32, device=dev))

    dq = torch.zeros((nq, 3), device=dev)
    qt = torch.ones(nq, dtype=torch.int32, device=dev)
    rec = room()
    if dev.type == "cuda":
        torch.cuda.synchronize()  # batches have streams of their own
    graph = b.knn_graph([other, g], qt, dq, kmax, *rec)  # recorded before any range misses a point
    for r in range(3):
        if seed % 3 == 0:
            add = uniform_cloud(rng, 800, -9, 9)
            ids = np.arange(next_id, next_id + 800, dtype=np.uint32)
            next_id += 800
            assert g.Add_Points(add, True, ids) == o.Add_Points(add, True, ids)
        box = random_boxes(rng, 1, -8, 8, 3, 8)
        assert g.Delete_Point_Boxes(box) == o.Delete_Point_Boxes(box)
        back = random_boxes(rng, 2, -8, 8, 3, 10)
        g.Add_Point_Boxes(back)
        o.Add_Point_Boxes(back)
        q = uniform_cloud(rng, nq, -9, 9)
        live, lid = g.flatten()
        for k in (1, 5, kmax):
            _, d2, ids, cnt = g.knn(q, k)
            want = np.sort(o.knn(q, k)[1], axis=1)
            exact = brute_knn(live, lid, q, k)[0]
            bits = lambda a: np.ascontiguousarray(a).view(np.uint32)
            oracles = np.all(bits(d2) == bits(want), axis=1)
            if seed % 2:
                continue
            assert np.all(oracles | np.all(bits(d2) == bits(exact), axis=1)), f"round {r} k {k}"
            assert np.count_nonzero(~oracles) <= 1, f"round {r} k {k}"
        dq.copy_(torch.from_numpy(q))
        out, noalloc = room(), room()
        if dev.type == "cuda":
            torch.cuda.synchronize()
        b.nearest_search_device([other, g], qt, dq, kmax, *out)
        b.nearest_search_noalloc([other, g], qt, dq, kmax, *noalloc)
        graph.launch()
        b.synchronize()
        for what, res in (("batch", out), ("no-alloc", noalloc), ("recorded", rec)):
            assert np.array_equal(bits(res[1].cpu().numpy()), bits(d2)), what
            assert np.array_equal(res[2].cpu().numpy().view(np.uint32), ids), what
            assert np.array_equal(res[3].cpu().numpy(), cnt), what
    graph.close()


@pytest.mark.parametrize("nq", [700, 20000])
def test_one_such_tree_among_others(nq):
    """A call over several trees of which none, one or all are such trees."""
    import torch

    ikd = importlib.import_module("ikd-tree_amd")
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    rng = np.random.default_rng(nq)
    trees = []
    for n in (3000, 5000, 400):
        t = ikd.KD_TREE(1.0, 1.0, 0.5)
        t.Build(uniform_cloud(rng, n, -8, 8))
        trees.append(t)
    k = 5
    q = uniform_cloud(rng, nq, -9, 9)
    qt = rng.integers(-1, 4, nq).astype(np.int32)  # -1 and 3 name no tree
    dq, dt = torch.from_numpy(q).to(dev), torch.from_numpy(qt).to(dev)
    outs = [(torch.zeros((nq, k, 3), device=dev), torch.zeros((nq, k), device=dev),
             torch.zeros((nq, k), dtype=torch.int32, device=dev), torch.zeros(nq, dtype=torch.int32, device=dev))
            for _ in range(3)]
    if dev.type == "cuda":
        torch.cuda.synchronize()
    b = ikd.Batch()
    graph = b.knn_graph(trees, dt, dq, k, *outs[2])
    for lists in ((), (1,), (0, 1, 2)):  # the trees whose ranges miss points
        for i in lists:
            trees[i].Delete_Point_Boxes(random_boxes(rng, 1, -8, 8, 3, 8))
            trees[i].Add_Point_Boxes(random_boxes(rng, 2, -8, 8, 3, 10))
        for o in outs:
            for x in o:
                x.fill_(-7)
        if dev.type == "cuda":
            torch.cuda.synchronize()
        b.nearest_search_device(trees, dt, dq, k, *outs[0])
        b.nearest_search_noalloc(trees, dt, dq, k, *outs[1])
        graph.launch()
        b.synchronize()
        for what, o in zip(("batch", "no-alloc", "recorded"), outs):
            d2, ids, cnt = (x.cpu().numpy() for x in o[1:])
            assert np.all(cnt[(qt < 0) | (qt > 2)] == 0), what
            for i, t in enumerate(trees):
                at = np.nonzero(qt == i)[0]
                _, wd2, wids, wcnt = t.knn(q[at], k)
                assert np.array_equal(cnt[at], wcnt), f"{what} {lists}"
                assert np.array_equal(d2[at].view(np.uint32), wd2.view(np.uint32)), f"{what} {lists}"
                assert np.array_equal(ids[at].view(np.uint32), wids), f"{what} {lists}"
    graph.close()
