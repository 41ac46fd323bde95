"""GPU: launches over many trees and the trees' own calls, queued without waits
in between, keep their order: a launch sees every update called before it and
none called after it, with one batch, two batches, a recorded launch, a tree
whose stream the caller holds, and a tree or batch closed right after a launch."""
import importlib

import numpy as np
import pytest

from common import uniform_cloud

pytestmark = pytest.mark.gpu


def _outs(torch, n, k=5):
    return (torch.zeros((n, k, 3), device="cuda:0"), torch.zeros((n, k), device="cuda:0"),
            torch.zeros((n, k), dtype=torch.int32, device="cuda:0"),
            torch.zeros((n,), dtype=torch.int32, device="cuda:0"))


@pytest.mark.parametrize("shared", [False, True])
def test_launches_and_updates_keep_their_order(shared):
    import torch

    ikd = importlib.import_module("ikd-tree_amd")
    rng = np.random.default_rng(7)
    nt, nq = 5, 30000
    base = [uniform_cloud(rng, 40000) for _ in range(nt)]
    steps = [[uniform_cloud(rng, 3000) for _ in range(nt)] for _ in range(4)]
    q = uniform_cloud(rng, nq)
    qt = rng.integers(0, nt, nq).astype(np.int32)
    dq, dt = torch.from_numpy(q).to("cuda:0"), torch.from_numpy(qt).to("cuda:0")

    def make():
        trees = []
        for p in base:
            t = ikd.KD_TREE(0.5, 0.6, 0.5)
            t.Build(p)
            if shared:
                t.stream()
            trees.append(t)
        return trees

    def update(t, add, i):
        if i % 2:
            t.Add_Points(add, False)
        else:
            t.Delete_Point_Boxes(np.array([[add[0, 0], -50, -50, add[0, 0] + 9, 50, 50]], np.float32))

    want = []
    trees = make()
    for i, s in enumerate(steps):  # everything waited for
        for t, p in zip(trees, s):
            update(t, p, i)
        out = _outs(torch, nq)
        for j, t in enumerate(trees):
            sel = np.nonzero(qt == j)[0]
            x, d, ids, c = t.knn(q[sel], 5)
            for a, b in zip(out, (x, d, ids.view(np.int32), c)):
                a[torch.from_numpy(sel).to("cuda:0")] = torch.from_numpy(np.ascontiguousarray(b)).to("cuda:0")
        want.append(out)
    torch.cuda.synchronize()
    trees = make()
    batches = [ikd.Batch(), ikd.Batch()]
    outs = [[_outs(torch, nq) for _ in range(3)] for _ in steps]
    torch.cuda.synchronize()
    graph = batches[0].knn_graph(trees, dt, dq, 5, *_outs(torch, nq))
    for i, s in enumerate(steps):
        for t, p in zip(trees, s):
            update(t, p, i)
        batches[0].nearest_search_device(trees, dt, dq, 5, *outs[i][0])
        batches[1].nearest_search_noalloc(trees, dt, dq, 5, *outs[i][1])
        batches[0].nearest_search_device(trees, dt, dq, 5, *outs[i][2])
        graph.launch()
    graph.close()
    batches[1].close()
    for t in trees[1:]:
        t.close()  # frees the nodes the launches read, behind them
    trees[0].Build(base[0][:10])
    batches[0].synchronize()
    torch.cuda.synchronize()
    for i in range(len(steps)):
        for o in outs[i]:
            for a, b in zip(o, want[i]):
                assert torch.equal(a, b), f"step {i}"
