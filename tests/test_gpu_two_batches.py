"""GPU: launches of two batches over lists of trees that overlap, queued without
waits in between.  The no-alloc form keeps its tree table, thresholds and query
counters in one array per GPU, so each launch has to run behind the one before;
a launch may also read what another batch's launch wrote."""
import importlib

import numpy as np
import pytest

from common import uniform_cloud

pytestmark = pytest.mark.gpu


def _outs(torch, n, k, dev):
    return (torch.zeros((n, k, 3), device=dev), torch.zeros((n, k), device=dev),
            torch.zeros((n, k), dtype=torch.int32, device=dev), torch.zeros((n,), dtype=torch.int32, device=dev))


def test_noalloc_launches_of_two_batches():
    import torch

    ikd = importlib.import_module("ikd-tree_amd")
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    rng = np.random.default_rng(12)
    trees = []
    for n in (50000, 20000, 80000):
        t = ikd.KD_TREE(0.5, 0.6, 0.5)
        t.Build(uniform_cloud(rng, n))
        trees.append(t)
    lists = [trees[:2], trees[1:], [trees[1]], trees[::-1]]
    k, calls = 5, []
    for i, tl in enumerate(lists * 3):
        nq = (60000, 500, 20000)[i % 3]
        q = torch.from_numpy(uniform_cloud(rng, nq)).to(dev)
        qt = torch.from_numpy(rng.integers(0, len(tl), nq).astype(np.int32)).to(dev)
        md = torch.from_numpy(rng.choice(np.array([1.0, 4.0, np.inf]), nq)).to(dev)
        calls.append((tl, qt, q, md, _outs(torch, nq, k, dev), _outs(torch, nq, k, dev)))
    if dev.type == "cuda":
        torch.cuda.synchronize()  # batches have streams of their own
    one = ikd.Batch()
    for tl, qt, q, md, want, _ in calls:  # everything waited for
        one.nearest_search_device(tl, qt, q, k, *want, max_dist=md)
        one.synchronize()
    batches = [ikd.Batch(), ikd.Batch()]
    for i, (tl, qt, q, md, _, got) in enumerate(calls):
        batches[i % 2].nearest_search_noalloc(tl, qt, q, k, *got, max_dist=md)
    for b in batches:
        b.synchronize()
    for i, (_, _, _, _, want, got) in enumerate(calls):
        assert all(torch.equal(a, b) for a, b in zip(want, got)), f"call {i}"


def test_a_launch_reads_what_another_batch_wrote():
    import torch

    ikd = importlib.import_module("ikd-tree_amd")
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    rng = np.random.default_rng(13)
    t = ikd.KD_TREE(0.5, 0.6, 0.5)
    t.Build(uniform_cloud(rng, 100000))
    n = 200000
    q = torch.from_numpy(uniform_cloud(rng, n)).to(dev)
    qt = torch.zeros(n, dtype=torch.int32, device=dev)
    a, b = ikd.Batch(), ikd.Batch()
    first, second = _outs(torch, n, 1, dev), _outs(torch, n, 1, dev)
    if dev.type == "cuda":
        torch.cuda.synchronize()
    a.nearest_search_device([t], qt, q, 1, *first)
    b.nearest_search_device([t], qt, first[0].reshape(n, 3), 1, *second)  # the nearest point's nearest point
    b.synchronize()
    assert float(second[1].max()) == 0.0 and torch.equal(first[0], second[0])
