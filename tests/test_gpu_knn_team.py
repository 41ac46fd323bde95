"""GPU: the shared list of a team of lanes where it can go wrong: k around the
list's slots per lane, fewer points than k, per-query k in one launch, exact
distance ties across lanes, batch sizes around the switches between team sizes.
Every shape returns the one-lane walk's bits."""
import importlib

import numpy as np
import pytest

from common import grid_cloud, uniform_cloud

pytestmark = pytest.mark.gpu


def _same(a, b, tag):
    for x, y in zip(a, b):
        assert np.array_equal(x.view(np.uint32) if x.dtype == np.float32 else x,
                              y.view(np.uint32) if y.dtype == np.float32 else y), tag


@pytest.mark.parametrize("k", [1, 2, 3, 5, 8, 15, 16, 17, 33, 64])
@pytest.mark.parametrize("n", [3, 40, 30000])
def test_team_list(k, n):
    ikd = importlib.import_module("ikd-tree_amd")
    rng = np.random.default_rng(n + k)
    p = np.concatenate([grid_cloud(rng, n // 2, extent=12), uniform_cloud(rng, n - n // 2, -3, 3)])
    t = ikd.KD_TREE(0.5, 0.6, 0.5)
    t.Build(p)
    q = np.concatenate([grid_cloud(rng, 150, extent=12), p[rng.integers(0, n, 50)], uniform_cloud(rng, 57, -4, 4)])
    for md in (float("inf"), 1.0):
        t.set_tuning(ikd.IKD_TUNE_LANES_PER_QUERY, 1)
        ref = t.knn(q, k, md)
        for lanes in (2, 4, 8, 16):
            t.set_tuning(ikd.IKD_TUNE_LANES_PER_QUERY, lanes)
            _same(ref, t.knn(q, k, md), f"lanes {lanes}, max_dist {md}")


@pytest.mark.parametrize("nq", [1, (1 << 14), (1 << 14) + 1, (1 << 15) + 1, (1 << 17) - 1, 1 << 17])
def test_team_sizes_by_batch(nq):
    ikd = importlib.import_module("ikd-tree_amd")
    rng = np.random.default_rng(nq)
    t = ikd.KD_TREE(0.5, 0.6, 0.5)
    t.Build(uniform_cloud(rng, 20000))
    q = uniform_cloud(rng, nq)
    got = t.knn(q, 5, 4.0)
    t.set_tuning(ikd.IKD_TUNE_LANES_PER_QUERY, 1)
    _same(t.knn(q, 5, 4.0), got, "chosen lanes")


@pytest.mark.parametrize("lanes", [4, 16])
def test_team_per_query_k(lanes):
    import torch

    ikd = importlib.import_module("ikd-tree_amd")
    rng = np.random.default_rng(lanes)
    trees = []
    for n in (2, 500, 9000):
        t = ikd.KD_TREE(0.5, 0.6, 0.5)
        t.Build(grid_cloud(rng, n, extent=10))
        trees.append(t)
    nq, kmax = 333, 20
    dev = "cuda:0"
    qt = torch.from_numpy(rng.integers(-1, 4, nq).astype(np.int32)).to(dev)  # also trees that do not exist
    q = torch.from_numpy(grid_cloud(rng, nq, extent=10)).to(dev)
    ks = torch.from_numpy(rng.integers(0, kmax + 1, nq).astype(np.int32)).to(dev)
    md = torch.from_numpy(rng.choice([0.3, 2.0, np.inf], nq)).to(dev)
    b, got = ikd.Batch(), []
    torch.cuda.synchronize()
    for ln in (1, lanes):
        b.set_tuning(ikd.IKD_TUNE_LANES_PER_QUERY, ln)
        out = (torch.full((nq, kmax, 3), 7.0, device=dev), torch.full((nq, kmax), 7.0, device=dev),
               torch.full((nq, kmax), 7, dtype=torch.int32, device=dev),
               torch.full((nq,), 7, dtype=torch.int32, device=dev))
        torch.cuda.synchronize()
        b.nearest_search_device(trees, qt, q, kmax, *out, k=ks, max_dist=md)
        b.synchronize()
        got.append([x.cpu().numpy() for x in out])
    _same(got[0], got[1], f"lanes {lanes}")
