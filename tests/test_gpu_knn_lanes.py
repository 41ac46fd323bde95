"""GPU: kNN launches around the sizes where the lanes per query change on a map of
more than 3 * 2^16 node slots (73728 and 90112 queries, k 5 and 6): the bits of one lane per query,
from the tree, a batch and a recorded launch."""
import importlib

import numpy as np
import pytest
import torch

from common import uniform_cloud

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [5, 6])
def test_lanes_above_a_full_device(k):
    ikd = importlib.import_module("ikd-tree_amd")
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    rng = np.random.default_rng(k)
    t = ikd.KD_TREE(0.5, 0.6, 0.5)
    t.Build(uniform_cloud(rng, 200000))
    b = ikd.Batch()
    for nq in (73728, 73729, 90112, 90113):
        q = torch.from_numpy(uniform_cloud(rng, nq)).to(dev)
        qt = torch.zeros(nq, dtype=torch.int32, device=dev)
        outs = [(torch.zeros((nq, k, 3), device=dev), torch.zeros((nq, k), device=dev),
                 torch.zeros((nq, k), dtype=torch.int32, device=dev), torch.zeros(nq, dtype=torch.int32, device=dev))
                for _ in range(4)]
        if dev.type == "cuda":
            torch.cuda.synchronize()
        t.set_tuning(ikd.IKD_TUNE_LANES_PER_QUERY, 1)
        t.knn_device(q, k, 9.0, *outs[0])
        t.set_tuning(ikd.IKD_TUNE_LANES_PER_QUERY, -1)
        t.knn_device(q, k, 9.0, *outs[1])
        t.synchronize()
        b.nearest_search_device([t], qt, q, k, *outs[2], max_dist=9.0)
        g = b.knn_graph([t], qt, q, k, *outs[3], max_dist=9.0)
        g.launch()
        b.synchronize()
        g.close()
        for got in outs[1:]:
            assert all(torch.equal(x, y) for x, y in zip(outs[0], got))
