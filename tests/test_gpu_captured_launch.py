"""GPU: a no-alloc launch that the caller captures from the batch's stream into a
graph of its own.  Replays give the eager launch's results, and the launches and
tree updates around the capture keep their order."""
import ctypes
import importlib

import numpy as np
import pytest

from common import uniform_cloud

pytestmark = pytest.mark.gpu


def test_captured_noalloc_launch():
    import torch

    ikd = importlib.import_module("ikd-tree_amd")
    hip = ctypes.CDLL("libamdhip64.so")
    rng = np.random.default_rng(21)
    base = uniform_cloud(rng, 60000)
    trees = [ikd.KD_TREE(0.5, 0.6, 0.5) for _ in range(2)]
    for t in trees:
        t.Build(base)
    n, k = 30000, 5
    q = torch.from_numpy(uniform_cloud(rng, n)).to("cuda:0")
    qt = torch.from_numpy(rng.integers(0, 2, n).astype(np.int32)).to("cuda:0")

    def outs():
        return (torch.zeros((n, k, 3), device="cuda:0"), torch.zeros((n, k), device="cuda:0"),
                torch.zeros((n, k), dtype=torch.int32, device="cuda:0"),
                torch.zeros((n,), dtype=torch.int32, device="cuda:0"))

    b = ikd.Batch()
    st = ctypes.c_void_p(b.stream())
    before, after, recorded = outs(), outs(), outs()
    torch.cuda.synchronize()
    b.nearest_search_noalloc(trees, qt, q, k, *before)
    graph, exe = ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamBeginCapture(st, 1) == 0
    b.nearest_search_noalloc(trees, qt, q, k, *recorded)
    assert hip.hipStreamEndCapture(st, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, ctypes.c_size_t(0)) == 0
    b.synchronize()
    assert int(recorded[3].sum()) == 0  # nothing ran yet
    for _ in range(3):
        for o in recorded:
            o.zero_()
        torch.cuda.synchronize()
        assert hip.hipGraphLaunch(exe, st) == 0
        b.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(recorded, before))
        b.nearest_search_device(trees, qt, q, k, *outs())
    trees[0].Delete_Point_Boxes(np.array([[-50, -50, -50, 0, 50, 50]], np.float32))
    b.nearest_search_device(trees, qt, q, k, *after)
    b.synchronize()
    assert float(after[0][qt == 0][:, :, 0].min()) >= 0.0
    assert torch.equal(after[2][qt == 1], before[2][qt == 1])
    assert hip.hipGraphExecDestroy(exe) == 0 and hip.hipGraphDestroy(graph) == 0
