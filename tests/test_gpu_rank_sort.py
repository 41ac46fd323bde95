"""GPU: builds and downsampled inserts at the sizes where the two-launch sort can
go wrong: one tile (2048 keys), its edges, ragged last tiles, its longest list
(65536) and the first one the library sorts, with all keys alike and with many
ties.  The tree of a Build is checked against the recursive median definition
with ties in input order, a downsampled insert against a map of voxels."""
import importlib

import numpy as np
import pytest

from common import grid_cloud, uniform_cloud

pytestmark = pytest.mark.gpu


def _median_tree(p):
    """Pre-order ids of the median-split tree, ties in input order (stable sort per axis)."""
    out, stack = [], [np.arange(len(p))]
    while stack:
        ix = stack.pop()
        if len(ix) == 0:
            continue
        q = p[ix]
        ext = q.max(axis=0) - q.min(axis=0)
        axis = 0
        for a in (1, 2):
            if ext[a] > ext[axis]:
                axis = a
        order = ix[np.argsort(q[:, axis], kind="stable")]
        m = (len(ix) - 1) >> 1
        out.append(order[m])
        keep = np.zeros(len(p), bool)
        keep[order[:m]] = True
        left = ix[keep[ix]]
        keep[order[:m]] = False
        keep[order[m + 1:]] = True
        stack.append(ix[keep[ix]])
        stack.append(left)
    return np.array(out, np.uint32)


@pytest.mark.parametrize("n,kind", [(1025, "uniform"), (200001, "uniform"), (131072, "grid"), (2047, "grid"), (2048, "uniform"), (2049, "same"),
                                    (4097, "grid"), (30001, "uniform"), (65535, "grid"), (65536, "uniform"),
                                    (65537, "uniform")])
def test_build_order(n, kind):
    ikd = importlib.import_module("ikd-tree_amd")
    rng = np.random.default_rng(n)
    p = {"uniform": uniform_cloud, "grid": lambda r, m: grid_cloud(r, m, extent=30),
         "same": lambda r, m: np.full((m, 3), 1.5, np.float32)}[kind](rng, n)
    p = p + np.float32(0.0)  # no negative zeros: they sort below zero here
    t = ikd.KD_TREE(0.5, 0.6, 0.5)
    t.Build(p)
    assert np.array_equal(t.dump_nodes()["id"], _median_tree(p))


@pytest.mark.parametrize("n", [1, 2048, 2049, 65536, 65537])
def test_downsample_order(n):
    """Same voxels: the nearest point to each voxel's centre stays (the last of equals)."""
    ikd = importlib.import_module("ikd-tree_amd")
    rng = np.random.default_rng(n)
    p = grid_cloud(rng, n, step=0.125, extent=60) + np.float32(0.0625)
    t = ikd.KD_TREE(0.5, 0.6, 0.5)
    t.Build(np.array([[500.0, 500, 500]], np.float32), ids=np.array([10 ** 9], np.uint32))
    t.Add_Points(p, True, ids=np.arange(n, dtype=np.uint32))
    v = np.floor(p / np.float32(0.5)).astype(np.int64)
    d = ((p - (v * 0.5 + 0.25)) ** 2).astype(np.float32).sum(axis=1)
    best = {}
    for i, key in enumerate(map(tuple, v)):
        if key not in best or d[i] <= d[best[key]]:
            best[key] = i
    _, ids = t.flatten()
    assert sorted(ids.tolist()) == sorted(list(best.values()) + [10 ** 9])
