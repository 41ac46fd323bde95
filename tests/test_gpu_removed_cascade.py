"""GPU: rebuilds that record removed points while violators lie below the
rebuilt subtree's root.

The refit leaves post-rebuild counts in the lower violators, and a recording
rebuild walks every node, so its buffers need the nodes those counts hide: with
too few the walk stopped early and the build read points no kernel had written.
The tree has to hold the same live points with and without the record.
"""
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _line(n, step):
    p = np.zeros((n, 3), np.float32)
    p[:, 0] = np.arange(n) * step
    return p


@pytest.mark.parametrize("kind,n,m", [("line", 210, 500), ("line", 411, 800), ("scan", 12000, 12000)])
def test_cascading_downsample_rebuilds_with_the_record_on(kind, n, m):
    ikd = importlib.import_module("ikd-tree_amd")
    if kind == "line":
        pts, add = _line(n, 0.01), _line(m, 0.01)
    else:
        scene = importlib.import_module("ikd-tree_amd.scenes").MappingScene(1001)
        pts, add = scene.scan(0)[:n], scene.scan(3)[:m]
    live = []
    for record in (0, 1):
        t = ikd.KD_TREE(0.5, 0.6, 1.0)
        t.set_tuning(ikd.IKD_TUNE_RECORD_REMOVED, record)
        t.Build(pts)
        added = [t.Add_Points(add + np.float32(0.3 * i), True) for i in range(2)]
        xyz, ids = t.flatten()
        assert t.validnum() == len(ids) == len(set(ids.tolist()))
        assert len(t.acquire_removed_points()[1]) == 0  # the downsample's own deletions are never recorded
        live.append((added, sorted(ids.tolist())))
    assert live[0] == live[1]
