"""GPU: one insert whose attach groups span every build shape (1-8, 9-128 and
129-1024 points, and larger ones) and both plan forms (up to 8192 groups and
more): the tree is node for node the one the level-synchronous build makes."""
import importlib

import numpy as np
import pytest

from common import uniform_cloud

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,sizes", [(64, [1, 2, 7, 8, 9, 10, 64, 65, 127, 128, 129, 130, 500, 1023, 1024]),
                                     (64, [8, 128, 1024, 1025, 3000]), (300, [3] * 200), (30000, [1] * 9500),
                                     (30000, [1] * 8192), (5, [1])])
def test_groups_of_every_shape(n, sizes):
    ikd = importlib.import_module("ikd-tree_amd")
    rng = np.random.default_rng(n + len(sizes))
    base = uniform_cloud(rng, n)
    # clusters far outside the base's cells end up in slots of their own, or share one
    parts = []
    for i, m in enumerate(sizes):
        c = base[rng.integers(0, n)] + rng.normal(0, 1e-3, 3)
        parts.append((c + rng.normal(0, 1e-4, (m, 3))).astype(np.float32))
    add = np.concatenate(parts)
    add[::5] = np.round(add[::5] * 8) / 8  # some equal coordinates
    got = []
    for small in (1, 0):
        t = ikd.KD_TREE(0.5, 0.6, 0.5)
        t.set_tuning(ikd.IKD_TUNE_SMALL_BUILD, small)
        t.Build(base)
        t.Add_Points(add, False)
        got.append((t.dump_nodes(), t.size(), t.validnum()))
        assert t.validnum() == n + len(add)
    assert got[0][0].tobytes() == got[1][0].tobytes() and got[0][1:] == got[1][1:]
