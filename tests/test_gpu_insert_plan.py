"""GPU: an insert of up to 8192 points is planned by one workgroup, a longer one
by several launches.  Two inserts on either side of the tree, far apart, leave
the same nodes in one call (long) as in two (the first one short)."""
import importlib

import numpy as np
import pytest

from common import check_dump_invariants, uniform_cloud

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spread", ["wide", "one slot", "pairs"])
@pytest.mark.parametrize("m", [1, 2, 63, 64, 65, 1023, 1025, 8191, 8192])
def test_short_plan_equals_long_plan(m, spread):
    ikd = importlib.import_module("ikd-tree_amd")
    rng = np.random.default_rng(m)
    base = uniform_cloud(rng, 3000)
    left = base[base[:, 0] < -25]
    if spread == "wide":
        a = rng.uniform((-50, -50, -50), (-30, 50, 50), (m, 3))
    elif spread == "one slot":
        a = left[0] + rng.normal(0, 1e-3, (m, 3))
    else:  # points of both sides of each node, in both of its slots
        a = left[rng.integers(0, len(left), m)] + rng.normal(0, 1e-2, (m, 3))
    a = a.astype(np.float32)
    b = rng.uniform((30, -50, -50), (50, 50, 50), (8193, 3)).astype(np.float32)
    got = []
    for calls in ([a, b], [np.concatenate([a, b])]):
        t = ikd.KD_TREE(0.99, 0.99, 0.5)
        t.Build(base)
        for p in calls:
            t.Add_Points(p, False)
        got.append((t.dump_nodes(), t.size(), t.validnum()))
    check_dump_invariants(got[0][0])
    assert got[0][1:] == got[1][1:] == (3000 + m + 8193,) * 2
    # ids: points are numbered in the order they came, which is the same here
    assert got[0][0].tobytes() == got[1][0].tobytes()
