"""GPU: a range search with more than 2^31 items of the usual size (20000 boxes
around a map of 2M points) is planned with larger ones."""
import ctypes
import importlib

import numpy as np
import pytest

from common import uniform_cloud

pytestmark = pytest.mark.gpu


def test_counts_of_very_many_points():
    ikd = importlib.import_module("ikd-tree_amd")
    rng = np.random.default_rng(9)
    n, nq = 2_100_000, 20_000  # 32-node items: 131071 a box, 2.6e9 in all
    t = ikd.KD_TREE(0.5, 0.6, 0.5)
    p = uniform_cloud(rng, n)
    t.Build(p)
    boxes = np.tile(np.array([-60] * 3 + [60] * 3, np.float32), (nq, 1))
    boxes[7] = [0, 0, 0, 1, 1, 1]
    off = np.zeros(nq + 1, np.int64)
    ptr = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    assert t._lib.ikd_box_search(t._h, ptr(boxes), nq, ptr(off), None, None, 0) == ikd.IKD_OK
    want = np.full(nq, n, np.int64)
    want[7] = np.count_nonzero(np.all((p >= 0) & (p < 1), axis=1))
    assert np.array_equal(np.diff(off), want)
    off, _, ids = t.box_search_batch(boxes[7:8])  # a plan of the usual size again
    assert len(ids) == want[7]
