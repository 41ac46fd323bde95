"""GPU: results delivered to host arrays, at the sizes where the way changes:
through page-locked memory (up to 64 KB of queries and results), by one DMA
into a page-locked block, and into ordinary arrays when too much is lent out.
Results stay valid while any array on them lives, whatever is searched next."""
import importlib
import threading

import numpy as np
import pytest

from common import in_box, random_boxes, uniform_cloud

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ikd():
    return importlib.import_module("ikd-tree_amd")


def _tree(ikd, rng, n=20000):
    t = ikd.KD_TREE(0.5, 0.6, 0.5)
    p = uniform_cloud(rng, n)
    t.Build(p)
    return t, p


@pytest.mark.parametrize("k", [1, 7])
def test_sizes_around_the_switches(ikd, k):
    rng = np.random.default_rng(k)
    t, _ = _tree(ikd, rng)
    per = 16 + 20 * k  # bytes a query moves
    q = uniform_cloud(rng, 2 * 65536 // per + 40)
    ref = t.knn(q, k, 3.0)
    for nq in (1, 65536 // per - 1, 65536 // per, 65536 // per + 1, 65536 // (4 + 20 * k) + 1, len(q)):
        got = t.knn(q[:nq], k, 3.0)
        for a, b in zip(ref, got):
            assert b.shape[0] == nq and np.array_equal(a[:nq], b)


def test_results_outlive_later_searches_and_the_tree(ikd):
    rng = np.random.default_rng(3)
    t, p = _tree(ikd, rng)
    q = uniform_cloud(rng, 9000)
    first = t.knn(q, 5)
    copy = [a.copy() for a in first]
    d2 = first[1]
    del first  # one array of the block stays
    for _ in range(5):
        t.knn(q[::-1], 5)
    assert np.array_equal(d2, copy[1])
    boxes = random_boxes(rng, 60)
    off, xyz, ids = t.box_search_batch(boxes)
    again = t.box_search_batch(boxes)  # with room from the first call
    bigger = t.box_search_batch(np.array([[-60] * 3 + [60] * 3] * 3, np.float32))  # more than there is room for
    t.close()
    assert bigger[0][-1] == 3 * len(p) and np.array_equal(np.sort(bigger[2][:len(p)]), np.arange(len(p)))
    for i in range(60):
        assert set(ids[off[i]:off[i + 1]].tolist()) == set(np.nonzero(in_box(p, boxes[i]))[0].tolist())
    for a, b in zip((off, xyz, ids), again):
        assert np.array_equal(a, b)


def test_lending_is_bounded_and_safe_with_threads(ikd):
    rng = np.random.default_rng(4)
    mem = ikd._ResultMemory(ikd.load_library())
    mem.LENT, mem.CACHED = 1 << 20, 200_000
    blocks = [mem.take(100_000) for _ in range(30)]
    lent = [b for b in blocks if b is not None]
    assert 0 < len(lent) < 30 and sum(b.nbytes for b in lent) <= mem.LENT
    del blocks, lent
    assert mem._lent == 0 and mem._cached <= mem.CACHED
    t, _ = _tree(ikd, rng)
    qs = [uniform_cloud(rng, 4000) for _ in range(6)]
    want = [[a.copy() for a in t.knn(q, 5)] for q in qs]
    bad = []

    def work(i):
        for _ in range(20):
            got = t.knn(qs[i], 5)
            bad.extend(i for a, b in zip(want[i], got) if not np.array_equal(a, b))

    th = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    [x.start() for x in th]
    [x.join() for x in th]
    assert not bad
