"""The package's range search (Box_Search, Radius_Search) over a stand-in for the
library: the room made for results follows earlier calls, but stays bounded by
what was searched, and results keep no more memory alive than they need."""
import ctypes
import importlib

import numpy as np
import pytest

ikd = importlib.import_module("ikd-tree_amd")


class Library:
    """ikd_box_search and ikd_radius_search of a tree whose query i finds counts[i]
    points, the j-th result being (j, 0, 0) with id j; no page-locked memory."""

    def __init__(self):
        self.counts, self.rooms, self.calls = [], [], 0

    def ikd_host_alloc(self, nbytes, out):
        return -1

    def ikd_destroy(self, h):
        return ikd.IKD_OK

    def _search(self, n, off, xyz, ids, capacity):
        self.calls += 1
        self.rooms.append(capacity)
        o = np.frombuffer((ctypes.c_int64 * (n + 1)).from_address(off.value), np.int64)
        o[:] = np.concatenate([[0], np.cumsum(self.counts[:n])])
        total = int(o[n])
        if xyz is None:
            return ikd.IKD_OK
        if capacity < total:
            return ikd.IKD_ERR_CAPACITY
        if total:
            np.frombuffer((ctypes.c_uint32 * total).from_address(ids.value), np.uint32)[:] = np.arange(total)
            x = np.frombuffer((ctypes.c_float * (3 * total)).from_address(xyz.value), np.float32).reshape(-1, 3)
            x[:] = 0
            x[:, 0] = np.arange(total)
        return ikd.IKD_OK

    def ikd_box_search(self, h, boxes, n, off, xyz, ids, capacity):
        return self._search(n, off, xyz, ids, capacity)

    def ikd_radius_search(self, h, centers, radii, n, off, xyz, ids, capacity):
        return self._search(n, off, xyz, ids, capacity)


@pytest.fixture(params=["box", "radius"])
def search(request):
    lib = Library()
    t = object.__new__(ikd.KD_TREE)
    t._lib, t._h, t._room = lib, None, {}

    def call(counts):
        lib.counts = counts
        if request.param == "box":
            r = t.box_search_batch(np.zeros((len(counts), 6), np.float32))
        else:
            r = t.radius_search_batch(np.zeros((len(counts), 3), np.float32), 1.0)
        off, xyz, ids = r
        total = sum(counts)
        assert off.tolist() == np.concatenate([[0], np.cumsum(counts)]).tolist()
        assert xyz.shape == (total, 3) and ids.tolist() == list(range(total))
        assert np.array_equal(xyz[:, 0], np.arange(total, dtype=np.float32))
        return r

    return lib, call


def _kept(a):
    """Bytes of the memory that the array keeps alive."""
    while isinstance(a.base, np.ndarray):
        a = a.base
    return a.nbytes


@pytest.mark.parametrize("few,many", [(1, 200), (1, 20000), (3, 60000)])
def test_a_dense_search_before_a_sparse_one(search, few, many):
    lib, call = search
    call([200_000] * few)
    sparse = [i % 2 for i in range(many)]
    for _ in range(2):
        lib.rooms.clear()
        _, xyz, ids = call(sparse)
        assert max(lib.rooms) <= 4_200_000  # points, about 64 MB
        assert _kept(xyz) <= 32 * len(ids) and _kept(ids) <= 32 * len(ids)


def test_repeated_searches_find_and_deliver_in_one_call(search):
    lib, call = search
    call([50] * 100)
    lib.calls = 0
    for scale in (50, 55, 45, 50):
        call([scale] * 100)
    assert lib.calls == 4
    lib.calls = 0
    call([5] * 100)
    call([0] * 100)
    call([7] * 100)  # nothing was found before: counted, then delivered
    call([])
    assert lib.calls == 5
