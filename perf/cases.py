"""What this framework is timed on: the calls a mapping program makes, from one
query to a map of two million points, through the package's public classes.

Points come from the repository's own generators (``ikd-tree_amd.scenes``): the
LiDAR-like mapping scene (32 x 1800 rays, about 37-42k points per scan) or a
uniform cloud, both from the seed alone.  Maps of a given size are raw scans of
every 7th pose of the scene's path; queries are scans of the poses in between.

``listed()`` names the cases, ``draw(rng)`` gives one more of the same ranges,
``prepare`` makes what the program holds before the call, ``run`` is one pass,
``work`` the bytes and operations a pass cannot do without, ``exact`` the
squared distances of a k-nearest search in 64 bits.
"""
import importlib
import math
import os
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

ikd = importlib.import_module("ikd-tree_amd")
scenes = importlib.import_module("ikd-tree_amd.scenes")

POSE_STEP = 7  # map scans every 7th pose, 1 m apart
SCAN = 29_000  # every scan holds more points than this


def listed():
    return [
        # one Nearest_Search from a program's own loop: host in, host out
        {"name": "one query", "op": "host_knn", "scene": "uniform", "points": 100_000, "queries": 1, "k": 5,
         "max_dist": None},
        # a point cloud against a small map, host in, host out
        {"name": "10k host queries", "op": "host_knn", "scene": "uniform", "points": 100_000, "queries": 10_000,
         "k": 10, "max_dist": None},
        # scan matching: one scan against a large map, resident on the GPU
        {"name": "one scan, 2M map", "op": "knn", "scene": "lidar", "points": 2_000_000, "queries": 37_003, "k": 5,
         "max_dist": 5.0},
        # the benchmark's launch: 32 scans at once against the same map
        {"name": "32 scans, 2M map", "op": "knn", "scene": "lidar", "points": 2_000_000, "queries": 1_180_000, "k": 5,
         "max_dist": 5.0},
        # many robots' maps in one launch, each query with its own k and max_dist
        {"name": "16 maps, mixed k", "op": "batch_knn", "maps": 16, "points": 3_000_000, "queries": 300_000, "k": 20},
        # balls around scan points over many maps, results left on the GPU
        {"name": "16 maps, balls", "op": "batch_radius", "maps": 16, "points": 3_000_000, "queries": 20_000,
         "radius": 1.0, "room": 8_000_000},
        # the first scan of a run becomes the map
        {"name": "build a scan", "op": "build", "scene": "lidar", "points": 29_001, "queries": 4_001},
        # a stored map is loaded and the first scan is matched against it
        {"name": "build 2M", "op": "build", "scene": "lidar", "points": 2_000_000, "queries": 29_000},
        # incremental mapping as a LiDAR odometry runs it: search, then insert with 0.5 m voxels
        {"name": "mapping, 20 scans", "op": "mapping", "api": "device", "frames": 20, "scan": 29_000, "voxel": 0.5,
         "k": 5, "max_dist": 5.0},
        # the same from host arrays with the class's default voxel size, thinned scans
        {"name": "mapping from host", "op": "mapping", "api": "host", "frames": 8, "scan": 15_001, "voxel": 0.2,
         "k": 5, "max_dist": 5.0},
        # a local window kept around the sensor: insert, delete single points, trim what lies outside
        {"name": "window on 1M map", "op": "window", "points": 1_000_000, "frames": 4, "scan": 29_000, "voxel": 0.5,
         "half": 60.0, "deletes": 300},
        # regions of a map read back to the host
        {"name": "boxes to host", "op": "host_boxes", "points": 1_000_000, "queries": 200, "side": 40},
    ]


def _log(rng, lo, hi):
    """A whole number, its logarithm uniform."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["host_knn", "knn", "knn", "batch_knn", "batch_radius", "build", "mapping", "mapping", "window",
                     "host_boxes"])
    scene = rng.choice(["lidar", "uniform"])
    k = rng.choice([1, 2, 5, 8, 10, 20])
    max_dist = rng.choice([None, 1.0, 5.0])
    if op == "host_knn":
        return {"op": op, "scene": scene, "points": _log(rng, 500, 300_000), "queries": _log(rng, 1, 20_000), "k": k,
                "max_dist": max_dist}
    if op == "knn":
        return {"op": op, "scene": "lidar", "points": _log(rng, 20_000, 2_000_000),
                "queries": _log(rng, 1_000, 500_000), "k": min(k, 10), "max_dist": rng.choice([1.0, 5.0])}
    if op == "batch_knn":
        return {"op": op, "maps": rng.randint(2, 16), "points": _log(rng, 50_000, 2_000_000),
                "queries": _log(rng, 2_000, 200_000), "k": rng.choice([5, 10, 20])}
    if op == "batch_radius":
        return {"op": op, "maps": rng.randint(2, 16), "points": _log(rng, 50_000, 2_000_000),
                "queries": _log(rng, 500, 10_000), "radius": rng.choice([0.3, 0.6, 1.0]), "room": 6_000_000}
    if op == "build":
        return {"op": op, "scene": scene, "points": _log(rng, 700, 1_500_000), "queries": _log(rng, 500, 30_000)}
    if op == "mapping":
        return {"op": op, "api": rng.choice(["device", "host"]), "frames": rng.randint(3, 12),
                "scan": _log(rng, 5_000, 29_000), "voxel": rng.choice([0.2, 0.25, 0.5, 1.0]), "k": min(k, 10),
                "max_dist": 5.0}
    if op == "window":
        return {"op": op, "points": _log(rng, 100_000, 1_000_000), "frames": rng.randint(1, 4),
                "scan": _log(rng, 5_000, 29_000), "voxel": rng.choice([0.25, 0.5, 1.0]),
                "half": rng.choice([40.0, 60.0, 90.0]), "deletes": rng.randint(50, 500)}
    return {"op": op, "points": _log(rng, 80_000, 1_000_000), "queries": _log(rng, 20, 200),
            "side": rng.randint(4, 40)}


# ------------------------------------------------------------------- inputs
def _cpus():
    return max(1, min(16, len(os.sched_getaffinity(0))))


def _scans(seed, frames):
    sc = scenes.MappingScene(1000 + seed)
    with ThreadPoolExecutor(_cpus()) as pool:  # the generator releases the interpreter lock
        return list(pool.map(sc.scan, frames))


def _cloud(case, seed):
    """(map points, query points) of a case, as float32 rows."""
    n, nq = case["points"], case["queries"]
    if case.get("scene") == "uniform":
        return scenes.uniform(1000 + seed, n), scenes.uniform(1000 + seed, nq, stream=1)
    nm, ns = -(-n // SCAN), -(-nq // SCAN)
    first = list(range(0, nm * POSE_STEP, POSE_STEP))
    between = [f for f in range(max(nm, ns) * POSE_STEP) if f % POSE_STEP][:: max(1, nm * (POSE_STEP - 1) // ns)][:ns]
    got = _scans(seed, first + between)
    m, q = np.concatenate(got[:nm]), np.concatenate(got[nm:])
    # a map below one scan and a query set below a scan are thinned over the whole scan
    return _thin(m, n), _thin(q, nq)


def _thin(p, n):
    """n of the points, evenly over their order."""
    return np.ascontiguousarray(p[(np.arange(n) * len(p)) // n])


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


def _outs(n, k):
    return (torch.empty((n, k, 3), dtype=torch.float32, device="cuda:0"),
            torch.empty((n, k), dtype=torch.float32, device="cuda:0"),
            torch.empty((n, k), dtype=torch.int32, device="cuda:0"),
            torch.empty((n,), dtype=torch.int32, device="cuda:0"))


def _inf(max_dist):
    return float("inf") if max_dist is None else float(max_dist)


def _maps(case, seed):
    """Uneven maps and query sets of one multi-tree call: points per map, queries, map of each query."""
    m = case["maps"]
    w, u = np.exp(np.random.default_rng(m).uniform(0.0, math.log(30.0), (2, m)))
    sizes = np.maximum((case["points"] * w / w.sum()).astype(int), 500)
    counts = np.maximum((case["queries"] * u / u.sum()).astype(int), 1)
    pts, qs = [], []
    for i in range(m):
        p, q = _cloud({"points": int(sizes[i]), "queries": int(counts[i])}, 100 * (seed % 10**6) + i)
        pts.append(p)
        qs.append(q)
    qt = np.concatenate([np.full(len(q), i, np.int32) for i, q in enumerate(qs)])
    q = np.concatenate(qs)
    return pts, q, qt, np.random.default_rng(seed)


def _box_cells(case):
    """Cells along the cube's edge, and along each box's edges: the same for every seed."""
    e = max(int(round(case["points"] ** (1 / 3))), case["side"] + 1)
    rng = np.random.default_rng(case["queries"])
    return e, np.exp(rng.uniform(0.0, math.log(case["side"] + 1), (case["queries"], 3))).astype(np.int64)


def _filled(case, seed):
    """A cube of 0.25 m cells with one point in each, in no order, and boxes of whole cells: the boxes' results
    are as many for every seed."""
    e, side = _box_cells(case)
    rng = np.random.default_rng(seed)
    at = np.stack(np.unravel_index(rng.permutation(e ** 3), (e, e, e)), axis=1)
    lo = rng.integers(0, e - side + 1)
    p = ((at + 0.05 + 0.9 * rng.random((e ** 3, 3))) * 0.25).astype(np.float32)
    return p, (np.concatenate([lo, lo + side], axis=1) * 0.25).astype(np.float32)


def _knn_mix(case, n, rng):
    ks = rng.choice(np.array([k for k in (1, 5, 10, 20) if k <= case["k"]], np.int32), n)
    return ks, rng.choice(np.array([1.0, 5.0, np.inf]), n)


def _trees(pts, box=0.5):
    got = []
    for p in pts:
        t = ikd.KD_TREE(0.5, 0.6, box)
        t.Build(p)
        got.append(t)
    return got


def _outside(center, half):
    """Six half-open slabs: everything outside a cube around the sensor."""
    big = 1e7
    lo, hi = center - half, center + half
    return np.array([[-big, -big, -big, lo[0], big, big], [hi[0], -big, -big, big, big, big],
                     [-big, -big, -big, big, lo[1], big], [-big, hi[1], -big, big, big, big],
                     [-big, -big, -big, big, big, lo[2]], [-big, -big, hi[2], big, big, big]], np.float32)


def prepare(case, seed):
    op = case["op"]
    s = {"case": case}
    if op == "host_knn":
        m, s["q"] = _cloud(case, seed)
        s["tree"] = _trees([m])[0]
    elif op == "knn":
        m, q = _cloud(case, seed)
        s["tree"], s["q"], s["out"] = _trees([m])[0], _dev(q), _outs(len(q), case["k"])
    elif op == "batch_knn":
        pts, q, qt, rng = _maps(case, seed)
        ks, md = _knn_mix(case, len(q), rng)
        s.update(trees=_trees(pts), batch=ikd.Batch(), q=_dev(q), qt=_dev(qt), ks=_dev(ks), md=_dev(md),
                 out=_outs(len(q), case["k"]))
    elif op == "batch_radius":
        pts, q, qt, rng = _maps(case, seed)
        r = (0.1 * case["radius"] + 0.9 * case["radius"] * rng.random(len(q))).astype(np.float32)
        s.update(trees=_trees(pts), batch=ikd.Batch(), q=_dev(q), qt=_dev(qt), r=_dev(r),
                 off=torch.empty(len(q) + 1, dtype=torch.int64, device="cuda:0"))
        # the program sizes its result buffers once; rows past the results stay zero
        s["xyz"] = torch.zeros((case["room"], 3), dtype=torch.float32, device="cuda:0")
        s["ids"] = torch.zeros(case["room"], dtype=torch.int32, device="cuda:0")
    elif op == "build":
        s["points"], q = _cloud(case, seed)
        s["tree"], s["q"], s["out"] = ikd.KD_TREE(0.5, 0.6, 0.5), _dev(q), _outs(len(q), 5)
    elif op == "mapping":
        got = [_thin(p, case["scan"]) for p in _scans(seed, range(case["frames"] + 1))]
        s["tree"], s["first"], k = ikd.KD_TREE(0.5, 0.6, case["voxel"]), got[0], case["k"]
        if case["api"] == "device":
            s["scans"] = [_dev(p) for p in got[1:]]
            s["out"] = _outs(sum(len(p) for p in got[1:]), k)
            at = np.cumsum([0] + [len(p) for p in got[1:]])
            s["rows"] = [tuple(o[a:b] for o in s["out"]) for a, b in zip(at[:-1], at[1:])]
            s["all"], s["live"] = _dev(np.concatenate(got)), _outs(sum(map(len, got)), 1)
        else:
            s["scans"], s["all"] = got[1:], np.concatenate(got)
    elif op == "window":
        nm = -(-case["points"] // SCAN)
        got = _scans(seed, [POSE_STEP * i for i in range(nm)] + [POSE_STEP * i + 3 for i in range(case["frames"])])
        m = _thin(np.concatenate(got[:nm]), case["points"])
        scans = [_thin(p, case["scan"]) for p in got[nm:]]
        at = np.cumsum([0] + [len(p) for p in scans])
        s["tree"] = _trees([m], case["voxel"])[0]
        s["scans"] = [_dev(p) for p in scans]
        s["ids"] = [_dev(np.arange(a, b, dtype=np.int32) + len(m)) for a, b in zip(at[:-1], at[1:])]
        s["out"] = _outs(int(at[-1]), 5)
        s["rows"] = [tuple(o[a:b] for o in s["out"]) for a, b in zip(at[:-1], at[1:])]
        s["gone"] = _thin(scans[0], min(case["deletes"], len(scans[0])))
        s["slabs"] = _outside(scenes.MappingScene(1000 + seed).pose(3), case["half"])
        torch.cuda.synchronize()  # the tree has a stream of its own
        # the sensor stands still: after these passes every further one finds and leaves the same points
        for _ in range(3):
            run(s)
    elif op == "host_boxes":
        m, s["boxes"] = _filled(case, seed)
        s["tree"] = _trees([m])[0]
    else:
        raise ValueError(op)
    return s


def run(s):
    case = s["case"]
    op = case["op"]
    if op == "host_knn":
        return s["tree"].knn(s["q"], case["k"], _inf(case["max_dist"]))
    if op == "knn":
        s["tree"].knn_device(s["q"], case["k"], _inf(case["max_dist"]), *s["out"])
        return s["out"]
    if op == "batch_knn":
        s["batch"].nearest_search_device(s["trees"], s["qt"], s["q"], case["k"], *s["out"], k=s["ks"],
                                         max_dist=s["md"])
        return s["out"]
    if op == "batch_radius":
        n = s["batch"].radius_search_device(s["trees"], s["qt"], s["q"], s["r"], s["off"], s["xyz"], s["ids"])
        return n, s["off"], s["xyz"], s["ids"]
    if op == "build":
        t = s["tree"]
        t.Build(s["points"])
        t.knn_device(s["q"], 5, 5.0, *s["out"])
        return s["out"], t.tree_range(), t.size(), t.validnum()
    if op == "mapping":
        t, k, md = s["tree"], case["k"], _inf(case["max_dist"])
        t.Build(s["first"])
        added, found = [], []
        for i, p in enumerate(s["scans"]):
            if case["api"] == "device":
                t.knn_device(p, k, md, *s["rows"][i])
                added.append(t.add_points_device(p, True))
            else:
                found.append(t.knn(p, k, md))
                added.append(t.Add_Points(p, True))
        # every live point is one of these scans' points: the nearest of each are the whole map
        if case["api"] == "device":
            t.knn_device(s["all"], 1, float("inf"), *s["live"])
            return s["out"], added, s["live"], t.validnum()
        return found, added, t.knn(s["all"], 1), t.validnum()
    if op == "window":
        t = s["tree"]
        added = []
        for p, ids, rows in zip(s["scans"], s["ids"], s["rows"]):
            t.knn_device(p, 5, 5.0, *rows)
            added.append(t.add_points_device(p, True, ids))
        t.Delete_Points(s["gone"])
        return s["out"], added, t.Delete_Point_Boxes(s["slabs"]), t.validnum()
    return s["tree"].box_search_batch(s["boxes"])


# ------------------------------------------------------------- what it takes
NODE = 92  # bytes a node of the resident tree holds


def work(case):
    """Each input and each point of a map read once (a search of few queries
    reads no more of the map than its results and one path down), each output
    and each new node written once; a squared distance is 8 operations."""
    op = case["op"]

    def knn(n, nq, k):
        seen = min(16 * n, nq * (16 * k + 64 * math.log2(n + 2)))
        return 12 * nq + seen + nq * (20 * k + 4), 8.0 * nq * (k + math.log2(n + 2))

    if op in ("host_knn", "knn"):
        b, f = knn(case["points"], case["queries"], case["k"])
    elif op == "batch_knn":
        b, f = knn(case["points"], case["queries"], case["k"])
        b += 16 * case["queries"]
    elif op == "batch_radius":
        hits = case["queries"] * 60.0 * case["radius"] ** 2  # these maps hold about 60 points in a ball of 1 m
        b, f = 16 * case["points"] + 28 * case["queries"] + 16 * hits, 8.0 * hits
    elif op == "build":
        b, f = knn(case["points"], case["queries"], 5)
        b += (12 + NODE) * case["points"]
        f += 3.0 * case["points"] * math.log2(case["points"] + 2)
    elif op == "mapping":
        n = case["scan"]
        b, f = knn(n, n * case["frames"], case["k"])
        b += (12 + NODE) * n + case["frames"] * n * 24 + 16 * n
        f += 16.0 * n * case["frames"]
    elif op == "window":
        n = case["scan"] * case["frames"]
        b, f = knn(case["points"], n, 5)
        b, f = b + 24 * n, f + 16.0 * n
    else:
        hits = float(_box_cells(case)[1].prod(axis=1).sum())
        b, f = 16 * case["points"] + 24 * case["queries"] + 16 * hits, 6.0 * hits
    return {"bytes": b, "flops": f}


# ------------------------------------------------------------------ 64 bits
PAIRS = 1.2e11  # query-point pairs gone through one by one within seconds


def _nearest(m, q, k, max_dist, limit=None):
    """Squared distances of the k nearest, ascending, in 64 bits; inf past max_dist (and past limit[i] results)."""
    m = _dev(m).double()
    q = _dev(q).double()
    kk = min(k, len(m))
    out = torch.full((len(q), k), float("inf"), dtype=torch.float64, device=q.device)
    step = max(1, int(2.5e8 // len(m)))
    for a in range(0, len(q), step):
        d = (q[a:a + step, 0:1] - m[None, :, 0]).square_()
        d += (q[a:a + step, 1:2] - m[None, :, 1]).square_()
        d += (q[a:a + step, 2:3] - m[None, :, 2]).square_()
        out[a:a + step, :kk] = d.topk(kk, dim=1, largest=False).values
    md = torch.as_tensor(max_dist, dtype=torch.float64, device=q.device).reshape(-1, 1)
    out[out > md * md] = float("inf")
    if limit is not None:
        out[torch.arange(k, device=q.device)[None, :] >= _dev(limit)[:, None]] = float("inf")
    return out


def exact(case, seed):
    """The squared distances; coordinates, ids and counts are the inputs' own values."""
    op = case["op"]
    if op in ("host_knn", "knn") and case["points"] * case["queries"] <= PAIRS:
        m, q = _cloud(case, seed)
        return None, _nearest(m, q, case["k"], _inf(case["max_dist"])).cpu(), None, None
    if op == "batch_knn" and case["points"] * case["queries"] / case["maps"] <= PAIRS:
        pts, q, qt, rng = _maps(case, seed)
        ks, md = _knn_mix(case, len(q), rng)
        d = torch.cat([_nearest(p, q[qt == i], case["k"], md[qt == i], ks[qt == i]) for i, p in enumerate(pts)])
        return None, d.cpu(), None, None
    return None
