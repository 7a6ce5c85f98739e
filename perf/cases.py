"""The timed workloads of this framework: what its users have it do.

Every case is one call sequence through the package's public entry points
(build a tree, query it, build and query a forest, ...) at a stated size.
``listed()`` names the standing workloads, ``draw(rng)`` gives others of the
same ranges, ``prepare`` / ``run`` carry one out, ``work`` counts the bytes
and operations it cannot do without, and ``exact`` gives its results in 64
bits where a brute force can.

Kinds and their ranges:
  build     one left-balanced tree over n points: 500 .. 10M (tree-layout
            builders: .. 1M), float or int, 2 .. 4 dims, the default, bitonic
            and in-place builders, payload structs with a split-dim field
  query     FCP or kNN of nq queries over one built tree: n 1000 .. 10M,
            nq 100 .. 1M, k 1 .. 64, fixed and heap lists, the three
            traversals, Morton-ordered launches or not, with and without a
            cutoff radius
  rounds    multi-round kNN over shards, then the extraction
  forest    many trees built and queried together
  sbuild    spatial k-d tree build
  squery    spatial k-d tree queries
"""
import math

import numpy as np
import torch

import cudakdtree_amd as ck

DEV = "cuda:0"
TRAV = {"stack": ck.STACK_BASED, "free": ck.STACK_FREE, "cct": ck.CCT}
LIST = {"fixed": ck.LIST_FIXED, "heap": ck.LIST_HEAP}
BUILDER = {"default": ck.BUILDER_ID_DEFAULT, "bitonic": ck.BUILDER_ID_BITONIC,
           "inplace": ck.BUILDER_ID_INPLACE}


def listed():
    return [
        # the smallest build: one object's samples, rebuilt every frame;
        # launches and host latency are all of it
        {"name": "build-2k", "kind": "build", "n": 2000, "dims": 3, "scalar": "f32",
         "payload": False, "builder": "default", "dist": "uniform"},
        # the plain-method size of the benchmark (one scan or mesh)
        {"name": "build-100k", "kind": "build", "n": 100_000, "dims": 3, "scalar": "f32",
         "payload": False, "builder": "default", "dist": "uniform"},
        # the benchmark's headline build
        {"name": "build-10m", "kind": "build", "n": 10_000_000, "dims": 3, "scalar": "f32",
         "payload": False, "builder": "default", "dist": "uniform"},
        # payload structs with a split-dim field over clustered points
        # (photon maps); an odd size
        {"name": "build-payload-1.5m", "kind": "build", "n": 1_500_007, "dims": 3,
         "scalar": "f32", "payload": True, "builder": "default", "dist": "clustered"},
        # the builder that needs no temporary memory, at an odd size
        {"name": "build-inplace-1m", "kind": "build", "n": 1_000_003, "dims": 3,
         "scalar": "f32", "payload": False, "builder": "inplace", "dist": "uniform"},
        # the benchmark's headline query: kNN-8, Morton-ordered launch
        {"name": "knn8-1m-of-10m", "kind": "query", "n": 10_000_000, "nq": 1_000_000, "dims": 3,
         "k": 8, "list": "fixed", "trav": "stack", "sort": True, "cutoff": 0.0,
         "dist": "uniform"},
        # closest point of every vertex of one mesh in another, as given
        {"name": "fcp-100k", "kind": "query", "n": 100_000, "nq": 100_000, "dims": 3, "k": 0,
         "list": "fixed", "trav": "stack", "sort": False, "cutoff": 0.0, "dist": "uniform"},
        # density estimation (photon gathering): heap list of 50 over
        # clustered points, closest-corner traversal
        {"name": "knn50-heap-cct", "kind": "query", "n": 1_000_000, "nq": 200_000, "dims": 3,
         "k": 50, "list": "heap", "trav": "cct", "sort": True, "cutoff": 0.0,
         "dist": "clustered"},
        # one GPU's share of a sharded kNN: 4 visiting shards, lists of 20
        {"name": "rounds-k20", "kind": "rounds", "n": 2_000_000, "nq": 250_000, "dims": 3,
         "k": 20, "shards": 4, "sort": True},
        # many independent objects at once (the benchmark's forest, fewer
        # trees): build and kNN-4 in each
        {"name": "forest-512", "kind": "forest", "trees": 512, "lo": 64, "hi": 131_072, "k": 4},
        # spatial tree build, 1% duplicate points
        {"name": "spatial-build-1m", "kind": "sbuild", "n": 1_000_000, "dims": 4,
         "scalar": "f32"},
        # the benchmark's spatial query: kNN-16 within 0.05, half the
        # queries beside data points and half anywhere
        {"name": "spatial-knn16", "kind": "squery", "n": 4_000_000, "nq": 2_000_000, "dims": 4,
         "k": 16, "list": "fixed", "trav": "stack", "radius": 0.05},
    ]


def _log(rng, lo, hi):
    """log-uniform in [lo, hi], odd or even alike"""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["build", "build", "build", "query", "query", "query", "query", "rounds",
                       "forest", "sbuild", "squery"])
    if kind == "build":
        builder = rng.choice(["default", "default", "default", "bitonic", "inplace"])
        payload = rng.random() < 0.3
        return {"kind": kind,
                "n": _log(rng, 500, 10_000_000 if builder == "default" else 1_000_000),
                "dims": 3 if payload else rng.choice([2, 3, 3, 4]),
                "scalar": "f32" if payload else rng.choice(["f32", "f32", "f32", "i32"]),
                "payload": payload, "builder": builder,
                "dist": rng.choice(["uniform", "uniform", "clustered", "grid"])}
    if kind == "query":
        k = rng.choice([0, 1, 4, 8, 8, 16, rng.randint(2, 32), rng.randint(33, 64)])
        most = 1_000_000 if k <= 16 else 200_000
        return {"kind": kind, "n": _log(rng, 1000, 10_000_000), "nq": _log(rng, 100, most),
                "dims": rng.choice([2, 3, 3, 3, 4]), "k": k,
                "list": rng.choice(["fixed", "fixed", "heap"]),
                "trav": rng.choice(["stack", "stack", "free", "cct"]),
                "sort": rng.random() < 0.7, "cutoff": rng.choice([0.0, 0.0, 0.05]),
                "dist": rng.choice(["uniform", "uniform", "clustered", "grid"])}
    if kind == "rounds":
        return {"kind": kind, "n": _log(rng, 10_000, 2_000_000), "nq": _log(rng, 1000, 250_000),
                "dims": 3, "k": rng.randint(4, 32), "shards": rng.choice([2, 4]),
                "sort": rng.random() < 0.7}
    if kind == "forest":
        return {"kind": kind, "trees": _log(rng, 16, 512), "lo": 64,
                "hi": _log(rng, 4096, 131_072), "k": rng.choice([0, 1, 4, 8])}
    if kind == "sbuild":
        return {"kind": kind, "n": _log(rng, 1000, 1_000_000), "dims": rng.choice([3, 4]),
                "scalar": rng.choice(["f32", "f32", "i32"])}
    return {"kind": kind, "n": _log(rng, 10_000, 4_000_000), "nq": _log(rng, 1000, 2_000_000),
            "dims": 4, "k": rng.choice([0, 4, 8, 16]), "list": rng.choice(["fixed", "heap"]),
            "trav": rng.choice(["stack", "stack", "cct"]), "radius": 0.05}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _mixture(n, dims, g, centres):
    which = torch.randint(0, centres.shape[0], (n,), generator=g, device=DEV)
    return centres[which] + 0.01 * torch.randn((n, dims), generator=g, device=DEV)


def _points(n, dims, dist, g, centres=None):
    """float32 [n, dims] in about [0, 1): uniform, 64 Gaussian clusters, or
    uniform on a grid of 4096 steps (measured coordinates, with ties)"""
    if dist == "clustered":
        return _mixture(n, dims, g, centres)
    if dist == "grid":
        return torch.randint(0, 4096, (n, dims), generator=g, device=DEV).float() / 4096.0
    return torch.rand((n, dims), generator=g, device=DEV)


def _centres(dims, g):
    return torch.rand((64, dims), generator=g, device=DEV)


def _query_inputs(case, seed):
    g = _gen(seed)
    c = _centres(case["dims"], g)
    pts = _points(case["n"], case["dims"], case.get("dist", "uniform"), g, c)
    # queries follow the points' own distribution; never on the grid itself
    dist = "clustered" if case.get("dist") == "clustered" else "uniform"
    return pts, _points(case["nq"], case["dims"], dist, g, c)


def _spatial_points(n, dims, g):
    """uniform in [-1, 1), the last 1% copies of others"""
    pts = torch.rand((n, dims), generator=g, device=DEV) * 2.0 - 1.0
    m = n // 100
    if m:
        pts[n - m:] = pts[torch.randint(0, n - m, (m,), generator=g, device=DEV)]
    return pts


def _forest_sizes(case, seed):
    r = np.random.RandomState(seed % (1 << 32))
    lo, hi = math.log(case["lo"]), math.log(case["hi"])
    # the sizes' quantiles are fixed, their order is the seed's: every seed
    # gives about the same amount of work
    u = (r.permutation(case["trees"]) + 0.5) / case["trees"]
    return np.exp(lo + u * (hi - lo)).astype(np.int64)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "build":
        g = _gen(seed)
        c = _centres(case["dims"], g)
        if case["scalar"] == "i32":
            pts = torch.randint(0, 1 << 20, (case["n"], case["dims"]), generator=g, device=DEV,
                                dtype=torch.int32)
            lay = ck.int_points(case["dims"])
        else:
            pts = _points(case["n"], case["dims"], case["dist"], g, c)
            lay = ck.float_points(case["dims"])
        if case["payload"]:
            rows = torch.zeros((case["n"], case["dims"] + 2), dtype=torch.int32, device=DEV)
            rows[:, :case["dims"]] = pts.view(torch.int32)
            rows[:, case["dims"]] = torch.arange(case["n"], dtype=torch.int32, device=DEV)
            pts = rows
            lay = ck.point_plus_payload(case["dims"], explicit_dim=True)
        s.update(points=pts, layout=lay, box=ck.bounds_tensor(lay, DEV))
    elif kind == "query":
        pts, q = _query_inputs(case, seed)
        lay = ck.float_points(case["dims"])
        box = ck.bounds_tensor(lay, DEV)
        ck.buildTree(pts, lay, box)
        s.update(tree=pts, queries=q, layout=lay, box=box)
    elif kind == "rounds":
        pts, q = _query_inputs(case, seed)
        lay = ck.float_points(case["dims"])
        off = [i * case["n"] // case["shards"] for i in range(case["shards"] + 1)]
        shards = [pts[a:b].clone() for a, b in zip(off, off[1:])]
        for t in shards:
            ck.buildTree(t, lay)
        s.update(shards=shards, offsets=off, queries=q, layout=lay,
                 lists=ck.knn_lists(case["nq"], case["k"], DEV))
    elif kind == "forest":
        sizes = _forest_sizes(case, seed)
        T = len(sizes)
        off = np.concatenate([[0], np.cumsum(sizes)])
        qoff = np.concatenate([[0], np.cumsum(sizes // 2)])
        g = _gen(seed)
        lo = torch.rand((T, 3), generator=g, device=DEV) * 100.0
        ext = torch.rand((T, 3), generator=g, device=DEV) * 10.0 + 0.1
        tid = torch.arange(T, device=DEV)
        own = torch.repeat_interleave(tid, torch.from_numpy(sizes).to(DEV))
        qown = torch.repeat_interleave(tid, torch.from_numpy(sizes // 2).to(DEV))
        pts = torch.rand((int(off[-1]), 3), generator=g, device=DEV) * ext[own] + lo[own]
        q = torch.rand((int(qoff[-1]), 3), generator=g, device=DEV) * ext[qown] + lo[qown]
        lay = ck.float_points(3)
        s.update(points=pts, queries=q, forest=ck.Forest(off, lay),
                 seg_off=torch.from_numpy(qoff.astype(np.int32)).to(DEV),
                 seg_tree=torch.arange(T, dtype=torch.int32, device=DEV))
    elif kind == "sbuild":
        g = _gen(seed)
        if case["scalar"] == "i32":
            pts = ((_spatial_points(case["n"], case["dims"], g) + 1.0) * (1 << 19)).int()
            lay = ck.int_points(case["dims"])
        else:
            pts = _spatial_points(case["n"], case["dims"], g)
            lay = ck.float_points(case["dims"])
        # the program's own node buffer: 3 words a node, at most 2n + 2 nodes
        s.update(points=pts, layout=lay, tree=None,
                 nodes=torch.zeros(3 * (2 * case["n"] + 2), dtype=torch.int32, device=DEV))
    else:
        g = _gen(seed)
        pts = _spatial_points(case["n"], case["dims"], g)
        lay = ck.float_points(case["dims"])
        half = case["nq"] // 2
        near = pts[torch.randint(0, case["n"], (half,), generator=g, device=DEV)]
        near = near + 0.001 * torch.randn(near.shape, generator=g, device=DEV)
        far = torch.rand((case["nq"] - half, case["dims"]), generator=g, device=DEV) * 2.0 - 1.0
        s.update(tree=_Spatial(pts, lay), queries=torch.cat([near, far]))
    return s


class _Spatial:
    """A spatial tree that is given back with its last reference."""

    def __init__(self, points, layout):
        self.tree = ck.buildSpatialTree(points, layout)

    def __del__(self):
        ck.free(self.tree)


class _Words:
    """Device memory as int32 words, for torch.as_tensor."""

    def __init__(self, ptr, words, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (words,), "typestr": "<i4",
                                         "data": (int(ptr), False), "version": 2}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "build":
        # the build is in place: the program keeps its points as they were
        tree = s["points"].clone()
        # a split-dim field needs the world bounds; others do not ask for them
        box = s["box"] if case["payload"] else None
        ck.build_tree(tree, s["layout"], BUILDER[case["builder"]], box)
        return [tree, box] if case["payload"] else [tree]
    if kind == "query":
        flags = ck.QUERY_SORT if case["sort"] else 0
        cut = case["cutoff"] or math.inf
        if case["k"] == 0:
            return ck.fcp(s["tree"], s["layout"], s["queries"], TRAV[case["trav"]], cutoff=cut,
                          world_bounds=s["box"], flags=flags)
        return ck.knn(s["tree"], s["layout"], s["queries"], case["k"], TRAV[case["trav"]],
                      LIST[case["list"]], cutoff=cut, world_bounds=s["box"], flags=flags)
    if kind == "rounds":
        flags = ck.QUERY_SORT if case["sort"] else 0
        for i, t in enumerate(s["shards"]):
            ck.knn_accumulate(t, s["layout"], s["queries"], s["lists"], init=(i == 0),
                              id_offset=s["offsets"][i], flags=flags)
        return ck.knn_extract(s["lists"])
    if kind == "forest":
        trees = s["points"].clone()
        s["forest"].build(trees)
        if case["k"] == 0:
            r = s["forest"].fcp(trees, s["queries"], s["seg_off"], s["seg_tree"])
        else:
            r = s["forest"].knn(trees, s["queries"], case["k"], s["seg_off"], s["seg_tree"])
        return [trees, *r]
    if kind == "sbuild":
        # the program holds one tree and replaces it
        s["tree"] = None
        t = s["tree"] = _Spatial(s["points"], s["layout"])
        raw = t.tree.raw
        words = raw.num_nodes * 3
        s["nodes"][:words].copy_(torch.as_tensor(_Words(raw.nodes, words, t), device=DEV))
        return {"nodes": s["nodes"],
                "prims": torch.as_tensor(_Words(raw.prim_ids, raw.num_prims, t), device=DEV),
                "bounds": [float(b) for b in t.tree.bounds], "num_nodes": raw.num_nodes}
    t = s["tree"].tree
    if case["k"] == 0:
        return ck.spatial_fcp(t, s["queries"], TRAV[case["trav"]], cutoff=case["radius"])
    return ck.spatial_knn(t, s["queries"], case["k"], TRAV[case["trav"]], LIST[case["list"]],
                          cutoff=case["radius"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    """Inputs read once and results written once; a comparison per tree level
    and point for a build, k distances per query for a query."""
    kind = case["kind"]
    if kind in ("build", "sbuild"):
        stride = 4 * (case["dims"] + (2 if case.get("payload") else 0))
        n = case["n"]
        out = n * stride if kind == "build" else n * 4 + 12 * (n // 4)
        return {"bytes": n * stride + out, "flops": n * math.log2(n)}
    if kind == "forest":
        n = int(_forest_sizes(case, 0).sum())
        nq = n // 2
        w = max(1, case["k"])
        return {"bytes": 24 * n + nq * (12 + 8 * w), "flops": n * 16 + nq * w * 8}
    w = max(1, case["k"])
    d = case["dims"]
    out = 8 * w + (4 if case["k"] else 0)
    return {"bytes": case["n"] * 4 * d + case["nq"] * (4 * d + out),
            "flops": case["nq"] * w * (3 * d - 1)}


# ---------------------------------------------------------------------------
# results in 64 bits
# ---------------------------------------------------------------------------

def exact(case, seed):
    """Squared distances by brute force in float64, for queries small enough.
    Ids are whole numbers, and a heap list's order is the order of its
    heap: neither has a value here."""
    if case["kind"] == "query":
        pts, q = _query_inputs(case, seed)
        cut = float(np.float32(case["cutoff"])) or math.inf
    elif case["kind"] == "rounds":
        pts, q = _query_inputs(case, seed)
        cut = math.inf
    else:
        return None
    k = max(1, case["k"])
    pairs = case["n"] * case["nq"]
    if pairs > (2e10 if case["k"] == 0 else 2e9) or k > case["n"]:
        return None
    p = pts.double()
    best = torch.empty((case["nq"], k), dtype=torch.float64, device=DEV)
    step = max(1, int(1e8) // case["n"])
    for a in range(0, case["nq"], step):
        b = q[a:a + step].double()
        d2 = torch.zeros((b.shape[0], case["n"]), dtype=torch.float64, device=DEV)
        for d in range(case["dims"]):
            d2 += (b[:, d, None] - p[None, :, d]).square_()
        if k == 1:
            best[a:a + step, 0] = d2.min(dim=1).values
        else:
            best[a:a + step] = torch.topk(d2, k, dim=1, largest=False, sorted=True).values
    best.clamp_(max=cut * cut)
    if case["kind"] == "rounds":
        return (None, best, best[:, -1].sqrt())
    if case["k"] == 0:
        return (None, best[:, 0])
    return (None, best if case["list"] == "fixed" else None, best[:, -1].clone())
