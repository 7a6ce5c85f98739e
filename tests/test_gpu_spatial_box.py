"""Spatial-tree queries: register-list capacities, box pruning, the Morton
order of large batches and the 50-entry stack's overflow give the oracle's
results bit for bit (fcp.h:256-427, knn.h:566-752)."""
import numpy as np
import pytest
import torch

import cudakdtree_amd as ck
import oracle as oc
from cudakdtree_amd import datagen
from tests.helpers import distribution
from tests.test_gpu_spatial import build_both

pytestmark = pytest.mark.gpu

METHODS = (ck.STACK_BASED, ck.CCT)
LISTS = (ck.LIST_FIXED, ck.LIST_HEAP)


def _same(got, want):
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        g = g.cpu().numpy()
        assert np.array_equal(g.view(np.int32), w.view(np.int32))


def _check(coords, lay, ref, t, q, k, m, lk, cutoff):
    dq = torch.from_numpy(q).cuda()
    if k == 0:
        _same(ck.spatial_fcp(t, dq, m, cutoff), oc.spatial_fcp(m, *ref, coords, lay, q, cutoff))
    else:
        _same(ck.spatial_knn(t, dq, k, m, lk, cutoff),
              oc.spatial_knn(m, lk, k, *ref, coords, lay, q, cutoff))


@pytest.mark.parametrize("dist", ["uniform", "gmm", "ties", "plane"])
@pytest.mark.parametrize("k", [0, 3, 4, 5, 8, 9, 16, 17, 32, 33, 64])
def test_capacities_and_ties(dist, k):
    coords = distribution(dist, 4001, 3, seed=k)
    lay, ref, t = build_both(coords)
    q = datagen.uniform(130, 3, k + 1) * np.float32(6.0 if dist == "ties" else 1.0)
    for m in METHODS:
        for lk in LISTS:
            for cutoff in (float("inf"), 0.2):
                _check(coords, lay, ref, t, q, k, m, lk, cutoff)
    ck.free(t)


@pytest.mark.parametrize("D", [1, 2, 4, 6, 7, 8])
@pytest.mark.parametrize("leaf", [1, 0, 100])
def test_dims_and_leaf_sizes(D, leaf):
    coords = distribution("coarse", 1500, D, seed=D)
    lay, ref, t = build_both(coords, leaf)
    q = datagen.uniform(70, D, 5)
    for m in METHODS:
        for k in (0, 8):
            _check(coords, lay, ref, t, q, k, m, ck.LIST_FIXED, float("inf"))
    ck.free(t)


@pytest.mark.parametrize("m", METHODS)
def test_deep_tree_overflows_as_the_reference(m):
    """120 points at 2^-i: every split peels one off, so the first descent of
    an unbounded query near 0 pushes 50 far children."""
    coords = np.zeros((120, 3), np.float32)
    coords[:, 0] = np.float32(2.0) ** -np.arange(120, dtype=np.float32)
    lay, ref, t = build_both(coords, 1)
    q = np.concatenate([np.zeros((1, 3), np.float32), datagen.uniform(66, 3, 3)])
    for k in (0, 4):
        for cutoff in (float("inf"), 1e-3):
            _check(coords, lay, ref, t, q, k, m, ck.LIST_FIXED, cutoff)
    ck.free(t)


def test_degenerate_splits_are_not_pruned():
    """Clumps of equal points beyond the leaf size, and clumps one ulp wide:
    splits whose children lie on either side of the plane."""
    base = datagen.uniform(60, 3, 9)
    coords = np.repeat(base, 40, axis=0)
    coords[::3] = np.nextafter(coords[::3], np.float32(2.0))
    lay, ref, t = build_both(coords)
    q = np.concatenate([coords[::50], datagen.uniform(100, 3, 10)])
    for m in METHODS:
        for lk in LISTS:
            for k in (0, 4, 24):
                _check(coords, lay, ref, t, q, k, m, lk, float("inf"))
    ck.free(t)


@pytest.mark.parametrize("n,nq", [(400_000, 1 << 18), (20_000, 1 << 19)])
def test_large_batches_equal_small_ones(n, nq):
    """At and above the sizes where batches are Morton-ordered (and where a
    small tree's closest points take the plain traversal), results equal
    those of the same queries in small batches, counted or not."""
    pts = torch.from_numpy(datagen.uniform(n, 3, 11)).cuda()
    t = ck.buildSpatialTree(pts, ck.float_points(3))
    q = torch.from_numpy(datagen.uniform(nq, 3, 12)).cuda()
    part = 1 << 15
    for m in METHODS:
        for k, lk in ((0, 0), (8, ck.LIST_FIXED), (8, ck.LIST_HEAP)):
            def run(x):
                return (ck.spatial_knn(t, x, k, m, lk, 0.1) if k else ck.spatial_fcp(t, x, m, 0.1))
            want = [torch.cat(c) for c in zip(*(run(q[a:a + part]) for a in range(0, nq, part)))]
            for a, b in zip(run(q), want):
                assert torch.equal(a, b)
            counter = torch.zeros(1, dtype=torch.int64, device="cuda")
            ck.set_traversal_stats(counter)
            try:
                got = run(q)
                torch.cuda.synchronize()
            finally:
                ck.set_traversal_stats(None)
            assert int(counter.item()) >= nq
            for a, b in zip(got, want):
                assert torch.equal(a, b)
    ck.free(t)


@pytest.mark.parametrize("m", METHODS)
def test_nan_cutoff(m):
    coords = distribution("uniform", 900, 3, seed=13)
    lay, ref, t = build_both(coords)
    q = datagen.uniform(40, 3, 14)
    for k in (0, 8):
        _check(coords, lay, ref, t, q, k, m, ck.LIST_FIXED, float("nan"))
    ck.free(t)
