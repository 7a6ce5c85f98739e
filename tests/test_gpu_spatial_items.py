"""The two-phase spatial build (rounds over large nodes, then one workgroup
per node of at most 2048 points) equals the oracle's tree byte for byte at
the edges of its range: sizes around 2048 and its multiples, leaf
thresholds from 1 to beyond 2048, every dimension count, skewed and
duplicated points, and trees too deep for its level table."""
import numpy as np
import pytest
import torch

import cudakdtree_amd as ck
import oracle as oc
from cudakdtree_amd import datagen
from tests.helpers import distribution

pytestmark = pytest.mark.gpu


def _check(coords, lay, leaf):
    rn, rp, rb = oc.spatial_build(coords, lay, leaf)
    t = ck.buildSpatialTree(torch.from_numpy(np.ascontiguousarray(coords)).cuda(), lay, leaf)
    assert t.num_nodes == len(rn)
    assert np.array_equal(t.nodes_numpy().view(np.uint8), rn.view(np.uint8))
    assert np.array_equal(t.prims_numpy(), rp)
    assert np.array_equal(np.array(t.bounds, lay.scalar_dtype).view(np.int32),
                          np.asarray(rb).view(np.int32))
    ck.free(t)


@pytest.mark.parametrize("n", [1, 2, 9, 2047, 2048, 2049, 4096, 4097, 6143, 20000, 70001])
@pytest.mark.parametrize("dist", ["uniform", "gmm", "ties", "signed_zero"])
def test_sizes(n, dist):
    _check(distribution(dist, n, 3, seed=n), ck.float_points(3), 0)


@pytest.mark.parametrize("leaf", [1, 2, 7, 64, 2047, 2048, 2049, 5000, 65535])
@pytest.mark.parametrize("dist", ["uniform", "ties", "coarse"])
def test_leaf_thresholds(leaf, dist):
    _check(distribution(dist, 12001, 3, seed=leaf), ck.float_points(3), leaf)


@pytest.mark.parametrize("D", range(1, 9))
@pytest.mark.parametrize("leaf", [0, 1])
def test_dims_and_scalars(D, leaf):
    _check(distribution("gmm", 9000, D, seed=D), ck.float_points(D), leaf)
    _check(distribution("uniform", 9000, D, seed=D, scalar_float=False), ck.int_points(D), leaf)


def test_skewed_points():
    """Half the points in a cube of 1e-4, whose node stays open long after
    the others; and every point in one place but a few."""
    c = datagen.uniform(30000, 3, 5)
    c[::2] = c[::2] * np.float32(1e-4) + np.float32(0.3)
    _check(c, ck.float_points(3), 0)
    d = np.full((9000, 3), 0.5, np.float32)
    d[::1000] = datagen.uniform(9, 3, 6)
    _check(d, ck.float_points(3), 0)


@pytest.mark.parametrize("levels", [40, 60, 61, 62, 63, 64, 66, 100])
@pytest.mark.parametrize("clump", [1, 3000])
def test_deep_trees(levels, clump):
    """One point (or a clump) per binary octave: a split peels one off, in the
    items or, with clumps, among the large nodes."""
    x = np.float32(2.0) ** -np.arange(levels, dtype=np.float32)
    c = np.zeros((levels * clump, 3), np.float32)
    c[:, 0] = np.repeat(x, clump)
    _check(c, ck.float_points(3), 1 if clump == 1 else clump)


def test_payload_stride():
    lay = ck.point_plus_payload(3)
    rows = np.zeros((5000, 5), np.float32)
    rows[:, :3] = distribution("gmm", 5000, 3, seed=8)
    rows[:, 3] = np.arange(5000)
    _check(rows, lay, 0)
