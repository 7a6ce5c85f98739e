"""Top levels built by one workgroup per subtree (subtrees of at most 16384
elements) equal the oracle's tree byte for byte: sizes where a level's
largest subtree is just at, below or above that bound, coordinates shared by
more elements than are ranked at once, extreme keys, element sizes of each
copy path, and forests that mix both kinds of level."""
import numpy as np
import pytest
import torch

import cudakdtree_amd as ck
import oracle as oc
from cudakdtree_amd import datagen
from tests.helpers import distribution, layout_for, make_elements

pytestmark = pytest.mark.gpu


def _check(elems, lay):
    ref, rbox = oc.build_host(elems, lay, want_bounds=True)
    d = torch.from_numpy(np.ascontiguousarray(elems).copy()).cuda()
    b = ck.bounds_tensor(lay)
    ck.buildTree(d, lay, b)
    torch.cuda.synchronize()
    got = d.cpu().numpy()
    assert np.array_equal(got.view(np.uint8), ref.view(np.uint8))


@pytest.mark.parametrize("n", [511, 512, 1023, 1024, 2049, 16383, 16384, 16385, 32767, 32768,
                               32769, 65535, 65537, 100_000])
@pytest.mark.parametrize("kind", ["float", "explicit"])
def test_sizes(n, kind):
    c = distribution("coarse", n, 3, seed=n)
    lay = layout_for(kind, 3)
    _check(make_elements(c, lay) if kind != "float" else c, lay)


@pytest.mark.parametrize("equal", [255, 256, 257, 258, 3000, 16384])
@pytest.mark.parametrize("kind", ["float", "explicit"])
def test_shared_coordinates(equal, kind):
    """'equal' elements share x around the median, the first 'equal' / 2 of
    them y too, and some are equal altogether."""
    n = 16384
    c = datagen.uniform(n, 3, equal)
    a = (n - equal) // 2
    order = np.argsort(c[:, 0], kind="stable")
    c = c[order]
    c[a:a + equal, 0] = c[min(a + equal // 2, n - 1), 0]
    c[a:a + equal // 2, 1] = 0.5
    c[a:a + equal // 4, 2] = 0.25
    c = c[np.random.RandomState(equal).permutation(n)]
    lay = layout_for(kind, 3)
    _check(make_elements(c, lay) if kind != "float" else np.ascontiguousarray(c), lay)


@pytest.mark.parametrize("D", [1, 2, 3, 4, 5, 8])
def test_dims_and_strides(D):
    for kind in ("float", "explicit"):
        c = distribution("gmm", 9001, D, seed=D)
        lay = layout_for(kind, D)
        _check(make_elements(c, lay) if kind != "float" else c, lay)


def test_extreme_keys():
    r = np.random.RandomState(3)
    c = r.randint(-2**31, 2**31, size=(12000, 3), dtype=np.int64).astype(np.int32)
    c[::7] = 2**31 - 1
    c[3::7, 0] = -2**31
    _check(c, ck.int_points(3))
    f = datagen.uniform(12000, 3, 4) - np.float32(0.5)
    f[::5] *= np.float32(1e38)
    f[1::11] = np.inf
    f[2::11, 1] = -np.inf
    f[3::13] = -0.0
    _check(f, ck.float_points(3))


def test_forest_of_both_kinds():
    sizes = [3, 600, 40_000, 16384, 0, 70_001, 9000, 1200]
    off = np.concatenate([[0], np.cumsum(sizes)])
    c = distribution("coarse", int(off[-1]), 3, seed=5)
    lay = ck.float_points(3)
    d = torch.from_numpy(c.copy()).cuda()
    for picked in (range(len(sizes)), [1, 3, 6, 7]):  # with and without the large trees
        o = np.concatenate([[0], np.cumsum([sizes[i] for i in picked])])
        src = np.concatenate([c[off[i]:off[i + 1]] for i in picked])
        d = torch.from_numpy(src.copy()).cuda()
        f = ck.Forest(o, lay)
        f.build(d)
        torch.cuda.synchronize()
        got = d.cpu().numpy()
        for a, b in zip(o, o[1:]):
            if b > a:
                ref, _ = oc.build_host(src[a:b], lay, want_bounds=True)
                assert np.array_equal(got[a:b], ref)
        f.close()
