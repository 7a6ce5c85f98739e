"""Spatial trees over extents whose centre is not strictly between their ends
as a float -- ends whose sum overflows, and infinite ones -- are the oracle's,
and so are queries over them."""
import numpy as np
import pytest
import torch

import cudakdtree_amd as ck
import oracle as oc
from cudakdtree_amd import datagen

pytestmark = pytest.mark.gpu


def _points(kind, n, D):
    u = datagen.uniform(n, D, n)
    r = np.random.RandomState(n).randint(0, 5, (n, D))
    inf = np.float32(np.inf)
    if kind == "sum overflows":
        u[:, 0] = np.float32(1.8e38) + np.float32(1.6e38) * u[:, 0]
    elif kind == "negative sum overflows":
        u = np.float32(-1.8e38) - np.float32(1.6e38) * u
    elif kind == "opposite infinities":
        u = np.where(r == 0, -inf, np.where(r == 1, inf, u))
    elif kind == "infinity in one dim":
        u[:, D - 1] = np.where(r[:, 0] < 3, inf, u[:, D - 1])
    elif kind == "minus infinity":
        u = np.where(r < 2, -inf, u)
    return np.ascontiguousarray(u, np.float32)


@pytest.mark.parametrize("n,leaf", [(9, 0), (9, 1), (2500, 1), (5000, 0), (100_001, 0)])
@pytest.mark.parametrize("kind", ["sum overflows", "negative sum overflows",
                                  "opposite infinities", "infinity in one dim",
                                  "minus infinity"])
def test_build_and_query(kind, n, leaf):
    for D in (1, 3):
        print(kind, n, leaf, D, flush=True)
        pts, lay = _points(kind, n, D), ck.float_points(D)
        ref = oc.spatial_build(pts, lay, leaf)
        t = ck.buildSpatialTree(torch.from_numpy(pts).cuda(), lay, leaf)
        assert t.num_nodes == len(ref[0])
        assert np.array_equal(t.nodes_numpy().view(np.uint8), ref[0].view(np.uint8))
        assert np.array_equal(t.prims_numpy(), ref[1])
        q = np.concatenate([pts[:70], datagen.uniform(60, D, 3)])
        dq = torch.from_numpy(q).cuda()
        for m in (ck.STACK_BASED, ck.CCT):
            ids, d2, _ = ck.spatial_knn(t, dq, 5, m, ck.LIST_FIXED, 0.3)
            want = oc.spatial_knn(m, ck.LIST_FIXED, 5, *ref, pts, lay, q, 0.3)
            torch.cuda.synchronize()
            assert np.array_equal(ids.cpu().numpy(), want[0])
            assert np.array_equal(d2.cpu().numpy().view(np.int32), want[1].view(np.int32))
        ck.free(t)
