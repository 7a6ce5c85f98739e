"""Spatial queries over points of one dim: the plain traversals (closest point,
and lists of 1, 2 or 4 entries) and the others give the oracle's results."""
import numpy as np
import pytest
import torch

import cudakdtree_amd as ck
import oracle as oc
from cudakdtree_amd import datagen
from tests.helpers import distribution
from tests.test_gpu_spatial import build_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dist", ["uniform", "ties", "gmm"])
@pytest.mark.parametrize("k", [0, 1, 2, 3, 4, 5, 8])
def test_lists(dist, k):
    coords = distribution(dist, 3001, 1, seed=k)
    lay, ref, t = build_both(coords)
    q = datagen.uniform(200, 1, k + 1) * np.float32(6.0 if dist == "ties" else 1.0)
    dq = torch.from_numpy(q).cuda()
    for m in (ck.STACK_BASED, ck.CCT):
        for lk in (ck.LIST_FIXED, ck.LIST_HEAP):
            for cutoff in (float("inf"), 0.01, float("nan")):
                if k:
                    got = ck.spatial_knn(t, dq, k, m, lk, cutoff)
                    want = oc.spatial_knn(m, lk, k, *ref, coords, lay, q, cutoff)
                else:
                    got = ck.spatial_fcp(t, dq, m, cutoff)
                    want = oc.spatial_fcp(m, *ref, coords, lay, q, cutoff)
                torch.cuda.synchronize()
                for a, b in zip(got, want):
                    assert np.array_equal(a.cpu().numpy().view(np.int32), b.view(np.int32))
    ck.free(t)
