"""Rows of kNN results are written 16 bytes at a time wherever they start: any k
and any word offset of the output arrays gives the results of aligned rows of
64 entries, and nothing beside the rows is touched."""
import ctypes

import numpy as np
import pytest
import torch

import cudakdtree_amd as ck
import oracle as oc
from cudakdtree_amd import datagen

pytestmark = pytest.mark.gpu

KS = [1, 2, 3, 4, 5, 6, 7, 8, 9, 11, 12, 16, 17, 20, 23, 31, 33, 34, 47, 50, 61, 63, 64]


def _rows(nq, k, off, fill):
    buf = torch.full((nq * k + 8,), fill, dtype=torch.int32, device="cuda")
    return buf, ctypes.c_void_p(buf.data_ptr() + 4 * off)


@pytest.mark.parametrize("off", [0, 1, 2, 3])
@pytest.mark.parametrize("list_kind", [ck.LIST_FIXED, ck.LIST_HEAP])
@pytest.mark.parametrize("kind", ["balanced", "spatial"])
def test_any_row(kind, list_kind, off):
    n, nq = 3000, 130
    lay = ck.float_points(3)
    pts, q = datagen.uniform(n, 3, 1), datagen.uniform(nq, 3, 2)
    dq = torch.from_numpy(q).cuda()
    L = ck.lib()
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    if kind == "balanced":
        tree, _ = oc.build_host(pts, lay)
        dt = torch.from_numpy(tree).cuda()
    else:
        ref = oc.spatial_build(pts, lay, 0)
        t = ck.buildSpatialTree(torch.from_numpy(pts).cuda(), lay)
    for k in KS:
        ibuf, ids = _rows(nq, k, off, -77)
        dbuf, d2 = _rows(nq, k, off, -77)
        tail = (dq.data_ptr(), nq, 0.2, ids, d2, None)
        if kind == "balanced":
            rc = L.cukd_knn(ck.STACK_BASED, list_kind, k, ctypes.c_void_p(dt.data_ptr()), n,
                            ctypes.byref(lay), None, *tail, 0, stream, None)
            want = oc.knn(oc.STACK_BASED, list_kind, k, tree, lay, q, cutoff=0.2)
        else:
            rc = L.cukd_spatial_knn(ck.STACK_BASED, list_kind, k, ctypes.byref(t.raw),
                                    ctypes.byref(lay), *tail, stream)
            want = oc.spatial_knn(oc.STACK_BASED, list_kind, k, *ref, pts, lay, q, 0.2)
        assert rc == 0, L.cukd_last_error()
        torch.cuda.synchronize()
        for buf, w in ((ibuf, want[0]), (dbuf, want[1])):
            got = buf.cpu().numpy()
            assert np.array_equal(got[off:off + nq * k], w.view(np.int32).reshape(-1)), k
            assert (got[:off] == -77).all() and (got[off + nq * k:] == -77).all(), k
    if kind == "spatial":
        ck.free(t)
