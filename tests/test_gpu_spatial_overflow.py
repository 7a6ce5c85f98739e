"""kNN queries that overflow the reference's 50-entry traversal stack, through
the C ABI without an array for the radii: every row is the oracle's."""
import ctypes

import numpy as np
import pytest
import torch

import cudakdtree_amd as ck
import oracle as oc
from cudakdtree_amd import datagen
from tests.test_gpu_spatial import build_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("list_kind", [ck.LIST_FIXED, ck.LIST_HEAP])
@pytest.mark.parametrize("m", [ck.STACK_BASED, ck.CCT])
def test_rows_without_radii(m, list_kind):
    coords = np.zeros((120, 3), np.float32)
    coords[:, 0] = np.float32(2.0) ** -np.arange(120, dtype=np.float32)
    lay, ref, t = build_both(coords, 1)
    nq, k = 500, 4
    q = datagen.uniform(nq, 3, 3)
    q[40::9] = 0
    want = oc.spatial_knn(m, list_kind, k, *ref, coords, lay, q, float("inf"))
    if m == ck.STACK_BASED:
        assert want[2][49] == -1 and want[2][0] != -1
    dq = torch.from_numpy(q).cuda()
    ids = torch.full((nq, k), -7, dtype=torch.int32, device="cuda")
    d2 = torch.full((nq, k), -7.0, dtype=torch.float32, device="cuda")
    rc = ck.lib().cukd_spatial_knn(
        m, list_kind, k, ctypes.byref(t.raw), ctypes.byref(lay), ctypes.c_void_p(dq.data_ptr()),
        nq, float("inf"), ctypes.c_void_p(ids.data_ptr()), ctypes.c_void_p(d2.data_ptr()), None,
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, ck.lib().cukd_last_error()
    torch.cuda.synchronize()
    assert np.array_equal(ids.cpu().numpy(), want[0])
    assert np.array_equal(d2.cpu().numpy().view(np.int32), want[1].view(np.int32))
    ck.free(t)
