"""knn_extract with an entry per lane: lists of 1 to 64 entries, so 64 lists
to one a wavefront, with counts of lists that leave a wave, a workgroup and
the last rank round unfilled; equal, empty and infinite entries; each output
left out.  Against a host sort of the keys (samples/mpiHugeQuery.cu:90-103)."""
import ctypes

import numpy as np
import pytest
import torch

import cudakdtree_amd as ck

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 2, 3, 8, 20, 33, 63, 64])
@pytest.mark.parametrize("nq", [1, 5, 64, 257, 3001])
def test_extract_sorts_each_list(k, nq):
    rng = np.random.default_rng(100 * k + nq)
    d2 = rng.choice(np.array([0.0, 0.25, 0.5, 2.0, np.inf], np.float32), (nq, k))
    ids = rng.permuted(np.tile(np.arange(k, dtype=np.int32), (nq, 1)), axis=1)
    ids[rng.random((nq, k)) < 0.2] = -1
    # empty entries of one list share one key
    keys = (d2.view(np.uint32).astype(np.uint64) << np.uint64(32)) | ids.view(np.uint32).astype(np.uint64)
    lists = torch.from_numpy(keys.view(np.int64)).cuda()
    want = np.sort(keys, axis=1)
    wid = (want & np.uint64(0xFFFFFFFF)).astype(np.uint32).view(np.int32)
    wd2 = (want >> np.uint64(32)).astype(np.uint32).view(np.float32)
    gid, gd2, _ = ck.knn_extract(lists)
    torch.cuda.synchronize()
    assert np.array_equal(gid.cpu().numpy(), wid)
    assert np.array_equal(gd2.cpu().numpy().view(np.uint32), wd2.view(np.uint32))
    for drop in (0, 1):
        out = torch.full((nq, k), 7, dtype=torch.int32, device="cuda")
        p = ctypes.c_void_p(out.data_ptr())
        rc = ck.lib().cukd_knn_extract(ctypes.c_void_p(lists.data_ptr()), nq, k,
                                       None if drop == 0 else p, p if drop == 0 else None, None,
                                       None)
        torch.cuda.synchronize()
        assert rc == ck.OK
        assert np.array_equal(out.cpu().numpy(), wd2.view(np.int32) if drop == 0 else wid)
