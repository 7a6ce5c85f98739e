"""The Morton launch order is a permutation, cell by cell, at the batch sizes
where its tiles change, for every dimension count and degenerate batches."""
import numpy as np
import pytest
import torch

import cudakdtree_amd as ck

pytestmark = pytest.mark.gpu


def _cells(q):
    D = q.shape[1]
    b = max(15 // D, 1)
    lo, hi = q.min(0).values, q.max(0).values
    w = hi - lo
    t = torch.where(w > 0, (q - lo) / w, torch.zeros_like(q))
    c = (t * (1 << b)).int().clamp_(0, (1 << b) - 1)
    code = torch.zeros(len(q), dtype=torch.int32, device=q.device)
    for d in range(D):
        for j in range(b):
            code |= ((c[:, d] >> j) & 1) << (j * D + d)
    return code


@pytest.mark.parametrize("nq", [1, 63, 4095, 4096, 4097, 1 << 18, (1 << 18) + 1, 1 << 20,
                                (1 << 20) + 1, 1 << 22])
def test_permutation_by_cells(nq):
    q = torch.from_numpy(np.random.RandomState(nq % 1000).rand(nq, 3).astype(np.float32)).cuda()
    o = ck.query_order(q).long()
    assert torch.equal(torch.sort(o).values, torch.arange(nq, device="cuda"))
    c = _cells(q)[o]
    assert (c[1:] >= c[:-1]).all()


@pytest.mark.parametrize("D", range(1, 9))
def test_dims_and_degenerate_batches(D):
    q = torch.rand((5001, D), device="cuda") * 7.0 - 3.0
    for x in (q, torch.zeros_like(q), torch.cat([q, q[:1] * 1e6])):
        o = ck.query_order(x).long()
        assert torch.equal(torch.sort(o).values, torch.arange(len(x), device="cuda"))
        c = _cells(x)[o]
        assert (c[1:] >= c[:-1]).all()
