"""The box-pruned batch kernel (the default launch over round-robin trees)
returns the oracle's results bit for bit at the edges of its register-list
capacities, for every traversal, list kind and tie pattern, and agrees with
the one-query-per-lane traversal on inputs the oracle's brute force does not
cover (NaN, infinite and far queries, unaligned result rows)."""
import numpy as np
import pytest
import torch

import cudakdtree_amd as ck
from cudakdtree_amd import datagen
from tests.helpers import distribution
from tests.test_gpu_query import METHODS, _setup, check_fcp, check_knn

pytestmark = pytest.mark.gpu

ONE = ck.QUERY_ONE_PER_LANE
LISTS = (ck.LIST_FIXED, ck.LIST_HEAP)


@pytest.mark.parametrize("k", [1, 3, 4, 7, 9, 15, 17, 23, 24, 25, 31, 33, 47, 49, 63, 64])
@pytest.mark.parametrize("dist", ["uniform", "gmm", "ties", "coarse"])
def test_capacity_edges(k, dist):
    s = _setup(distribution(dist, 6007, 3, seed=k))
    q = datagen.uniform(197, 3, k + 7) * np.float32(6.0 if dist == "ties" else 1.0)
    check_knn(*s, q, k, float("inf"))
    check_knn(*s, q, k, 0.11)


@pytest.mark.parametrize("D", [1, 2, 4, 5, 7])
@pytest.mark.parametrize("n", [1, 2, 7, 8, 64, 1000])
def test_dims_and_small_trees(D, n):
    s = _setup(distribution("coarse", n, D, seed=D + n))
    q = datagen.uniform(65, D, 3)
    check_knn(*s, q, 8, float("inf"))
    check_fcp(*s, q, float("inf"))


def _bits(t):
    return t.view(torch.int32) if t.dtype == torch.float32 else t


def _agree(s, dq, k, lk, m, cutoff=float("inf")):
    lay, _, _, dt, db = s
    a = ck.knn(dt, lay, dq, k, m, lk, cutoff, db)
    b = ck.knn(dt, lay, dq, k, m, lk, cutoff, db, flags=ONE)
    for x, y in zip(a, b):
        assert torch.equal(_bits(x), _bits(y)), (m, lk, k)


@pytest.mark.parametrize("m", METHODS)
@pytest.mark.parametrize("lk", LISTS)
def test_special_values_agree_with_one_per_lane(m, lk):
    pts = distribution("gmm", 5000, 3, seed=4)
    pts[::97] = np.inf
    pts[5::89, 1] = np.float32(1e30)  # squares overflow
    s = _setup(pts)
    q = datagen.uniform(640, 3, 5)
    q[::5] *= np.float32(1e4)
    q[1::7, 0] = np.inf
    q[2::7, 1] = -np.inf
    q[3::7, 2] = np.nan
    q[4::11] = np.float32(3e38)
    dq = torch.from_numpy(q).cuda()
    for k in (4, 20):
        for cutoff in (float("inf"), 0.5, 0.0, float("nan")):
            _agree(s, dq, k, lk, m, cutoff)


@pytest.mark.parametrize("shift", [1, 2, 3])
def test_unaligned_result_rows(shift):
    s = _setup(distribution("uniform", 3000, 3, seed=6))
    lay, _, _, dt, db = s
    dq = torch.from_numpy(datagen.uniform(100, 3, 7)).cuda()
    for k, lk in ((8, ck.LIST_FIXED), (12, ck.LIST_HEAP)):
        want = ck.knn(dt, lay, dq, k, list_kind=lk, world_bounds=db)
        ids = torch.full((100 * k + shift,), -7, dtype=torch.int32, device="cuda")
        d2 = torch.full((100 * k + shift,), -7.0, device="cuda")
        r = torch.empty(100, device="cuda")
        ck.knn(dt, lay, dq, k, list_kind=lk, world_bounds=db, out=(ids[shift:], d2[shift:], r))
        assert torch.equal(ids[shift:].view(100, k), want[0])
        assert torch.equal(d2[shift:].view(100, k), want[1])
        assert (ids[:shift] == -7).all() and (d2[:shift] == -7).all()


@pytest.mark.parametrize("m", METHODS)
def test_rounds_match_the_single_list(m):
    """Multi-round lists continue the heap across shards: the first round
    equals the heap list, and repeating a shard offers equal keys."""
    s = _setup(distribution("ties", 4000, 3, seed=8))
    lay, _, _, dt, db = s
    dq = torch.from_numpy(datagen.uniform(300, 3, 9) * np.float32(6.0)).cuda()
    for k in (5, 16, 33):
        lists = ck.knn_lists(300, k)
        ids, d2, _ = ck.knn(dt, lay, dq, k, m, ck.LIST_HEAP, world_bounds=db)
        ck.knn_accumulate(dt, lay, dq, lists, True, m, world_bounds=db)
        assert torch.equal(lists & 0xffffffff, ids.long() & 0xffffffff)
        assert torch.equal((lists >> 32).int(), d2.view(torch.int32))
        again = lists.clone()
        one = lists.clone()
        ck.knn_accumulate(dt, lay, dq, again, False, m, world_bounds=db)
        ck.knn_accumulate(dt, lay, dq, one, False, m, world_bounds=db, flags=ONE)
        assert torch.equal(again, one)
