"""Temporaries of calls without a memory resource come from the pool that the
program chose for its device, where it chose one."""
import ctypes

import pytest
import torch

import cudakdtree_amd as ck
from cudakdtree_amd import datagen

pytestmark = pytest.mark.gpu

ATTR_RELEASE_THRESHOLD, ATTR_USED_HIGH = 4, 8


@pytest.fixture(scope="module")
def hip():
    L = ctypes.CDLL("libamdhip64.so")
    for name in ("hipDeviceGetDefaultMemPool", "hipMemPoolGetAttribute", "hipMemPoolSetAttribute"):
        getattr(L, name).restype = ctypes.c_int
    return L


def _build(n=300_000):
    lay = ck.float_points(3)
    t = torch.from_numpy(datagen.uniform(n, 3, 1)).cuda()
    ck.buildTree(t, lay)
    torch.cuda.synchronize()
    return t


def test_default_pool_with_a_threshold_serves(hip):
    pool, v = ctypes.c_void_p(), ctypes.c_uint64()
    assert hip.hipDeviceGetDefaultMemPool(ctypes.byref(pool), 0) == 0

    def attr(a, value=None):
        if value is None:
            assert hip.hipMemPoolGetAttribute(pool, a, ctypes.byref(v)) == 0
            return v.value
        v.value = value
        assert hip.hipMemPoolSetAttribute(pool, a, ctypes.byref(v)) == 0

    want = _build()
    assert attr(ATTR_RELEASE_THRESHOLD) == 0
    attr(ATTR_USED_HIGH, 0)
    _build()
    assert attr(ATTR_USED_HIGH) == 0  # the library's own pool
    attr(ATTR_RELEASE_THRESHOLD, 64 << 20)
    try:
        got = _build()
        assert attr(ATTR_USED_HIGH) >= 300_000 * 12  # at least the working copy
    finally:
        attr(ATTR_RELEASE_THRESHOLD, 0)
    assert torch.equal(got, want)


@pytest.mark.parametrize("stream", [0, 1, 2])  # null, hipStreamLegacy, hipStreamPerThread
def test_stock_streams(stream):
    lay = ck.float_points(3)
    pts = torch.from_numpy(datagen.uniform(20_000, 3, 4)).cuda()
    want = pts.clone()
    ck.buildTree(want, lay)
    torch.cuda.synchronize()
    rc = ck.lib().cukd_build_tree(ctypes.c_void_p(pts.data_ptr()), len(pts), ctypes.byref(lay),
                                  ck.BUILDER_DEFAULT, None, ctypes.c_void_p(stream), None)
    assert rc == 0, ck.lib().cukd_last_error()
    torch.cuda.synchronize()
    assert torch.equal(pts, want)
