"""Temporaries kept between calls: builds and sorted queries interleaved over
streams and threads, with the kept memory given back in between, give the
single-stream results."""
import threading

import pytest
import torch

import cudakdtree_amd as ck
from cudakdtree_amd import datagen

pytestmark = pytest.mark.gpu


def _work(pts, q, lay, out, i):
    with torch.cuda.stream(torch.cuda.Stream()):
        for r in range(3):
            t = pts.clone()
            ck.buildTree(t, lay)
            ids, d2, _ = ck.knn(t, lay, q, 4, flags=ck.QUERY_SORT)
            if r == 1:
                ck.release_memory()
        torch.cuda.current_stream().synchronize()
        out[i] = (t, ids, d2)


def test_streams_threads_and_release():
    lay = ck.float_points(3)
    sets = [(torch.from_numpy(datagen.uniform(30000 + 7001 * i, 3, i)).cuda(),
             torch.from_numpy(datagen.uniform(9000, 3, 50 + i)).cuda()) for i in range(4)]
    torch.cuda.synchronize()
    want, got = [None] * 4, [None] * 4
    for i, (p, q) in enumerate(sets):
        _work(p, q, lay, want, i)
    threads = [threading.Thread(target=_work, args=(p, q, lay, got, i))
               for i, (p, q) in enumerate(sets)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    ck.release_memory()
    for w, g in zip(want, got):
        for a, b in zip(w, g):
            assert torch.equal(a, b)
