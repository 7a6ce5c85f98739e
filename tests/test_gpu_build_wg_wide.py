"""Elements of more than five words: levels built by one workgroup per subtree
while the subtree has at most 768 KiB, and by the chip-wide launches above
that, equal the oracle's tree byte for byte, with ties that reach every word of
the key."""
import numpy as np
import pytest
import torch

import cudakdtree_amd as ck
import oracle as oc
from cudakdtree_amd import datagen
from tests.helpers import make_elements

pytestmark = pytest.mark.gpu

LIMIT = 768 << 10


def _points(kind, n, D):
    c = datagen.uniform(n, D, n)
    if kind == "grid":  # more than 256 elements a step: every word is looked at
        c = np.floor(c * np.float32(5))
    elif kind == "shared":  # 600 elements share the first coordinate, 300 of them two
        a = (n - 600) // 2
        c = c[np.argsort(c[:, 0], kind="stable")]
        c[a:a + 600, 0] = c[a + 300, 0]
        c[a + 100:a + 400, 1 % D] = np.float32(0.5)
        c = c[np.random.RandomState(n).permutation(n)]
    return np.ascontiguousarray(c, np.float32)


@pytest.mark.parametrize("words", [6, 7, 24, 63, 64])
@pytest.mark.parametrize("kind", ["uniform", "grid", "shared"])
@pytest.mark.parametrize("explicit", [False, True])
def test_subtree_bytes(words, kind, explicit):
    D = 3
    lay = ck.Layout(D, ck.SCALAR_F32, 4 * words, 4 if words > 6 else 0,
                    4 * (words - 1) if explicit else -1, 4)
    fit = min(16384, LIMIT // (4 * words))
    for n in (1025, fit, fit + 1, 2 * fit + 3):
        print(words, kind, explicit, n, flush=True)
        e = make_elements(_points(kind, n, D), lay)
        ref, _ = oc.build_host(e, lay, want_bounds=True)
        d = torch.from_numpy(np.ascontiguousarray(e).copy()).cuda()
        ck.buildTree(d, lay, ck.bounds_tensor(lay))
        torch.cuda.synchronize()
        assert np.array_equal(d.cpu().numpy().view(np.uint8), ref.view(np.uint8))
