"""Bitonic and in-place builds of 24-word elements, which take one merge step
per pass through memory, at sizes of many passes: the default builder's tree
byte for byte (with unique coordinates for the in-place builder, whose order
among equal ones is its own)."""
import numpy as np
import pytest
import torch

import cudakdtree_amd as ck
from tests.helpers import distribution, layout_for, make_elements
from tests.test_gpu_builders_tl import unique_coords

pytestmark = pytest.mark.gpu


def _build(elems, lay, builder):
    d = torch.from_numpy(np.ascontiguousarray(elems).copy()).cuda()
    ck.build_tree(d, lay, builder)
    torch.cuda.synchronize()
    return d


@pytest.mark.parametrize("n", [131073, 262143])
def test_wide_elements(n):
    lay = layout_for("rec96", 3)
    tied = make_elements(distribution("ties", n, 3, seed=n), lay)
    assert torch.equal(_build(tied, lay, ck.BUILDER_BITONIC), _build(tied, lay, ck.BUILDER_DEFAULT))
    unique = make_elements(unique_coords(n, 3, "rec96", n), lay)
    assert torch.equal(_build(unique, lay, ck.BUILDER_INPLACE),
                       _build(unique, lay, ck.BUILDER_DEFAULT))
