"""The bitonic and in-place builders take up to three steps of a merge per
pass through memory for elements of up to 5 words, one for wider ones, and
tiles of 2048 or 1024 elements: sizes at which a merge has one to seven such
steps and a ragged end, each tile size and word count, both tie rules.  The
oracle's builder, exactly, wherever its order is the builder's own."""
import pytest

import cudakdtree_amd as ck
from tests.helpers import distribution
from tests.test_gpu_builders_tl import check, unique_coords

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,D", [("float", 2), ("float", 3), ("payload", 3), ("explicit", 3),
                                    ("float", 6), ("rec96", 3)])
@pytest.mark.parametrize("n", [4099, 8190, 16385, 33000, 70001, 131073, 262143])
def test_merge_steps(n, kind, D):
    if kind == "rec96" and n > 70001:
        pytest.skip("the oracle's time")
    check(distribution("ties", n, D, seed=n), kind, ck.BUILDER_BITONIC, exact=True)
    check(unique_coords(n, D, kind, n), kind, ck.BUILDER_INPLACE, exact=True)
    check(distribution("ties", n, D, seed=n + 1), kind, ck.BUILDER_INPLACE, exact=False)
