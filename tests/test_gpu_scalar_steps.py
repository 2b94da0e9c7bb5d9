"""The scalar step in the middle of an iteration, within the update kernel (at
most 256 partial sums a right-hand side and 512 update blocks) and in a launch
of its own: solves with every solver against the oracle, bit for bit, at the
edges of that rule."""

import pytest

from test_gpu_small_planes import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,nrhs", [((4, 8, 8), 1), ((32, 32, 128), 1), ((16, 32, 64), 4), ((16, 32, 128), 2),
                                       ((32, 32, 128), 2), ((32, 64, 64), 1), ((16, 32, 64), 5)])
def test_scalar_steps(orc32, dims, nrhs):
    """Within: the first four (256 partials and 512 blocks at the second);
    apart: 1024 blocks, 512 partials, 640 blocks."""
    check(orc32, dims, nrhs, False)
