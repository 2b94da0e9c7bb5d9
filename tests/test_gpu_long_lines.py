"""The z and y passes of long lines, which run 512 threads (z from 128 points
up, the inverse one in small launches only; y from 256 points up): both
convolutions and the matvec of a random field and solves with every solver
against the oracle, bit for bit, on both sides of 2^18 cells x right-hand
sides."""

import pytest

from test_gpu_small_planes import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,nrhs", [((4, 32, 128), 2), ((4, 64, 128), 1), ((4, 16, 256), 3), ((4, 8, 512), 2),
                                       ((4, 256, 16), 2), ((4, 512, 8), 1), ((4, 512, 32), 1)])
def test_long_lines(orc32, dims, nrhs):
    check(orc32, dims, nrhs, True)


@pytest.mark.parametrize("dims,nrhs", [((16, 32, 128), 4), ((16, 32, 128), 5), ((4, 16, 256), 17), ((4, 256, 16), 17)])
def test_long_lines_large_launch(orc32, dims, nrhs):
    """(16, 32, 128) x 4 stays at 2^18; the others are beyond it."""
    check(orc32, dims, nrhs, False)
