"""The far field of a field from outside the solver counts its dipole cells
only, whatever the others hold, in every form of the sum and bit for bit, and
the context keeps the field as it was given."""

import numpy as np
import pytest

import ddafft
from conftest import bits


def masked_off_the_dipoles(dims):
    rng = np.random.default_rng(sum(dims))
    occ = (rng.random(dims) < 0.3).astype(np.int8)
    occ[0, 0, 0], occ[-1, -1, -1] = 1, 0
    p = (rng.standard_normal(dims + (3,)) + 1j * rng.standard_normal(dims + (3,))).astype(np.complex64)
    clean, foul = p.copy(), p.copy()
    clean[occ == 0] = 0
    foul[occ == 0] = np.nan
    foul[-1, -1, -1] = np.inf
    d = rng.standard_normal((5, 3))
    d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    with ddafft.Context(dims, np.float32(0.3), nrhs_max=1) as ctx:
        ctx.set_target(occ, [0, 1])
        for group, sums in ((1, 0), (0, 0), (-1, 1)):
            ctx.set_tuning(ff_group=group)
            ctx.set_sum_mode(sums)
            ref = ctx.far_field(clean, d)
            for q in (p, foul):
                got = ctx.far_field(q, d)
                assert np.isfinite(got).all() and np.array_equal(bits(got), bits(ref)), (dims, group, sums)
                assert np.array_equal(bits(ctx.dipoles(0)), bits(q))


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(4, 4, 4), (4, 8, 16), (32, 4, 64), (16, 16, 128)])
def test_far_field_of_dipole_cells_only(dims):
    masked_off_the_dipoles(dims)
