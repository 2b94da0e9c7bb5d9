"""The allocation-free solve at the limit of its scratch on planes of eight
rows, whose fused inverse passes need more block partials (3 n_i a right-hand
side) than the passes apart (n_i n_j / 4): a request that fits with those is
accepted, and its results are bit for bit those of an ordinary solve with the
passes apart."""

import re

import numpy as np
import pytest

import ddafft
from conftest import bits

KINC = np.array([0, 0, 1], np.float32)
EINC = np.eye(3, dtype=np.complex64)[:1]
SCRATCH = 32 << 20


def at_the_limit(ni, nl, nrhs_max, sum_mode):
    dims = (ni, 8, nl)
    kd = np.float32(0.3)
    occ = (np.random.default_rng(ni + nl).random(dims) < 0.6).astype(np.int8)
    alpha = np.array([0, ddafft.polarizability(1, kd, 1.5 + 0.01j)], np.complex64)

    def solve(ctx, **kw):
        r = ctx.solve("cg", alpha, KINC, EINC, err_max=1e-4, **kw)[0]
        return [r["steps"], r["err_hist"], bits(np.float32(r["cext"])), bits(np.float32(r["cabs"])),
                bits(ctx.dipoles(0))]

    with ddafft.Context(dims, kd, nrhs_max=nrhs_max) as ctx:
        ctx.set_target(occ, [0, 1])
        ctx.set_sum_mode(sum_mode)
        # a step of the history takes 8 bytes for each right-hand side of the
        # context and 8 in the results; what else the scratch holds, but for
        # the partials, is below 8 KB (the sequential sums: two floats a dipole)
        fixed = 8 * int(occ.sum()) * sum_mode
        fused, apart = 3 * ni * 48, 2 * ni * 48   # partial sums of one right-hand side, in bytes
        step = 8 * nrhs_max + 8
        tight = (SCRATCH - fixed - (fused + apart) // 2) // step   # only the smaller partials fit
        over = (SCRATCH - fixed) // step                            # neither fits
        print("scratch limit", dims, nrhs_max, "sum mode", sum_mode, "steps", tight, over, flush=True)
        assert (fused - apart) // 2 > 8192
        got = solve(ctx, max_step=tight, noalloc=True)
        with pytest.raises(ddafft.DdafftError, match="allocation-free s"):
            solve(ctx, max_step=over, noalloc=True)
        after = solve(ctx, max_step=50)   # the limit holds for that call only
    with ddafft.Context(dims, kd, nrhs_max=nrhs_max) as ctx:
        ctx.set_target(occ, [0, 1])
        ctx.set_sum_mode(sum_mode)
        fused = solve(ctx, max_step=50)
        ctx.set_tuning(fuse_zy=0)
        apart = solve(ctx, max_step=50)
    for a, b in zip(got + after, apart + fused):
        assert np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("sum_mode", [0, 1])
def test_noalloc_at_the_scratch_limit(sum_mode):
    at_the_limit(512, 8, 32, sum_mode)
