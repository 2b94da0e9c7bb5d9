"""The fused plane passes (k_zyf_wide, k_zyf, k_yzi) of every plane shape they
are built for, against the oracle: both convolutions and the matvec of a random
field, and solves with every solver (each prologue and epilogue) bit for bit,
in a small launch and, for a few shapes, in one of more than 2^18 cells x
right-hand sides, where the forward pass takes its other form."""

import numpy as np
import pytest

import ddafft
from conftest import bits, directions

pytestmark = pytest.mark.gpu

KD = np.float32(0.35)
PLANES = [(nj, nl) for nj in (8, 16, 32, 64, 128, 256) for nl in (8, 16, 32, 64, 128, 256) if nj * nl <= 2048]


def check(orc, dims, nrhs, conv):
    rng = np.random.default_rng(sum(dims) + nrhs)
    occ = ((rng.random(dims) < 0.6) * (1 + (rng.random(dims) < 0.3))).astype(np.int8)
    mv = [0, 1, 1]
    alpha = np.array([0, orc.polarizability(1, KD, 1.5 + 0.01j), orc.polarizability(1, KD, 1.7 + 0.1j)], np.complex64)
    kinc = np.array([0, 0, 1], np.float32)
    einc = np.stack([np.array([np.cos(r), np.sin(r), 0]) for r in range(nrhs)]).astype(np.complex64)
    dirs = directions(np.arange(0, 181, 90))
    print("planes", dims, nrhs, flush=True)
    with ddafft.Context(dims, KD, nrhs_max=nrhs) as ctx:
        A = ctx.ahat()
        ctx.set_target(occ, mv)
        if conv:
            x = (rng.standard_normal(dims + (3,)) + 1j * rng.standard_normal(dims + (3,))).astype(np.complex64)
            for conj in (False, True):
                assert np.array_equal(bits(ctx.convolution(x, conj=conj)), bits(orc.convolution(A, x, conj=conj)))
                assert np.array_equal(bits(ctx.matvec(alpha, x, conj=conj)),
                                      bits(orc.matvec(A, occ, mv, alpha, x, conj=conj)))
        for solver in range(4):
            res = ctx.solve(solver, alpha, kinc, einc, dirs=dirs, max_step=3, err_max=1e-12, tau=0.5)
            for r in {0, nrhs - 1}:
                ref = orc.dda_fft(solver, occ, mv, alpha, KD, kinc, einc[r], A, dirs, max_step=3, err_max=1e-12,
                                  tau=0.5, return_p=True)
                assert res[r]["steps"] == ref["steps"]
                np.testing.assert_allclose(res[r]["err_hist"], ref["err_hist"], rtol=1e-9)
                assert np.array_equal(bits(ctx.dipoles(r)), bits(ref["p"].astype(np.complex64))), (solver, r)


@pytest.mark.parametrize("nj,nl", PLANES)
def test_small_planes(orc32, nj, nl):
    check(orc32, (8, nj, nl), 2, True)


@pytest.mark.parametrize("dims,nrhs", [((64, 8, 8), 65 - 1), ((128, 32, 64), 2), ((128, 16, 128), 2), ((64, 64, 64), 2)])
def test_small_planes_large_launch(orc32, dims, nrhs):
    """(64, 8, 8) x 64 stays at 2^18; the others are beyond it."""
    check(orc32, dims, nrhs, False)
