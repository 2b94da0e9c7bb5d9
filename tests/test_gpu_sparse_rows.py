"""Solves on targets that leave planes, rows and parts of rows of the lattice
empty, through the launches that skip them (more than 2^18 cells x right-hand
sides) and the small launches that do not, split and fused forward passes: the
dipoles of every solver against the oracle bit for bit, zero off the dipoles,
after another target's solve has filled the context's vectors.  The skipped
values are zeros, so there is no tolerance."""

import numpy as np
import pytest

import ddafft
from conftest import directions

pytestmark = pytest.mark.gpu

KD = np.float32(0.4)


def sparse_target(dims, kind):
    occ = np.zeros(dims, np.int8)
    ni, nj, nl = dims
    if kind == "one":
        occ[ni - 1, nj // 2, 1] = 1
    elif kind == "corner":   # planes and rows empty on one side, holes inside
        occ[: ni // 4, nj // 2 + 1: nj - 1, 2: nl // 2] = 1
        occ[1, nj // 2 + 2, :] = 0
        occ[ni // 8, :, :] = 0
    else:   # two pieces with empty planes between them
        occ[1, 0, nl - 2:] = 1
        occ[ni - 3: ni - 1, nj - 1, : nl // 3] = 1
    return occ


@pytest.mark.parametrize("dims,nrhs,fuse", [((8, 16, 8), 2, False), ((32, 32, 32), 9, False), ((32, 32, 32), 9, True),
                                            ((16, 128, 32), 5, False), ((32, 16, 256), 3, False),
                                            ((16, 256, 128), 1, False), ((64, 64, 16), 5, True)])
@pytest.mark.parametrize("kind", ["one", "corner", "two"])
def test_sparse_rows(orc32, dims, nrhs, fuse, kind):
    occ = sparse_target(dims, kind)
    alpha = np.array([0, orc32.polarizability(1, KD, 1.6 + 0.05j)], np.complex64)
    k = np.array([0, 0, 1], np.float32)
    einc = np.stack([np.array([np.cos(r), np.sin(r), 0]) for r in range(nrhs)]).astype(np.complex64)
    dirs = directions(np.arange(0, 181, 60))
    print("sparse", dims, nrhs, fuse, kind, int(occ.sum()), flush=True)
    with ddafft.Context(dims, KD, nrhs_max=nrhs) as ctx:
        A = ctx.ahat()
        ctx.set_tuning(fuse_zy=fuse)
        ctx.set_target(np.ones(dims, np.int8), [0, 1])   # every vector filled everywhere
        ctx.solve("bicgstab", alpha, k, einc, dirs=dirs, max_step=1, err_max=1e-9)
        ctx.set_target(occ, [0, 1])
        for solver in range(4):
            res = ctx.solve(solver, alpha, k, einc, dirs=dirs, max_step=3, err_max=1e-12, tau=0.5)
            for r in (0, nrhs - 1):
                ref = orc32.dda_fft(solver, occ, [0, 1], alpha, KD, k, einc[r], A, dirs, max_step=3, err_max=1e-12,
                                    tau=0.5, return_p=True)
                P = ctx.dipoles(r)
                assert res[r]["steps"] == ref["steps"], (solver, r)
                got, want = P[occ > 0], ref["p"][occ > 0].astype(np.complex64)
                # one dipole interacts with nothing: 0 / 0 in both, a NaN whose sign bit is the machine's
                num = ~np.isnan(want.view(np.float32))
                assert np.array_equal(num, ~np.isnan(got.view(np.float32))), (solver, r)
                assert np.array_equal(got.view(np.uint32)[num], want.view(np.uint32)[num]), (solver, r)
                assert not np.any(P[occ == 0]), (solver, r)
