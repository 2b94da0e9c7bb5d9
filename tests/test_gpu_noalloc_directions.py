"""The resident direction set after an allocation-free solve that brought
directions of its own: the same number of directions, split into other groups
of equal z, so that a split left behind passes every count check.  A gradient
with S11 weights, a solve and a far field on the resident set give the bits
they gave before, whichever of the two sets is the grouped one."""

import numpy as np
import pytest

import ddafft
from conftest import bits, directions

KINC = np.array([0, 0, 1], np.float32)
EINC = np.eye(3, dtype=np.complex64)[:2]


def planes(nang, degrees):
    return np.concatenate([directions(np.linspace(0, 180, nang), p) for p in degrees])


SETS = {"one plane of 12": planes(12, (0.0,)), "two planes of 6": planes(6, (0.0, 90.0)),
        "four planes of 3": planes(3, (0.0, 30.0, 60.0, 90.0))}


def resident_set_survives(dims, resident, own):
    kd = np.float32(0.5)
    occ, _ = ddafft.target_ellipsoid(dims, 1.0, 1.0)
    m = np.array([1, 1.5 + 0.01j], np.complex64)
    alpha = np.array([[0, ddafft.polarizability(1, kd, m[1])]] * 2, np.complex64)
    dadm = np.array([[0, ddafft.polarizability_deriv(1, kd, m[1])]] * 2, np.complex64)
    dirs, other = SETS[resident], SETS[own]
    normals = np.tile([0, 1.0, 0], (len(dirs), 1)).astype(np.float32)
    W = np.concatenate([np.zeros(2), np.linspace(1, 0.1, len(dirs))])[None].astype(np.float32)
    with ddafft.Context(dims, kd, nrhs_max=2) as ctx:
        ctx.set_target(occ, [0, 1])
        ctx.set_directions(dirs)

        def results():
            g = ctx.gradient("bicgstab", alpha, dadm, m, KINC, EINC, W, normals=normals, max_step=3, err_max=1e-9)
            s = ctx.solve("bicgstab", alpha, KINC, EINC, max_step=3, err_max=1e-9)
            return [g[k] for k in ("f", "s11", "grad_m", "grad_chi", "esc")] + [r["esc"] for r in s]

        before = results()
        ctx.solve("bicgstab", alpha, KINC, EINC, dirs=other, max_step=3, err_max=1e-9, noalloc=True)
        after = results()
    for k, (a, b) in enumerate(zip(before, after)):
        assert np.array_equal(bits(a), bits(b)), (resident, own, k)


@pytest.mark.gpu
@pytest.mark.parametrize("resident", SETS)
@pytest.mark.parametrize("own", SETS)
def test_resident_directions_survive_noalloc(resident, own):
    print("resident", resident, "own", own, flush=True)
    resident_set_survives((8, 8, 8), resident, own)
