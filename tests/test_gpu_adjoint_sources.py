"""The scale of the adjoint sources (k_adj_scale) itself, over one, some, 256
and more block partials.  CG without an iteration leaves the scaled source
b / s in the dipoles, s = sum_j |b_j| / sum_j |alpha_j| |E|, so that its norms
add up to sum_j |alpha_j| |E| whatever the objective; a sum that misses a
partial misses this by that partial's share.

Bound: b is float, and the scaling rounds it twice more (1 / s, the product):
three roundings a component, 3 * 2^-24 of each norm; |alpha| comes from the
same floats as the library's."""

import numpy as np
import pytest

import ddafft

KINC = np.array([0, 0, 1], np.float32)
EINC = np.array([[1, 0, 0], [0, 1, 0]], np.complex64)


def norms_and_sums(dims, seed):
    """sum |b / s| of each adjoint source over the dipoles, and sum |alpha| |E|."""
    rng = np.random.default_rng(seed)
    kd = np.float32(0.3)
    occ = ((rng.random(dims) < 0.5) * (1 + (rng.random(dims) < 0.3))).astype(np.int8)
    m = np.array([1, 1.5 + 0.01j, 1.7 + 0.1j], np.complex64)
    alpha = np.array([[0] + [ddafft.polarizability(1, kd, complex(v)) for v in m[1:]]] * 2, np.complex64)
    dadm = np.array([[0] + [ddafft.polarizability_deriv(1, kd, complex(v)) for v in m[1:]]] * 2, np.complex64)
    th = np.array([0.3, 2.0])
    dirs = np.stack([np.sin(th), 0 * th, np.cos(th)], 1).astype(np.float32)
    normals = np.tile([0, 1.0, 0], (2, 1)).astype(np.float32)
    W = np.array([[1.0, 0, 0, 0], [0, 1, 0, 0], [0.5, 1, 0.25, 0.5]], np.float32)
    with ddafft.Context(dims, kd, nrhs_max=6) as ctx:
        ctx.set_target(occ, [0, 1, 1])
        g = ctx.gradient("cg", alpha, dadm, m, KINC, EINC, W, dirs=dirs, normals=normals, max_step=0)
        b = [ctx.dipoles(r).astype(np.complex128) for r in range(6)]
    assert not g["info"][:, [0, 2]].any()   # no step, nothing restored: the dipoles are the sources
    want = np.sum(np.bincount(occ.ravel(), minlength=3) * np.abs(alpha[0].astype(np.complex128)))
    return [np.sum(np.linalg.norm(v, axis=-1)) for v in b], want


def check(dims):
    got, want = norms_and_sums(dims, sum(dims))
    print("adjoint sources", dims, ["%.2e" % (v / want - 1) for v in got], flush=True)
    for v in got:
        assert abs(v / want - 1) <= 3 * 2.0 ** -24


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(4, 8, 8), (16, 16, 16), (16, 32, 64), (32, 32, 64), (32, 64, 64), (64, 64, 64)])
def test_adjoint_source_norms(dims):
    """1, 16, 128, 256, 512 and 1024 partials a source."""
    check(dims)
