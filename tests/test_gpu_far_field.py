"""The far field by columns (k_far_field_cols) at the edges of its tiles,
against direct FP64 sums over the dipoles: lattices whose l axis is shorter
than, equal to and much longer than a 16-point chunk, column counts that leave
partial pieces and batches, direction sets of one to eight members per group
(and of 9, which splits into threes, and 13, which does not split) with group
counts on both sides of a 16-group tile; and right-hand sides with direction
sets of their own against the per-direction kernel.

Bound: FP32 phases (three factors, each the rounded exp of a float argument of
at most |k r| <= 0.3 * max(n) * 3 / 2) and FP32 sums over one column's chunks,
one piece's 8 columns and the two phase products, then FP64: with u = 2^-24,
|error| <= u (n_l + 16 + 4 sum of the arguments' bounds) sum |P| per component."""

import numpy as np
import pytest

import ddafft

pytestmark = pytest.mark.gpu

KD = np.float32(0.3)


def planes(nang, nplanes, rng):
    """nplanes rotations about z of nang random directions: z equal bit for bit."""
    th = np.sort(rng.uniform(0, np.pi, nang))
    ph = rng.uniform(0, 2 * np.pi, nplanes)
    z = np.cos(th).astype(np.float32)
    d = np.stack([np.outer(np.cos(ph), np.sin(th)), np.outer(np.sin(ph), np.sin(th)),
                  np.broadcast_to(z, (nplanes, nang))], 2)
    return d.reshape(-1, 3).astype(np.float32)


def fp64_far_field(dims, occ, p, dirs):
    r = [np.arange(v, dtype=np.float32) * KD - np.float32((v - 1) * float(KD) / 2) for v in dims]
    ph = [np.exp(1j * np.outer(dirs[:, a], r[a]).astype(np.float64)) for a in range(3)]
    q = np.where((occ > 0)[..., None], p, 0).astype(np.complex128)
    s = np.stack([np.einsum("di,dj,ijl,dl->d", ph[0], ph[1], q[..., c], ph[2], optimize=True) for c in range(3)], 1)
    n = dirs.astype(np.float64)
    return s - n * np.sum(n * s, 1, keepdims=True)


@pytest.mark.parametrize("dims,nang,nplanes", [
    ((4, 4, 4), 1, 1), ((8, 4, 8), 3, 2), ((4, 8, 16), 16, 3), ((8, 8, 32), 17, 4), ((4, 16, 64), 15, 5),
    ((16, 4, 16), 33, 6), ((8, 8, 128), 5, 7), ((4, 4, 512), 31, 8), ((16, 8, 8), 7, 9), ((8, 8, 16), 2, 13),
    ((512, 4, 4), 9, 1), ((4, 512, 8), 19, 2), ((32, 32, 16), 257, 1)])
def test_far_field_columns(dims, nang, nplanes):
    rng = np.random.default_rng(sum(dims) + 7 * nang + nplanes)
    occ = (rng.random(dims) < 0.4).astype(np.int8)
    occ[0, 0, 0] = 1
    p = (rng.standard_normal(dims + (3,)) + 1j * rng.standard_normal(dims + (3,))).astype(np.complex64)
    dirs = planes(nang, nplanes, rng)
    print("far field", dims, nang, nplanes, flush=True)
    with ddafft.Context(dims, KD, nrhs_max=1) as ctx:
        ctx.set_target(occ, [0, 1])
        esc = ctx.far_field(p, dirs)   # p is not zero off the dipoles
    ref = fp64_far_field(dims, occ, p, dirs)
    amp = np.sum(np.abs(p[occ > 0]))
    arg = 0.3 * sum(dims) / 2
    tol = 2.0 ** -24 * (dims[2] + 16 + 4 * arg) * amp
    err = np.max(np.abs(esc - ref))
    print("error %.3g bound %.3g" % (err, tol), flush=True)
    assert err <= tol


@pytest.mark.parametrize("nrhs,shared", [(1, True), (3, True), (3, False), (5, False)])
def test_far_field_columns_per_rhs_sets(nrhs, shared):
    """Every right-hand side against the per-direction kernel on the same
    dipoles (bit for bit: the far field does not feed back into the solve)."""
    rng = np.random.default_rng(40 + nrhs)
    dims = (8, 16, 32)
    occ = (rng.random(dims) < 0.5).astype(np.int8)
    alpha = np.array([0, ddafft.polarizability(1, KD, 1.5 + 0.02j)], np.complex64)
    sets = np.stack([planes(13, 1, rng) for _ in range(nrhs)])
    k = np.broadcast_to(np.array([0, 0, 1], np.float32), (nrhs, 3))
    e = np.stack([np.eye(3)[r % 2] for r in range(nrhs)]).astype(np.complex64)
    out = {}
    print("far field sets", nrhs, shared, flush=True)
    with ddafft.Context(dims, KD, nrhs_max=nrhs) as ctx:
        ctx.set_target(occ, [0, 1])
        for mode in (0, 1):
            ctx.set_tuning(ff_group=mode)
            out[mode] = ctx.solve_ex("bicgstab", alpha, k, e, dirs=sets[0] if shared else sets, max_step=3,
                                     err_max=1e-9)
            P = [ctx.dipoles(r) for r in range(nrhs)]
    for r in range(nrhs):
        amp = np.sum(np.abs(P[r]))
        # both forms within the module's bound of the exact sum; the per-direction one adds its terms in FP32 over
        # at most ceil(cells / 256) dipoles per thread
        tol = 2.0 ** -24 * (2 * (16 + 4 * 0.3 * sum(dims) / 2) + dims[2] + 16) * amp
        assert np.max(np.abs(out[0][r]["esc"] - out[1][r]["esc"])) <= tol
        assert out[0][r]["cext"] == out[1][r]["cext"]
