"""The far field by columns is no further from 64-bit sums than the
per-direction kernel, where its runs of FP32 sums count most: small lattices,
one direction a group, random moments (no plane wave's large sums to hide
them).

The error of a value is taken relative to the largest value of its set, and
its RMS over 8 seeds of three sets a lattice: 117 directions x 3 complex
components a seed, 5616 real errors.  Two forms of equal error then differ by
a ratio within 1 +- 2 / sqrt(2 * 5616) = 1 +- 0.02 (two standard deviations);
the bound is 1.05."""

import numpy as np
import pytest

import ddafft

pytestmark = pytest.mark.gpu

SETS = (None, 19, 61)   # 37 directions at random; one plane of so many angles


def directions(kind, rng):
    if kind is None:
        d = rng.standard_normal((37, 3))
        return (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    th = np.linspace(0, np.pi, kind)
    return np.stack([np.sin(th), 0 * th, np.cos(th)], 1).astype(np.float32)


def sums64(dims, kd, occ, p, dirs):
    ph = [np.exp(1j * np.outer(dirs[:, a].astype(np.float64), (np.arange(v) - (v - 1) / 2) * float(kd)))
          for a, v in enumerate(dims)]
    t = (np.where((occ > 0)[..., None], p, 0).astype(np.complex128).transpose(3, 0, 1, 2).reshape(-1, dims[2])
         @ ph[2].T).reshape(3, dims[0], dims[1], -1)
    s = np.stack([np.einsum("id,id->d", np.einsum("ijd,dj->id", t[c], ph[1]), ph[0].T) for c in range(3)], 1)
    n = dirs.astype(np.float64)
    return s - n * np.sum(n * s, 1, keepdims=True)


def error_ratio(dims, x, seeds):
    occ, _ = ddafft.target_ellipsoid(dims, dims[1] / dims[0], dims[2] / dims[0])
    e = {0: 0.0, 1: 0.0}
    for seed in range(seeds):
        for kind in SETS:
            rng = np.random.default_rng(100 * seed + (kind or 0))
            kd = np.float32(2 * x * (1 + 0.05 * rng.random()) / dims[0])
            dirs = directions(kind, rng)
            p = (rng.standard_normal(dims + (3,)) + 1j * rng.standard_normal(dims + (3,))).astype(np.complex64)
            ref = sums64(dims, kd, occ, p, dirs)
            with ddafft.Context(dims, kd, nrhs_max=1) as ctx:
                ctx.set_target(occ, [0, 1])
                for mode in e:
                    ctx.set_tuning(ff_group=mode)
                    e[mode] += np.sum(np.abs(ctx.far_field(p, dirs) - ref) ** 2) / np.max(np.abs(ref)) ** 2
    return np.sqrt(e[1] / e[0])


@pytest.mark.parametrize("dims,x", [((16, 16, 16), 3.0), ((8, 16, 32), 2.0), ((32, 32, 32), 5.0)])
def test_far_field_columns_error(dims, x):
    print("far-field error", dims, flush=True)
    ratio = error_ratio(dims, x, 8)
    print("columns / per direction %.3f" % ratio, flush=True)
    assert ratio <= 1.05
