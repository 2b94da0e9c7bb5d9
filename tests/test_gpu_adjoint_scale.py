"""The scale of the adjoint sources (k_adj_scale) over one, some, 256 and more
block partials: objectives four times as large give gradients exactly four
times as large, because the scale of each source is its own and exact in a
factor of four, and each adjoint solution is finite and not zero."""

import numpy as np
import pytest

from test_gpu_gradient import _gpu_gradient

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(4, 8, 8), (16, 16, 16), (32, 32, 64), (32, 64, 64), (64, 32, 64)])
def test_adjoint_scale(dims):
    rng = np.random.default_rng(sum(dims))
    occ = (rng.random(dims) < 0.5).astype(np.int8)
    th = np.array([0.3, 2.0])
    dirs = np.stack([np.sin(th), 0 * th, np.cos(th)], 1).astype(np.float32)
    normals = np.tile([0, 1.0, 0], (2, 1)).astype(np.float32)
    W = np.array([[1.0, 0, 0, 0], [0.5, 1, 0.25, 0.5]])
    print("adjoint scale", dims, flush=True)
    a, b = (_gpu_gradient(occ, [0, 1], [1, 1.5 + 0.01j], 0.3, w, dirs, normals, max_step=4) for w in (W, 4 * W))
    for k in ("grad_m", "grad_chi"):
        assert np.isfinite(a[k]).all() and (np.abs(a[k]).reshape(2, -1).max(1) > 0).all()
        assert np.array_equal(4 * a[k], b[k]), k
