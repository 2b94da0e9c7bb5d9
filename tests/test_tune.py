"""The autotuner measures what the library runs: planes of at most 2^11 cells
always take the fused passes, so that tune.py neither measures nor tunes
anything else on the two-pass form there; larger planes of up to 64 x 64 it
measures both ways and tunes on the faster one."""

import numpy as np
import pytest

import tune


class Recorder:
    """A context whose fused passes lose, and that remembers how it was tuned
    when a solve ran."""

    def __init__(self, dims, kd, nrhs_max):
        self.fuse, self.fuses, self.solved = -1, [], []

    def set_target(self, occ, mv):
        pass

    def set_tuning(self, fuse_zy=None, **other):
        if fuse_zy is not None:
            self.fuse = int(fuse_zy)
            self.fuses.append(self.fuse)

    def time_matvec(self, nrhs, reps):
        t = 2e-3 if self.fuse == 1 else 1e-3
        return np.array([t, t, 1e-2, t, t]), 2e-2

    def solve(self, *a, **kw):
        self.solved.append(self.fuse)

    def close(self):
        pass


@pytest.mark.parametrize("dims,nrhs", [((32, 32, 32), 2), ((32, 32, 64), 16), ((8, 8, 256), 1), ((64, 64, 64), 2),
                                       ((128, 128, 128), 1)])
def test_fuse_is_left_alone_on_small_planes(monkeypatch, dims, nrhs):
    made = []
    monkeypatch.setattr(tune.ddafft, "Context", lambda *a, **kw: made.append(Recorder(*a, **kw)) or made[-1])
    monkeypatch.setattr(tune, "target", lambda d: (0.1, np.ones(d, np.int8), np.zeros(2, np.complex64)))
    entry = tune.tune_case(dims, nrhs, 4, lambda msg: None)
    ctx, = made
    if dims[1] * dims[2] <= 2048:
        assert ctx.fuses == [] and set(ctx.solved) == {-1} and entry["fuse"] == 1
    elif max(dims[1:]) <= 64:
        assert {0, 1} <= set(ctx.fuses) and set(ctx.solved) == {0} and entry["fuse"] == 0
    else:
        assert entry["fuse"] == 0


def test_table_agrees_with_the_schedule():
    """The compiled-in table holds no two-pass entry for a plane that never runs it."""
    import os
    import re
    path = os.path.join(os.path.dirname(tune.__file__), "csrc", "tuned_table.hpp")
    rows = re.findall(r"\{(\d+), (\d+), (\d+), \d+, \d+, [^,]+, \d, (\d)\}", open(path).read())
    assert len(rows) >= 10
    for ni, nj, nl, fuse in rows:
        if int(nj) * int(nl) <= 2048 and min(int(nj), int(nl)) >= 8:
            assert fuse == "1", (ni, nj, nl)
