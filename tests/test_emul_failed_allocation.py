"""Calls on a context after a device allocation has failed, on the CPU
emulation of the library (tests/emul), whose allocations fail on demand and
whose every access AddressSanitizer checks: they are refused with an error
until the failed call has been repeated, and then give the results of a fresh
context.  Like test_emul.py it runs when DDAFFT_EMUL=1 is set."""

import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EMUL = os.path.join(ROOT, "tests", "emul")
CASES = ["set_target", "directions"]


@pytest.mark.skipif(os.environ.get("DDAFFT_EMUL") != "1", reason="set DDAFFT_EMUL=1 to run")
@pytest.mark.parametrize("case", CASES)
def test_failed_allocation(case):
    subprocess.run(["make", "-C", EMUL, "-s"], check=True)
    libs = [subprocess.run(["gcc", "-print-file-name=" + n], capture_output=True, text=True).stdout.strip()
            for n in ("libasan.so", "libubsan.so")]
    env = dict(os.environ, LD_PRELOAD=" ".join(libs), ASAN_OPTIONS="detect_leaks=0:abort_on_error=1",
               UBSAN_OPTIONS="halt_on_error=1:print_stacktrace=1")
    r = subprocess.run([sys.executable, os.path.abspath(__file__), case], env=env, capture_output=True, text=True,
                       timeout=900)
    print(r.stdout[-4000:], r.stderr[-4000:])
    assert r.returncode == 0 and "ALL OK" in r.stdout


KINC = np.array([0, 0, 1], np.float32)
EINC = np.eye(3, dtype=np.complex64)[:1]
DIMS = (4, 4, 8)


def alpha_of(kd):
    return np.array([0, ddafft.polarizability(1, kd, 1.5 + 0.01j)], np.complex64)


def refused(call, message):
    with pytest.raises(ddafft.DdafftError, match=message):
        call()


def set_target():
    """A larger target whose block cannot be allocated: every call that needs
    a target is refused, and set_target again makes the context whole."""
    kd = np.float32(0.5)
    alpha, small, full = alpha_of(kd), np.zeros(DIMS, np.int8), np.ones(DIMS, np.int8)
    small[1, 2, 3:5] = 1
    dirs = np.array([[0, 0, 1], [1, 0, 0]], np.float32)
    p = np.ones(DIMS + (3,), np.complex64)

    def solve(ctx, **kw):
        return ctx.solve("bicgstab", alpha, KINC, EINC, dirs=dirs, max_step=1, err_max=1e-9, **kw)[0]

    with ddafft.Context(DIMS, kd, nrhs_max=2) as ctx:
        ctx.set_target(small, [0, 1])
        solve(ctx)
        ddafft._lib.emul_fail_malloc(0)
        refused(lambda: ctx.set_target(full, [0, 1]), "hipMalloc")
        m = np.array([1, 1.5], np.complex64)
        for call in (lambda: solve(ctx), lambda: solve(ctx, noalloc=True), lambda: ctx.matvec(alpha, p),
                     lambda: ctx.far_field(p, dirs), lambda: ctx.cabs_cext(alpha, KINC, EINC[0], p),
                     lambda: ctx.time_matvec(1, 1), lambda: ctx.convolution(p),
                     lambda: ctx.gradient("bicgstab", alpha, alpha, m, KINC, EINC, np.ones((1, 2)), ndirs=0)):
            refused(call, "set_target first")
        ctx.set_target(full, [0, 1])
        got = solve(ctx)
    with ddafft.Context(DIMS, kd, nrhs_max=2) as ctx:
        ctx.set_target(full, [0, 1])
        ref = solve(ctx)
    assert np.array_equal(got["esc"], ref["esc"]) and got["cext"] == ref["cext"]


def directions():
    """A larger direction set that cannot be allocated, resident or brought by
    a solve: the set that was resident is gone, and solves that ask for it are
    refused until a set is given again."""
    kd = np.float32(0.5)
    alpha = alpha_of(kd)
    dirs = np.array([[0, 0, 1], [1, 0, 0]], np.float32)
    more = np.repeat(dirs, 8, 0)

    def solve(ctx, **kw):
        return ctx.solve("bicgstab", alpha, KINC, EINC, max_step=1, err_max=1e-9, **kw)[0]

    with ddafft.Context(DIMS, kd, nrhs_max=2) as ctx:
        ctx.set_target(np.ones(DIMS, np.int8), [0, 1])
        for fails in (lambda: ctx.set_directions(more), lambda: solve(ctx, dirs=more)):
            ctx.set_directions(dirs)
            ref = solve(ctx)
            ddafft._lib.emul_fail_malloc(0)
            refused(fails, "hipMalloc")
            refused(lambda: solve(ctx), "differs from the resident directions")
            refused(lambda: solve(ctx, noalloc=True), "differs from the resident directions")
            refused(lambda: ctx.gradient("bicgstab", alpha, alpha, np.array([1, 1.5]), KINC, EINC, np.ones((1, 4))),
                    "bad directions")
            ctx.set_directions(dirs)
            assert np.array_equal(solve(ctx)["esc"], ref["esc"])


if __name__ == "__main__":
    sys.path.insert(0, os.path.join(ROOT, "dda-fft_amd"))
    import ddafft

    ddafft.load(os.path.join(EMUL, "libddafft_emul.so"))
    globals()[sys.argv[1]]()
    print("ALL OK")
