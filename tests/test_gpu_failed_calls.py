"""A call that reports a failed launch leaves the handle fit for the next one: the
counts and stages of its builds start afresh.  The failure is another library
call's error in the same thread, which the launches' check finds."""
import ctypes
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

import spc2_langevin_integration_amd as spc2  # noqa: E402

pytestmark = pytest.mark.gpu

N = 700


def sticky_error():
    """hipErrorInvalidDevice as the thread's last error: the device stays as it is."""
    spc2.load()
    hip = ctypes.CDLL("libamdhip64.so.7")
    assert hip.hipSetDevice(9999) != 0


def state_of(n, seed=3):
    rng = np.random.default_rng(seed)
    st = rng.uniform(0.0, 1.0, 3 * n)
    st[2::3] = rng.uniform(0.0, 2 * np.pi, n)
    return st


CALLS = {
    "set_state": lambda s: s.set_state(state_of(N, 4)),
    "eval_rhs": lambda s: s.eval_rhs(np.zeros(3 * N), 0.0, 0.01, np.zeros(3 * N)),
    "eval_rhs_ito": lambda s: s.eval_rhs_ito(),
    "neighbour_counts": lambda s: s.neighbour_counts(),
    "step": lambda s: s.step("srk", 0.01, 0, 3),
}


@pytest.mark.parametrize("call", sorted(CALLS))
@pytest.mark.parametrize("path,side", [("cells", 9), ("cells", 129), ("all_pairs", 3), ("verlet", 9)])
def test_handle_after_a_failed_call(path, side, call):
    p = spc2.params("chimera", "fp64", path, n=N, L=1.0, rho=1.0 / (side + 0.5), v0=0.5, seed=7)

    def after(s):
        s.set_state(state_of(N))
        out = [*s.neighbour_counts(), *s.eval_rhs_ito()]
        s.step("se", 0.001, 0, 5)
        return out + [s.get_state()]

    with spc2.Sim(p) as s:
        want = after(s)
    with spc2.Sim(p) as s:
        s.set_state(state_of(N, 4))
        sticky_error()
        with pytest.raises(spc2.Spc2Error):
            CALLS[call](s)
        for a, b in zip(after(s), want):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("method", ["se", "srk"])
def test_batch_after_a_failed_call(method):
    reps = [spc2.params(sy, "fp32k", "auto", n=n, L=1.0, rho=0.1, xi_a=0.02, xi_r=0.01, seed=n)
            for sy, n in (("chimera", 700), ("vortex", 301), ("chimera", 2500))]

    def after(b):
        for r, p in enumerate(reps):
            b.set_state(r, state_of(p.n))
        b.step(0.001, 5, method=method)
        return [b.get_state(r) for r in range(len(reps))]

    with spc2.Batch(reps) as b:
        want = after(b)
    with spc2.Batch(reps) as b:
        sticky_error()
        with pytest.raises(spc2.Spc2Error):
            b.step(0.001, 5, method=method)
        got = after(b)
    # (the draws go by each replica's count of steps done, which a failed call leaves alone)
    for a, w in zip(got, want):
        assert np.array_equal(a, w)
