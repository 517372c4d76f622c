"""The all-pairs passes (a wavefront per particle) at the sizes where their lane
split can go wrong, against the oracle, and batched replicas against single
handles bit for bit.  Bars: tests/_parity.py."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (ROOT, os.path.join(ROOT, "oracle"), os.path.join(ROOT, "tests")):
    if p not in sys.path:
        sys.path.insert(0, p)

import oracle as O  # noqa: E402
import spc2_langevin_integration_amd as spc2  # noqa: E402
from _parity import TOL, assert_rhs_terms, assert_state  # noqa: E402

pytestmark = pytest.mark.gpu

L, RHO, DT = 1.0, 0.3, 0.005
VORT = dict(velocity=0.15, mu_plus=100.0, mu_minus=80.0, xi_a=0.06, xi_r=0.03, kappa=20.0)
# one particle, a pair, the edges of the 64 lanes and of the particles a batch's block takes, several rounds
SIZES = [1, 2, 31, 33, 63, 64, 65, 129, 515]


def systems(system, prec, n, seed=5):
    if system == "chimera":
        kw = dict(n=n, L=L, rho=RHO, v0=0.05, sigma=1.3, alpha=1.45, D=0.02)
        return spc2.params("chimera", prec, "auto", seed=seed, **kw), O.chimera(**kw)
    return (spc2.params("vortex", prec, "auto", n=n, L=L, rho=RHO, D=0.02, seed=seed, **VORT),
            O.vortex(n, L, rho=RHO, D=0.02, **VORT))


def state_of(n, turns=0.0):
    rng = np.random.default_rng(n)
    st = rng.uniform(0.0, L, 3 * n)
    st[2::3] = rng.uniform(0.0, 2 * np.pi, n) + 2 * np.pi * np.round(turns * rng.uniform(-1.0, 1.0, n))
    return st


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("prec", ["fp64", "fp32k", "fp64f"])
@pytest.mark.parametrize("system", ["chimera", "vortex"])
def test_allpairs_rhs_and_srk_step(system, prec, n):
    p, orc = systems(system, prec, n)
    st = state_of(n)
    # stage positions outside the box, in/out phase entries kept without partners
    kp, kn = np.random.default_rng(n + 1).normal(0.0, 1.0, 3 * n), np.full(3 * n, 7.5)
    U = np.random.default_rng(n + 2).standard_normal(2 * n)
    with spc2.Sim(p) as s:
        s.set_state(st)
        got = s.eval_rhs(kp, 0.5, DT, kn)
        s.step("srk", DT, 0, 1, noise=U)
        after = s.get_state()
    ref, _, scale = O.rhs_k(orc, st, kp, 0.5, DT, kn, term_scale=True)
    assert_rhs_terms(got, ref, scale, p.v0, TOL[prec], f"{system} {prec} n={n}")
    assert_state(after, O.step_srk(orc, st, DT, U), st, L, TOL[prec], f"{system} {prec} n={n} srk")


@pytest.mark.parametrize("system", ["chimera", "vortex"])
def test_allpairs_phases_beyond_the_fast_reduction(system):
    """Phases of up to 10^6 turns take the library's sine in the FP64 form."""
    n = 130
    p, orc = systems(system, "fp64", n)
    st, kn = state_of(n, turns=1e6), np.zeros(3 * n)
    with spc2.Sim(p) as s:
        s.set_state(st)
        got = s.eval_rhs(np.zeros(3 * n), 0.0, DT, kn)
    ref, _, scale = O.rhs_k(orc, st, np.zeros(3 * n), 0.0, DT, kn, term_scale=True)
    assert_rhs_terms(got, ref, scale, p.v0, TOL["fp64"], system)


@pytest.mark.parametrize("method", ["se", "srk"])
@pytest.mark.parametrize("prec", ["fp64", "fp32k"])
def test_allpairs_batch_equals_single(prec, method):
    reps = [systems(("chimera", "vortex")[k % 2], prec, n, seed=20 + k)[0] for k, n in enumerate(SIZES)]
    with spc2.Batch(reps) as b:
        b.init_random_state(0.1)
        b.step(DT, 20, method=method)
        got = [b.get_state(r) for r in range(len(reps))]
    for p, g in zip(reps, got):
        with spc2.Sim(p) as s:
            s.init_random_state(0.1)
            s.step(method, DT, 0, 20)
            assert np.array_equal(s.get_state(), g), f"n={p.n}"
