"""The matrix-core passes of dense FP32 chimera cells at the cell fillings and grid
sizes where their tiles and groups can go wrong, against the oracle; batched
replicas against single handles bit for bit.  Bars: tests/_parity.py."""
import math
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

DT, RHO = 0.005, 0.1
# (cells per side, mean particles per cell): around the least filling that takes
# the passes, one to several groups of 16 centres, grids whose chunks wrap around
CASES = [(4, 11.9), (4, 12.1), (4, 40.0), (5, 15.5), (5, 47.0), (7, 49.0), (9, 70.0), (6, 130.0), (23, 13.0),
         (31, 40.0), (4, 19.9), (4, 20.1), (5, 20.4), (7, 24.0), (23, 21.0)]


def system(cells, filling, prec="fp32k", sigma=1.3, seed=5):
    L = cells * RHO * 1.04
    n = int(round(cells * cells * filling))
    kw = dict(n=n, L=L, rho=RHO, v0=0.05, sigma=sigma, alpha=1.45, D=0.02)
    return spc2.params("chimera", prec, "auto", seed=seed, **kw), O.chimera(threads=8, **kw), L, n


def state_of(n, L, clump=0.0):
    rng = np.random.default_rng(n)
    st = rng.uniform(0.0, L, 3 * n)
    st[2::3] = rng.uniform(0.0, 2 * np.pi, n)
    k = int(clump * n)  # that share of the particles in a fifth of the box's height
    st[1:3 * k:3] = rng.uniform(0.3 * L, 0.5 * L, k)
    return st


@pytest.mark.parametrize("cells,filling", CASES)
@pytest.mark.parametrize("sigma,clump", [(1.3, 0.0), (-0.02, 0.0), (37.0, 0.5)])
def test_rhs_and_srk_step(cells, filling, sigma, clump):
    p, orc, L, n = system(cells, filling, sigma=sigma)
    st = state_of(n, L, clump)
    kp, kn = np.random.default_rng(n + 1).normal(0.0, 1.0, 3 * n), np.full(3 * n, 7.5)
    U = np.random.default_rng(n + 2).standard_normal(2 * n)
    what = f"{cells} cells, {filling} per cell, sigma {sigma}"
    with spc2.Sim(p) as s:
        s.set_state(st)
        s.set_counting(True)
        got = s.eval_rhs(kp, 0.5, DT, kn)
        cnt = s.counts()
        gd, ga = s.eval_rhs_ito()
        s.step("srk", DT, 0, 1, noise=U)
        after = s.get_state()
    ref, rc, scale = O.rhs_k(orc, st, kp, 0.5, DT, kn, term_scale=True)
    assert_rhs_terms(got, ref, scale, p.v0, TOL["fp32k"], what, ref[2::3] == kn[2::3])
    assert np.array_equal(cnt, rc), (cnt, rc)
    _, ra, _ = O.rhs_ito(orc, st)
    for c in (0, 1):
        err = np.abs(ga[c::2] - ra[c::2]).max()
        assert err <= TOL["fp32k"] * np.abs(ra[c::2]).max(), f"{what}: additional[{c}] {err:.3e}"
    assert_state(after, O.step_srk(orc, st, DT, U), st, L, TOL["fp32k"], what)


def test_phase_that_is_not_finite_reaches_its_partners_only():
    p, orc, L, n = system(9, 40.0)
    st = state_of(n, L)
    st[2 + 3 * 17] = np.nan
    z = np.zeros(3 * n)
    with spc2.Sim(p) as s:
        s.set_state(st)
        got = s.eval_rhs(z, 0.0, DT, z)
    ref, _, scale = O.rhs_k(orc, st, z, 0.0, DT, z, term_scale=True)
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.isnan(ref).sum() > 20
    ok = ~np.isnan(ref[2::3])
    err = np.abs(got[2::3] - ref[2::3])[ok]
    assert (err <= TOL["fp32k"] * np.maximum(np.abs(ref[2::3]), scale)[ok]).all()


@pytest.mark.parametrize("method", ["se", "srk"])
def test_batch_equals_single(method):
    reps = [system(c, f, sigma=0.3 + 0.2 * k, seed=20 + k)[0] for k, (c, f) in enumerate(CASES)]
    with spc2.Batch(reps) as b:
        b.init_random_state(0.1)
        b.set_tile_targets([64.0 + 96.0 * (k % 8) for k in range(len(reps))])
        b.step(DT, 18, method=method)  # across a re-homing
        got = [b.get_state(r) for r in range(len(reps))]
    for p, g in zip(reps, got):
        with spc2.Sim(p) as s:
            s.init_random_state(0.1)
            s.step(method, DT, 0, 18)
            assert np.array_equal(s.get_state(), g), f"n={p.n}"
