"""The FP64 cell walks (a particle's candidates split over 1 to 16 lanes, the
plain form's partners collected as bits first) over the lane counts, sparse and
dense cells and the phases beyond the fast sine, against the oracle; batched
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

DT = 0.005
# 16 lanes (one cell row of 3, sparse cells, dense cells), 8, 4, 2 and 1 lanes
SIZES = [(301, 400.0), (1003, 100.0), (1003, 4000.0), (9001, 30000.0), (17001, 4000.0), (40003, 4000.0),
         (66001, 4000.0), (140001, 4000.0)]


def systems(system, prec, n, density, seed=5):
    L = math.sqrt(n / density)
    if system == "chimera":
        kw = dict(n=n, L=L, rho=min(0.1, 0.24 * L), v0=0.05, sigma=1.3, alpha=1.45, D=0.02)
        return spc2.params("chimera", prec, "cells", seed=seed, **kw), O.chimera(threads=8, **kw), L
    kw = dict(rho=min(0.05, 0.24 * L), D=0.02, velocity=0.025, mu_plus=100.0, mu_minus=80.0, xi_a=0.01, xi_r=0.006,
              kappa=20.0)
    return spc2.params("vortex", prec, "cells", n=n, L=L, seed=seed, **kw), O.vortex(n, L, threads=8, **kw), L


def state_of(n, L, turns=0.0):
    rng = np.random.default_rng(n)
    st = rng.uniform(0.0, L, 3 * n)
    st[2::3] = rng.uniform(0.0, 2 * np.pi, n) + 2 * np.pi * np.round(turns * rng.uniform(-1.0, 1.0, n))
    return st


@pytest.mark.parametrize("n,density", SIZES)
@pytest.mark.parametrize("prec", ["fp64", "fp64f"])
@pytest.mark.parametrize("system", ["chimera", "vortex"])
def test_cell_walk_lanes(system, prec, n, density):
    p, orc, L = systems(system, prec, n, density)
    st = state_of(n, L)
    kp, kn = np.random.default_rng(n + 1).normal(0.0, 1.0, 3 * n), np.full(3 * n, 7.5)
    U = np.random.default_rng(n + 2).standard_normal(2 * n)
    with spc2.Sim(p) as s:
        s.set_state(st)
        s.set_counting(True)
        got = s.eval_rhs(kp, 0.5, DT, kn)
        cnt = s.counts()
        s.step("srk", DT, 0, 1, noise=U)
        after = s.get_state()
    ref, rc, scale = O.rhs_k(orc, st, kp, 0.5, DT, kn, term_scale=True)
    assert_rhs_terms(got, ref, scale, p.v0, TOL[prec], f"{system} {prec} n={n}")
    assert np.array_equal(cnt, rc), (cnt, rc)
    assert_state(after, O.step_srk(orc, st, DT, U), st, L, TOL[prec], f"{system} {prec} n={n} srk")


@pytest.mark.parametrize("turns", [1e6, 1e14])
@pytest.mark.parametrize("neighbour", ["cells", "verlet"])
@pytest.mark.parametrize("system", ["chimera", "vortex"])
def test_phases_beyond_the_fast_reduction(system, neighbour, turns):
    """10^6 turns are within the fast sine's reduction, 10^14 beyond it."""
    n = 20011
    p, orc, L = systems(system, "fp64", n, 4000.0)
    p.neighbour = {"cells": spc2.NEIGH_CELLS, "verlet": spc2.NEIGH_VERLET}[neighbour]
    st, kn = state_of(n, L, turns), np.zeros(3 * n)
    with spc2.Sim(p) as s:
        s.set_state(st)
        got = s.eval_rhs(np.zeros(3 * n), 0.0, DT, kn)
    ref, _, scale = O.rhs_k(orc, st, np.zeros(3 * n), 0.0, DT, kn, term_scale=True)
    assert_rhs_terms(got, ref, scale, p.v0, TOL["fp64"], system)


@pytest.mark.parametrize("method", ["se", "srk"])
@pytest.mark.parametrize("prec", ["fp64", "fp64f"])
def test_cell_walk_batch_equals_single(prec, method):
    reps = [systems(("chimera", "vortex")[k % 2], prec, n, 4000.0, seed=20 + k)[0]
            for k, n in enumerate([1003, 1501, 9001, 9002, 40003, 140001])]
    for p in reps:
        p.neighbour = spc2.NEIGH_AUTO
    with spc2.Batch(reps) as b:
        b.init_random_state(0.1)
        b.step(DT, 17, method=method)  # across a re-homing
        got = [b.get_state(r) for r in range(len(reps))]
    for p, g in zip(reps, got):
        with spc2.Sim(p) as s:
            s.init_random_state(0.1)
            s.step(method, DT, 0, 17)
            assert np.array_equal(s.get_state(), g), f"n={p.n}"
