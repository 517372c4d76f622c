"""Positions at the edges of what the passes take, against the oracle: positions
that are not finite, boxes of three cells along an axis, positions
several boxes apart.  Bars: tests/_parity.py."""
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
from _parity import TOL  # noqa: E402

pytestmark = pytest.mark.gpu


def systems(system, prec, path, n, Lx=1.0, Ly=1.0, rho=0.3, xi_a=0.06, xi_r=0.03):
    if system == "chimera":
        kw = dict(n=n, rho=rho, v0=0.05, sigma=1.3, alpha=1.45, D=0.02)
        return spc2.params("chimera", prec, path, Lx=Lx, Ly=Ly, **kw), O.chimera(L=Lx, Ly=Ly, **kw)
    kw = dict(rho=rho, velocity=0.15, mu_plus=100.0, mu_minus=80.0, xi_a=xi_a, xi_r=xi_r, kappa=20.0, D=0.02)
    return spc2.params("vortex", prec, path, n=n, Lx=Lx, Ly=Ly, **kw), O.vortex(n, Lx, Ly=Ly, **kw)


def state_of(n, Lx=1.0, Ly=1.0):
    rng = np.random.default_rng(n)
    return np.stack([rng.uniform(0.0, Lx, n), rng.uniform(0.0, Ly, n), rng.uniform(0.0, 2 * np.pi, n)], 1).ravel()


def check(p, orc, st, prec, what):
    """Partner counts, the phase derivatives and both Ito terms of one state."""
    n = p.n
    z = np.zeros(3 * n)
    with spc2.Sim(p) as s:
        s.set_state(st)
        counts = s.neighbour_counts()
        got = s.eval_rhs(z, 0.0, 0.01, z)
        gd, ga = s.eval_rhs_ito()
    for a, b in zip(counts, O.neighbour_counts(orc, st)):
        assert np.array_equal(a, b), what
    ref, _, scale = O.rhs_k(orc, st, z, 0.0, 0.01, z, term_scale=True)
    rd, ra, _ = O.rhs_ito(orc, st)
    for g, r in ((got, ref), (gd, rd), (ga, ra)):
        assert np.array_equal(np.isnan(g), np.isnan(r)), what
    for g, r in ((got, ref), (gd, rd)):
        assert (np.abs(g - r)[2::3] <= TOL[prec] * np.maximum(np.abs(r[2::3]), scale)).all(), what
    for c in (0, 1):
        assert np.abs(ga - ra)[c::2].max() <= TOL[prec] * np.abs(ra[c::2]).max(), what


# (3 x 3 cells hold the same candidates as all pairs, the path that the oracle takes at this rho)
@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("prec", ["fp64", "fp32k", "fp64f"])
@pytest.mark.parametrize("path", ["all_pairs", "cells"])
@pytest.mark.parametrize("system", ["chimera", "vortex"])
def test_position_that_is_not_finite_is_no_partner(system, path, prec, bad):
    n = 130
    p, orc = systems(system, prec, path, n)
    st = state_of(n)
    st[3 * 17] = bad
    check(p, orc, st, prec, f"{system} {path} {prec} {bad}")


# three cells along an axis and partners beyond a cell's side: from the middle cells some lie more than half the box
# away, so that the nearer image counts although no halo wraps (3 x 3 cells forced, then 4 x 3 as the reference takes)
@pytest.mark.parametrize("Lx,Ly,rho,xi_r", [(1.0, 1.0, 0.33, 0.45), (1.0, 0.8, 0.25, 0.3), (0.8, 1.0, 0.25, 0.3)])
@pytest.mark.parametrize("filling", [9, 61])
@pytest.mark.parametrize("prec", ["fp64", "fp64f"])
def test_three_cells_along_an_axis(monkeypatch, prec, filling, Lx, Ly, rho, xi_r):
    n = filling * int(Lx / rho) * int(Ly / rho)
    p, orc = systems("vortex", prec, "cells", n, Lx, Ly, rho, 0.2 * rho, xi_r)
    if Lx < Ly:  # the oracle takes all pairs there (rho > Lx / 4): the walks against each other only
        orc = None
    st, out = state_of(n, Lx, Ly), []
    for cap in (None, "0"):
        if cap is not None:
            monkeypatch.setenv("SPC2_LDS_CAP", cap)
        if orc is not None:
            check(p, orc, st, prec, f"{prec} {Lx} x {Ly}")
        with spc2.Sim(p) as s:
            s.set_state(st)
            out.append((*s.neighbour_counts(), *s.eval_rhs_ito()))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


# positions several boxes apart on the all-pairs path, rho the reference's separation itself: its product of the box
# count (3, 5) and L is rounded, and a fused one puts the partner a hair beyond rho
@pytest.mark.parametrize("L,d,rho", [(0.7, 1.107265286604193, 0.9927347133958067),
                                     (1.7, 2.7338815754156287, 2.366118424584371),
                                     (1.1, 3.213312990181401, 2.286687009818599)])
@pytest.mark.parametrize("prec", ["fp64", "fp32k", "fp64f"])
@pytest.mark.parametrize("system", ["chimera", "vortex"])
def test_all_pairs_several_boxes_apart(system, prec, L, d, rho):
    p, orc = systems(system, prec, "all_pairs", 2, L, L, rho)
    st = np.array([0.0, 0.1, 1.0, d, 0.1, 2.5])
    assert list(O.neighbour_counts(orc, st)[0]) == [1, 1]
    check(p, orc, st, prec, f"{system} {prec}")
