"""All-pairs phases beyond the fast sine's reduction (2^45): both passes take the
library's functions there.  Bars: tests/_parity.py."""
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
from _parity import TOL, assert_rhs_terms  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("turns", [1e6, 1e14])
@pytest.mark.parametrize("system", ["chimera", "vortex"])
def test_both_passes(system, turns):
    """10^6 turns are within the reduction, 10^14 beyond it."""
    n, prec = 130, "fp64"  # (the factored form rounds phi + alpha, 1e-9 at 10^6 turns)
    if system == "chimera":
        kw = dict(n=n, L=1.0, rho=0.3, v0=0.05, sigma=1.3, alpha=1.45, D=0.02)
        p, orc = spc2.params("chimera", prec, "auto", **kw), O.chimera(**kw)
    else:
        kw = dict(rho=0.3, D=0.02, velocity=0.15, mu_plus=100.0, mu_minus=80.0, xi_a=0.06, xi_r=0.03, kappa=20.0)
        p, orc = spc2.params("vortex", prec, "auto", n=n, L=1.0, **kw), O.vortex(n, 1.0, **kw)
    rng = np.random.default_rng(n)
    st, z = rng.uniform(0.0, 1.0, 3 * n), np.zeros(3 * n)
    st[2::3] = rng.uniform(0.0, 2 * np.pi, n) + 2 * np.pi * np.round(turns * rng.uniform(-1.0, 1.0, n))
    assert (np.abs(st[2::3]).max() > 2.0**45) == (turns > 1e13)
    with spc2.Sim(p) as s:
        s.set_state(st)
        got = s.eval_rhs(z, 0.0, 0.01, z)
        gd, ga = s.eval_rhs_ito()
    ref, _, scale = O.rhs_k(orc, st, z, 0.0, 0.01, z, term_scale=True)
    assert_rhs_terms(got, ref, scale, p.v0, TOL[prec], system)
    rd, ra, _ = O.rhs_ito(orc, st)
    assert_rhs_terms(gd, rd, scale, p.v0, TOL[prec], system)
    for c in (0, 1):
        assert np.abs(ga - ra)[c::2].max() <= TOL[prec] * np.abs(ra[c::2]).max(), system
