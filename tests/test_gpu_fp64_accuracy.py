"""The plain FP64 form's error against extended precision is no larger than that of
the reference's method: its sines, correctly rounded, added one by one in FP64."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

import spc2_langevin_integration_amd as spc2  # noqa: E402

pytestmark = pytest.mark.gpu

ALPHA = 1.45


@pytest.mark.parametrize("spread", [2 * np.pi, 0.3])
@pytest.mark.parametrize("path", ["verlet", "cells", "all_pairs"])
def test_phase_derivative_error(path, spread):
    side, filling = (9, 40) if path != "all_pairs" else (3, 300)
    n, rho = side * side * filling, 1.0 / (side + 0.02)
    rng = np.random.default_rng(7)
    st = rng.uniform(0.0, 1.0, 3 * n)
    st[2::3] = 1.234 + spread * rng.uniform(-0.5, 0.5, n)
    x, y, p = st[0::3], st[1::3], st[2::3]
    exact, added = np.zeros(n, np.longdouble), np.zeros(n)
    for i in range(n):
        dx, dy = x - x[i], y - y[i]
        dx, dy = dx - np.trunc(dx * 2.0), dy - np.trunc(dy * 2.0)
        m = np.nonzero(dx * dx + dy * dy <= rho * rho)[0]
        m = m[m != i]
        exact[i] = np.sin(p[m].astype(np.longdouble) - p[i] - np.longdouble(ALPHA)).sum() / len(m)
        sines = np.sin(((p[m] - p[i]) - ALPHA).astype(np.longdouble)).astype(np.float64)
        added[i] = np.cumsum(sines)[-1] / len(m)
    z = np.zeros(3 * n)
    with spc2.Sim(spc2.params("chimera", "fp64", path, n=n, L=1.0, rho=rho, v0=0.01, sigma=1.0, alpha=ALPHA)) as s:
        s.set_state(st)
        got = s.eval_rhs(z, 0.0, 0.01, z)[2::3]

    def rms(a):
        return float(np.sqrt(((a - exact).astype(np.float64) ** 2).mean()))

    assert rms(got) <= rms(added), (rms(got), rms(added))
