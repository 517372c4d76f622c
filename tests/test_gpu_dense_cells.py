"""Cells of more particles than the staged halos hold, or of hardly any, at the
fillings where the choice of walk changes, against the oracle and with every walk over the global
tiles, bit for bit; batched replicas against single handles.  Bars: tests/_parity.py."""
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

DT, SIDE = 0.005, 5


def systems(system, prec, filling, side=SIDE, seed=5):
    n, rho = int(filling * side * side), 1.0 / (side + 0.02)
    if system == "chimera":
        kw = dict(n=n, rho=rho, v0=0.05, sigma=1.3, alpha=1.45, D=0.02)
        return spc2.params("chimera", prec, "auto", L=1.0, seed=seed, **kw), O.chimera(L=1.0, threads=8, **kw)
    kw = dict(rho=rho, velocity=0.025, mu_plus=100.0, mu_minus=80.0, xi_a=0.2 * rho, xi_r=0.1 * rho, kappa=20.0, D=0.02)
    return (spc2.params("vortex", prec, "auto", n=n, L=1.0, seed=seed, **kw),
            O.vortex(n, 1.0, threads=8, **kw))


def state_of(n, clump=0.0):
    rng = np.random.default_rng(n)
    st = rng.uniform(0.0, 1.0, 3 * n)
    k = int(clump * n)  # that share of the particles in a fifth of the box's height
    st[1:3 * k:3] = rng.uniform(0.3, 0.5, k)
    st[2::3] = rng.uniform(0.0, 2 * np.pi, n)
    return st


def compare(monkeypatch, system, prec, filling, clump, side=SIDE):
    p, orc = systems(system, prec, filling, side)
    st = state_of(p.n, clump)
    z = np.zeros(3 * p.n)
    U = np.random.default_rng(1).standard_normal(2 * p.n)
    out = []
    for cap in (None, "0"):
        if cap is not None:
            monkeypatch.setenv("SPC2_LDS_CAP", cap)
        with spc2.Sim(p) as s:
            s.set_state(st)
            s.set_counting(True)
            out.append([s.eval_rhs(z, 0.0, DT, z), s.counts(), *s.eval_rhs_ito()])
            s.step("srk", DT, 0, 1, noise=U)
            out[-1].append(s.get_state())
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    got, cnt, _, ga, after = out[0]
    what = f"{system} {prec} {filling} per cell"
    ref, rc, scale = O.rhs_k(orc, st, z, 0.0, DT, z, term_scale=True)
    assert_rhs_terms(got, ref, scale, p.v0, TOL[prec], what)
    assert np.array_equal(cnt, rc), (cnt, rc)
    _, ra, _ = O.rhs_ito(orc, st)
    for c in (0, 1):
        err = np.abs(ga[c::2] - ra[c::2]).max()
        assert err <= TOL[prec] * np.abs(ra[c::2]).max(), f"{what}: additional[{c}] {err:.3e}"
    assert_state(after, O.step_srk(orc, st, DT, U), st, 1.0, TOL[prec], what)


# chunks of 256, 128, 64 and 32 slots, the last filling of the matrix-core passes and the first beyond
@pytest.mark.parametrize("filling,clump", [(145, 0.0), (165, 0.0), (200, 0.0), (213, 0.0), (215, 0.0), (300, 0.0),
                                           (60, 0.6), (130, 0.6)])
def test_dense_chimera_cells(monkeypatch, filling, clump):
    compare(monkeypatch, "chimera", "fp32k", filling, clump)


# the FP64 forms' lanes per particle in sparse cells: 1, 2, 4, 8 and 16 of them; a system of 16384 in dense cells
@pytest.mark.parametrize("filling,side", [(0.3, 15), (1.1, 15), (1.4, 15), (2.6, 15), (5.5, 15), (9.5, 15), (172, 10)])
@pytest.mark.parametrize("prec", ["fp64", "fp64f"])
@pytest.mark.parametrize("system", ["chimera", "vortex"])
def test_sparse_fp64_cells(monkeypatch, system, prec, filling, side):
    compare(monkeypatch, system, prec, filling, 0.0, side)


@pytest.mark.parametrize("method", ["se", "srk"])
@pytest.mark.parametrize("prec", ["fp64", "fp64f"])
def test_sparse_batch_equals_single(prec, method):
    reps = [systems(("chimera", "vortex")[k % 2], prec, f, 12 + k % 5, seed=20 + k)[0]
            for k, f in enumerate([0.3, 0.3, 1.3, 1.3, 2.7, 2.7, 6.0, 6.0, 175, 175])]
    with spc2.Batch(reps) as b:
        b.init_random_state(0.1)
        b.step(DT, 3, method=method)
        got = [b.get_state(r) for r in range(len(reps))]
    for p, g in zip(reps, got):
        with spc2.Sim(p) as s:
            s.init_random_state(0.1)
            s.step(method, DT, 0, 3)
            assert np.array_equal(s.get_state(), g), f"n={p.n}"


@pytest.mark.parametrize("method", ["se", "srk"])
def test_dense_batch_equals_single(method):
    reps = [systems("chimera", "fp32k", f, seed=20 + k)[0] for k, f in enumerate([10, 40, 150, 180, 212, 216, 260])]
    with spc2.Batch(reps) as b:
        b.init_random_state(0.1)
        b.step(DT, 3, method=method)
        got = [b.get_state(r) for r in range(len(reps))]
    for p, g in zip(reps, got):
        with spc2.Sim(p) as s:
            s.init_random_state(0.1)
            s.step(method, DT, 0, 3)
            assert np.array_equal(s.get_state(), g), f"n={p.n}"


# both sides of the filling from which pass 2 no longer finds the near partners first; what 2560 candidates hold
@pytest.mark.parametrize("filling,clump", [(41, 0.0), (43, 0.0), (60, 0.6), (145, 0.0), (170, 0.0), (300, 0.0)])
def test_dense_vortex_cells(monkeypatch, filling, clump):
    compare(monkeypatch, "vortex", "fp32k", filling, clump)


# the FP64 forms: both sides of the filling from which the factored one takes a lane per particle; halos beyond the LDS
@pytest.mark.parametrize("filling,clump", [(60, 0.6), (165, 0.0), (175, 0.0), (300, 0.0)])
@pytest.mark.parametrize("prec", ["fp64", "fp64f"])
@pytest.mark.parametrize("system", ["chimera", "vortex"])
def test_dense_fp64_cells(monkeypatch, system, prec, filling, clump):
    compare(monkeypatch, system, prec, filling, clump)


# overfull cells side by side in one wavefront and whole wavefronts in one cell (homes in id order, then in cell order)
@pytest.mark.parametrize("spots,share", [(1, 1.0), (3, 0.9), (40, 0.5), (300, 0.5)])
@pytest.mark.parametrize("side", [4, 100])
def test_overfull_cells_are_sorted(side, spots, share):
    n = 20011
    rng = np.random.default_rng(spots)
    st = rng.uniform(0.0, 1.0, 3 * n)
    k = int(share * n)
    at = rng.uniform(0.05, 0.95, (spots, 2))[rng.integers(0, spots, k)]
    for c in (0, 1):
        st[c:3 * k:3] = at[:, c] + 1e-3 * rng.uniform(-1.0, 1.0, k)
    st = st.reshape(n, 3)[rng.permutation(n)].ravel()
    c = (st[1::3] * side).astype(int) * side + (st[0::3] * side).astype(int)
    with spc2.Sim(spc2.params("chimera", "fp64", "cells", n=n, L=1.0, rho=1.0 / (side + 0.5))) as s:
        for _ in range(3):
            s.set_state(st)
            cell_of, start, order = s.cell_list()
            assert np.array_equal(cell_of, c)
            assert np.array_equal(start, np.concatenate([[0], np.cumsum(np.bincount(c, minlength=side * side))]))
            assert np.array_equal(order, np.argsort(c, kind="stable"))
