"""The cell build (lists filled at binning, ranks by a thread per particle) and
the stages written by the passes: cell lists bit for bit against a stable sort,
with lists that overflow, on both sides of the histogram scan's place; steps of
one call against single steps, and batched replicas against single handles, bit
for bit."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

import spc2_langevin_integration_amd as spc2  # noqa: E402

pytestmark = pytest.mark.gpu

STEPS = 19  # past a re-homing


def state_of(n, spread, seed=3):
    """Positions in the unit box, or all within `spread` of its centre."""
    rng = np.random.default_rng(seed)
    st = rng.uniform(0.0, 1.0, 3 * n)
    if spread is not None:
        st = 0.5 + spread * (st - 0.5)
    st[2::3] = rng.uniform(0.0, 2 * np.pi, n)
    return st


# cells per side: the fewest, below and above the histograms that the sort sums itself (16384)
@pytest.mark.parametrize("spread", [None, 0.3, 1e-4])
@pytest.mark.parametrize("n", [1, 255, 257, 5003])
@pytest.mark.parametrize("side", [3, 16, 128, 129])
def test_cell_list_is_the_stable_sort(side, n, spread):
    st = state_of(n, spread)
    with spc2.Sim(spc2.params("chimera", "fp64", "cells", n=n, L=1.0, rho=1.0 / (side + 0.5))) as s:
        for _ in range(2):  # both sets of counts
            s.set_state(st)
            cell_of, start, order = s.cell_list()
            c = (st[1::3] * side).astype(int) * side + (st[0::3] * side).astype(int)
            assert np.array_equal(cell_of, c)
            assert np.array_equal(start, np.concatenate([[0], np.cumsum(np.bincount(c, minlength=side * side))]))
            assert np.array_equal(order, np.argsort(c, kind="stable"))


def model(system, prec, n, path, seed=7):
    rho = 0.3 if path == "all_pairs" else 0.09
    kw = dict(n=n, L=1.0, rho=rho, D=0.02, seed=seed)
    if system == "chimera":
        return spc2.params("chimera", prec, path, v0=0.5, sigma=1.3, alpha=1.45, **kw)
    return spc2.params("vortex", prec, path, velocity=0.5, mu_plus=10.0, mu_minus=8.0, xi_a=0.2 * rho, xi_r=0.1 * rho,
                       kappa=2.0, **kw)


@pytest.mark.parametrize("spread", [None, 0.2])
@pytest.mark.parametrize("n", [65, 2049])  # 2049: the matrix-core cells of the FP32 chimera form too
@pytest.mark.parametrize("method", ["se", "srk", "rk4"])
@pytest.mark.parametrize("path", ["cells", "all_pairs"])
@pytest.mark.parametrize("prec", ["fp64", "fp32k", "fp64f"])
@pytest.mark.parametrize("system", ["chimera", "vortex"])
def test_steps_of_one_call_are_single_steps(system, prec, path, method, n, spread):
    st, out = state_of(n, spread), []
    for calls in (1, STEPS):
        with spc2.Sim(model(system, prec, n, path)) as s:
            s.set_state(st)
            for q in range(calls):
                s.step(method, 0.01, q * (STEPS // calls), STEPS // calls)
            out.append(s.get_state())
    assert np.isfinite(out[0]).all()
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("method", ["se", "srk"])
@pytest.mark.parametrize("prec", ["fp64", "fp32k"])
def test_clustered_replicas_are_single_handles(prec, method):
    sizes, spreads = [700, 65, 2049, 3], [0.05, None, 0.2, 1e-3]
    reps = [model(("chimera", "vortex")[q % 2], prec, n, "auto", seed=q) for q, n in enumerate(sizes)]
    reps.append(spc2.params("chimera", prec, "auto", n=90, L=1.0, rho=0.3, v0=0.5, seed=9))  # all pairs
    states = [state_of(p.n, sp, seed=p.n) for p, sp in zip(reps, spreads + [None])]
    with spc2.Batch(reps) as b:
        for r, st in enumerate(states):
            b.set_state(r, st)
        b.step(0.01, STEPS, method=method)
        got = [b.get_state(r) for r in range(len(reps))]
    for r, (p, st) in enumerate(zip(reps, states)):
        with spc2.Sim(p) as s:
            s.set_state(st)
            s.step(method, 0.01, 0, STEPS)
            assert np.array_equal(got[r], s.get_state()), f"replica {r}"


# both sides of the chunk lengths of the matrix-core passes (32, 64, 128, 256 slots); a batch's are 256
@pytest.mark.parametrize("method", ["se", "srk"])
@pytest.mark.parametrize("n", [16384, 16385, 32769, 65537, 131073])
def test_chunk_length_leaves_the_bits(n, method):
    L = float(np.sqrt(n / 4000.0))
    p = spc2.params("chimera", "fp32k", "auto", n=n, L=L, rho=0.1, v0=0.01, sigma=1.0, alpha=1.45, D=0.01, seed=3)
    st = state_of(n, None)
    st[0::3] *= L
    st[1::3] *= L
    with spc2.Batch([p]) as b, spc2.Sim(p) as s:
        b.set_state(0, st)
        b.step(0.01, 3, method=method)
        s.set_state(st)
        s.step(method, 0.01, 0, 3)
        assert np.array_equal(b.get_state(0), s.get_state())


@pytest.mark.parametrize("n", [1, 255, 257, 5003])
@pytest.mark.parametrize("path", ["cells", "all_pairs", "verlet"])
def test_state_goes_up_and_comes_back(path, n):
    st = state_of(n, None, seed=n)
    with spc2.Sim(model("chimera", "fp64", n, path)) as s:
        s.set_state(st)
        assert np.array_equal(s.get_state(), st)
    with spc2.Batch([model("chimera", "fp64", n, "auto"), model("vortex", "fp64", 7, "auto")]) as b:
        b.set_state(0, st)
        assert np.array_equal(b.get_state(0), st)


# the FP32 vortex pass 2 that finds the near partners first, against its walk over the global tiles: no, few and
# many partners (more words of bits than are kept at once, full cohesion queues), boxes that wrap
@pytest.mark.parametrize("spread", [None, 0.5, 0.12])
@pytest.mark.parametrize("n", [1, 65, 700, 2049])
@pytest.mark.parametrize("rho", [0.24, 0.09])
def test_near_partners_first_leaves_the_bits(monkeypatch, rho, n, spread):
    out = []
    for cap in (None, "0"):
        if cap is not None:
            monkeypatch.setenv("SPC2_LDS_CAP", cap)
        p = spc2.params("vortex", "fp32k", "cells", n=n, L=1.0, rho=rho, D=0.02, seed=5, velocity=0.1, mu_plus=10.0,
                        mu_minus=8.0, xi_a=0.4 * rho, xi_r=0.3 * rho, kappa=2.0)
        with spc2.Sim(p) as s:
            s.set_state(state_of(n, spread))
            rhs = s.eval_rhs_ito()
            s.step("srk", 0.005, 0, 2)
            out.append((*rhs, s.get_state()))
    for a, b in zip(*out):
        assert np.isfinite(a).all()
        assert np.array_equal(a, b)
