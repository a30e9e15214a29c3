"""Crystal plasticity's local systems with partial pivoting (pgf_set_pivoting): at bounds that no, some
or all lanes of a wave exceed, in the Newton steps and in the tangent, against the CPU oracle, in the
displacement and the three-field form, from plain and from callers' starts.

Tolerance: that of test_gpu_cp_flow.py, 1e-10 relative.  The iterations end when a step is below 1e-12,
so the two eliminations, which differ by rounding, take the same number of steps or one more."""
import numpy as np
import pytest
import torch

import oracle as O
import pgfem3d_amd as P
from conftest import rel_csr_rows, rel_inf
from problems import CPBoxProblem, fcc_crystal_he

TOL = 1e-10
BOUNDS = {"none": (1e300, 1e300), "some": (2.0, 0.5), "step": (0.0, 1e300), "tangent": (1e300, 0.0), "all": (0.0, 0.0)}

pytestmark = pytest.mark.gpu


def _dev(x, device):
    return torch.from_numpy(np.ascontiguousarray(x)).to(device)


@pytest.mark.parametrize("law", ["cubic", "hyperelastic"])
@pytest.mark.parametrize("flow", [dict(), dict(m=0.07), dict(m=0.05, w=0.1)], ids=["whole", "fraction", "whole-w"])
@pytest.mark.parametrize("n,etype", [(1, P.PGF_TET4), (3, P.PGF_TET4), (2, P.PGF_HEX8)])
def test_every_bound_against_the_oracle(device, law, flow, n, etype):
    """6, 162 (two and a half waves) and 64 points."""
    mat = P.fcc_crystal(**flow) if law == "cubic" else fcc_crystal_he(**flow)
    prob = CPBoxProblem(n, etype, mat, n_grains=3, seed=5)
    f = torch.empty(prob.ndof, dtype=torch.float64, device=device)
    vals = torch.empty(int(prob.Ap[-1]), dtype=torch.float64, device=device)
    states = {}
    for kind, bounds in BOUNDS.items():
        h = P.Handle(prob.mesh, prob.ids, prob.ndof, prob.Ap, prob.Ai, prob.mats)
        h.set_orientations(prob.R, prob.grain)
        h.set_pivoting(*bounds)
        h.set_graph(kind == "some")
        st = O.CPState(prob.nqp, mat.g0)
        for s in range(1, 5):
            r, defl = prob.displacement(2.5e-4 * s, 2e-5, seed=s)
            rd, dd = _dev(r, device), _dev(defl, device)
            err = h.residual_tangent(f, vals, rd, defl=dd, dt=1.0)
            fo, vo, erro = prob.assemble(st, r, defl, dt=1.0)
            assert err == erro == 0
            assert rel_inf(f.cpu().numpy(), fo) < TOL
            assert rel_csr_rows(vals.cpu().numpy(), vo, prob.Ap) < TOL
            assert rel_inf(h.get_state(P.STATE_PLASTIC_NP1), st.pF_np1) < TOL
            assert rel_inf(h.get_state(P.STATE_TAU), st.tau) < TOL
            its = h.get_state(P.STATE_ITERS).copy()
            states[kind, s] = h.get_state(P.STATE_PLASTIC_NP1).copy(), vals.cpu().numpy(), its
            assert np.abs(its - states["none", s][2]).max() <= 1
            h.commit_step()
            st.commit()
        h.close()
    # the bounds select what they say: another elimination leaves another rounding
    x, K, _ = zip(*(states[kind, 4] for kind in BOUNDS))
    same = lambda v, a, b: np.array_equal(v[list(BOUNDS).index(a)], v[list(BOUNDS).index(b)])  # noqa: E731
    assert same(x, "none", "tangent") and same(x, "step", "all") and not same(x, "none", "step")
    assert not same(K, "none", "tangent") and not same(K, "step", "all")
    assert not same(x, "some", "none")
    if prob.nqp > 6:  # six points may all exceed it
        assert not same(x, "some", "all")


@pytest.mark.parametrize("etype,n", [(P.PGF_TET4, 3), (P.PGF_TET10, 2), (P.PGF_HEX8, 2)])
def test_three_field(device, etype, n):
    mat = fcc_crystal_he()
    prob = CPBoxProblem(n, etype, mat, n_grains=4, seed=2)
    rng = np.random.default_rng(7)
    f = torch.zeros(prob.ndof, dtype=torch.float64, device=device)
    vals = torch.zeros(int(prob.Ap[-1]), dtype=torch.float64, device=device)
    for bounds in BOUNDS.values():
        h = P.Handle(prob.mesh, prob.ids, prob.ndof, prob.Ap, prob.Ai, prob.mats)
        h.set_orientations(prob.R, prob.grain)
        h.set_three_field(True)
        h.set_pivoting(*bounds)
        st = O.CPState(prob.nqp, mat.g0)
        r, defl = prob.displacement(1.2e-3, 2e-5, seed=1)
        theta = 1.0 + 2e-4 * rng.standard_normal(prob.mesh.n_elem)
        Pe = 60.0 * rng.standard_normal(prob.mesh.n_elem)
        for fld, v in ((P.TF_V_NP1, theta), (P.TF_P_NP1, Pe), (P.TF_DV, 0 * theta), (P.TF_DP, 0 * Pe)):
            h.tf_set(fld, v)
        assert h.residual_tangent(f, vals, _dev(r, device), defl=_dev(defl, device)) == 0
        fo, vo, err = O.assemble_cp_tf(prob.mesh, prob.mats, prob.grain, prob.gP, prob.gL, prob.ids, prob.ndof,
                                       prob.Ap, prob.Ai, st, theta, Pe, r, defl=defl)
        assert err == 0 and np.abs(st.gdot).max() > 1e-5
        assert rel_inf(f.cpu().numpy(), fo) < TOL
        assert rel_inf(vals.cpu().numpy(), vo) < TOL
        assert rel_inf(h.get_state(P.STATE_PLASTIC_NP1), st.pF_np1) < TOL
        h.close()


def test_callers_starts_and_failures(device):
    """Starts far off, beside good ones, and points that do not converge in the iterations they have:
    the same points solved from the same start, the same failures counted, at every bound."""
    mat = P.fcc_crystal(max_itr=7)
    prob = CPBoxProblem(3, P.PGF_TET4, mat, n_grains=3, seed=5)
    r, defl = prob.displacement(2e-3, 2e-5, seed=1)
    rd, dd = _dev(r, device), _dev(defl, device)
    f = torch.empty(prob.ndof, dtype=torch.float64, device=device)
    rng = np.random.default_rng(3)
    warm = np.zeros((11, prob.nqp))
    warm[:9] = np.eye(3).reshape(9, 1) + 4e-3 * rng.standard_normal((9, prob.nqp)) * (np.arange(prob.nqp) % 3)
    warm[10] = 17.0
    w = _dev(warm, device)
    out = []
    for bounds in BOUNDS.values():
        h = P.Handle(prob.mesh, prob.ids, prob.ndof, prob.Ap, prob.Ai, prob.mats)
        h.set_orientations(prob.R, prob.grain)
        h.set_pivoting(*bounds)
        h.set_warm_start(w)
        err = h.residual(f, rd, defl=dd, dt=1.0)
        its = h.get_state(P.STATE_ITERS).astype(np.int64)
        out.append((err, its >> 24, h.get_state(P.STATE_PLASTIC_NP1).copy()))
        h.close()
    assert 0 < out[0][0] < prob.nqp
    for err, kind, x in out[1:]:
        assert err == out[0][0] and np.array_equal(kind, out[0][1])
        assert np.abs(x - out[0][2]).max() < TOL


def test_pivoting_leaves_no_trace_of_the_neighbours(device):
    """146,334 points: a point's result does not depend on the lanes that pivot beside it."""
    prob = CPBoxProblem(29, P.PGF_TET4, P.fcc_crystal(), n_grains=3, seed=5)
    out = []
    for chunk in (1, 64, 192):
        h = P.Handle(prob.mesh, prob.ids, prob.ndof, prob.Ap, prob.Ai, prob.mats)
        h.set_orientations(prob.R, prob.grain)
        h.set_tuning(cp_chunk=chunk)
        h.set_pivoting(2.0, 0.5)
        f = torch.empty(prob.ndof, dtype=torch.float64, device=device)
        for s in (1, 2):
            r, defl = prob.displacement(6e-4 * s, 2e-5, seed=s)
            assert h.residual(f, _dev(r, device), defl=_dev(defl, device), dt=1.0) == 0
            h.commit_step()
        out.append([h.get_state(k) for k in (P.STATE_PLASTIC_N, P.STATE_SCALAR_N, P.STATE_ITERS)])
        h.close()
    for o in out[1:]:
        for a, b in zip(out[0], o):
            assert np.array_equal(a, b)


def test_bounds_are_checked(device):
    prob = CPBoxProblem(1, P.PGF_TET4, P.fcc_crystal(), n_grains=1, seed=5)
    h = P.Handle(prob.mesh, prob.ids, prob.ndof, prob.Ap, prob.Ai, prob.mats)
    for bad in ((-1.0, 1.0), (1.0, -1.0), (float("nan"), 1.0), (1.0, float("nan"))):
        with pytest.raises(P.PGFError):
            h.set_pivoting(*bad)
    h.close()
