"""The forms of the crystal-plasticity local solve against the CPU oracle: the flow rule's exponent
1/m - 1 whole or not, the saturation stress constant or rate-dependent (w), both elastic laws, point
counts around the 64 of a wave, and steps so large that dt lambda pJ leaves the range of the
tangent's series (0.01) and the points take the pivoted 9 x 9 system, alone or beside points that do
not.

Tolerance: the stress of the elastic intermediate configuration carries round-off of C eps / tau =
1.7e5 * 1.1e-16 / 16 = 1e-12 relative to tau, which the flow rule takes into the tangent times
1/m <= 20: 2e-11.  1e-10 relative in the infinity norm of each array and of each CSR row.
"""
import numpy as np
import pytest
import torch

import oracle as O
import pgfem3d_amd as P
from conftest import rel_csr_rows, rel_inf
from problems import CPBoxProblem, fcc_crystal_he

TOL = 1e-10

pytestmark = pytest.mark.gpu


def _step(prob, h, st, device, stretch, seed):
    r, defl = prob.displacement(stretch, 2e-5, seed=seed)
    rd, dd = (torch.from_numpy(np.ascontiguousarray(x)).to(device) for x in (r, defl))
    f = torch.empty(prob.ndof, dtype=torch.float64, device=device)
    vals = torch.empty(int(prob.Ap[-1]), dtype=torch.float64, device=device)
    err = h.residual_tangent(f, vals, rd, defl=dd, dt=1.0)
    fo, vo, erro = prob.assemble(st, r, defl, dt=1.0)
    assert err == erro == 0
    assert rel_inf(f.cpu().numpy(), fo) < TOL
    assert rel_inf(vals.cpu().numpy(), vo) < TOL
    assert rel_csr_rows(vals.cpu().numpy(), vo, prob.Ap) < TOL
    assert rel_inf(h.get_state(P.STATE_PLASTIC_NP1), st.pF_np1) < TOL
    assert rel_inf(h.get_state(P.STATE_SCALAR_NP1)[0], st.g_np1) < TOL
    assert rel_inf(h.get_state(P.STATE_TAU), st.tau) < TOL


def _setup(n, etype, law, **kw):
    mat = P.fcc_crystal(**kw) if law == "cubic" else fcc_crystal_he(**kw)
    prob = CPBoxProblem(n, etype, mat, n_grains=3, seed=5)
    h = P.Handle(prob.mesh, prob.ids, prob.ndof, prob.Ap, prob.Ai, prob.mats)
    h.set_orientations(prob.R, prob.grain)
    return prob, h, O.CPState(prob.nqp, mat.g0)


@pytest.mark.parametrize("law", ["cubic", "hyperelastic"])
@pytest.mark.parametrize("flow", [dict(m=0.07), dict(m=0.05, w=0.1), dict(m=0.07, w=0.1), dict(m=0.1)],
                         ids=["fraction", "whole-w", "fraction-w", "whole"])
@pytest.mark.parametrize("n,etype", [(1, P.PGF_TET4), (2, P.PGF_TET4), (2, P.PGF_TET10), (2, P.PGF_HEX8)])
def test_flow_rules(device, law, flow, n, etype):
    """6 (one ragged wave), 48, 192 (whole waves) and 64 points, elastic to plastic in six steps."""
    prob, h, st = _setup(n, etype, law, **flow)
    for s in range(1, 7):
        _step(prob, h, st, device, 1.5e-4 * s, seed=s)
        h.commit_step()
        st.commit()
    assert np.abs(st.gdot).max() > 1e-5
    h.close()


@pytest.mark.parametrize("law", ["cubic", "hyperelastic"])
@pytest.mark.parametrize("m,stretch,some", [(0.3, 0.3, True), (0.3, 0.5, False), (0.5, 0.5, False)])
def test_pivoted_tangent_at_large_steps(device, law, m, stretch, some):
    prob, h, st = _setup(2, P.PGF_TET4, law, m=m)
    _step(prob, h, st, device, stretch, seed=1)
    lp = np.abs(st.lam_np1 * np.linalg.det(st.pF_np1.T.reshape(-1, 3, 3)))
    assert (lp > 0.01).any() and (lp < 0.01).any() == some
    h.close()


@pytest.mark.parametrize("etype,n", [(P.PGF_TET4, 2), (P.PGF_TET10, 2), (P.PGF_HEX8, 2)])
def test_three_field_initial_gradients(device, etype, n):
    """pgf_tf_initial stores F at n and n-1 of the given displacements: an integrating pass's F at
    them."""
    prob, h, _ = _setup(n, etype, "hyperelastic")
    h3 = P.Handle(prob.mesh, prob.ids, prob.ndof, prob.Ap, prob.Ai, prob.mats)
    h3.set_orientations(prob.R, prob.grain)
    h3.set_three_field(True)
    f = torch.empty(prob.ndof, dtype=torch.float64, device=device)
    args, F = [], []
    for s in (2e-3, 1e-3):
        r, defl = prob.displacement(s, 2e-4, seed=3)
        rd, dd = (torch.from_numpy(np.ascontiguousarray(x)).to(device) for x in (r, defl))
        h.residual(f, rd, defl=dd, dt=1.0)
        F.append(h.get_state(P.STATE_F_NP1).copy())
        args += [rd, dd]
    h3.tf_initial(*args)
    for fld, ref in ((P.STATE_F_N, F[0]), (P.STATE_F_NM1, F[1])):
        assert np.abs(ref - np.eye(3).reshape(9, 1)).max() > 1e-4
        assert np.abs(h3.get_state(fld) - ref).max() < 1e-15
    h3.close()
    h.close()


def test_work_queue_gives_the_ranges_results(device):
    """146,334 points, enough for the local Newton's global queue: which wave and lane solves a point,
    and beside which others, leaves no trace in its state."""
    prob = CPBoxProblem(29, P.PGF_TET4, P.fcc_crystal(), n_grains=3, seed=5)
    out = []
    for chunk in (1, 64, 192):
        h = P.Handle(prob.mesh, prob.ids, prob.ndof, prob.Ap, prob.Ai, prob.mats)
        h.set_orientations(prob.R, prob.grain)
        h.set_tuning(cp_chunk=chunk)
        f = torch.empty(prob.ndof, dtype=torch.float64, device=device)
        for s in (1, 2):
            r, defl = prob.displacement(6e-4 * s, 2e-5, seed=s)
            rd, dd = (torch.from_numpy(np.ascontiguousarray(x)).to(device) for x in (r, defl))
            assert h.residual(f, rd, defl=dd, dt=1.0) == 0
            h.commit_step()
        out.append([h.get_state(k) for k in (P.STATE_PLASTIC_N, P.STATE_SCALAR_N, P.STATE_ITERS)])
        h.close()
    assert out[0][2].max() > 3
    for o in out[1:]:
        for a, b in zip(out[0], o):
            assert np.array_equal(a, b)
