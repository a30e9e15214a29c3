"""Grain orientations that are no rotations to the last bit -- rounded to single precision, or written
with few digits -- stand for the nearest rotation: results against the CPU oracle at that rotation.
The local solve works in the crystal frame, where an R with R^T R != I would leave that difference,
times stiffness over slip resistance (1e4), in the stress.

Tolerance: that of test_gpu_cp_flow.py, 1e-10 relative."""
import numpy as np
import pytest
import torch

import oracle as O
import pgfem3d_amd as P
from conftest import rel_csr_rows, rel_inf
from problems import CPBoxProblem, fcc_crystal_he

TOL = 1e-10

pytestmark = pytest.mark.gpu


def _nearest(R):
    u, _, vt = np.linalg.svd(R)
    return u @ vt


@pytest.mark.parametrize("law", ["cubic", "hyperelastic"])
@pytest.mark.parametrize("given", ["as made", "single precision", "four digits", "scaled", "improper"])
def test_orientation_stands_for_the_nearest_rotation(device, law, given):
    mat = P.fcc_crystal() if law == "cubic" else fcc_crystal_he()
    prob = CPBoxProblem(2, P.PGF_TET10, mat, n_grains=3, seed=5)
    R = {"as made": lambda R: R, "single precision": lambda R: R.astype(np.float32).astype(np.float64),
         "four digits": lambda R: np.round(R, 4), "scaled": lambda R: 1.25 * R, "improper": lambda R: -R}[given](prob.R)
    tabs = [O.cp_grain(mat, _nearest(Q)) for Q in R.reshape(-1, 3, 3)]
    prob.gP = np.ascontiguousarray(np.stack([t[0] for t in tabs]).reshape(3, 108))
    prob.gL = np.ascontiguousarray(np.stack([t[1] for t in tabs]).reshape(3, 81))
    h = P.Handle(prob.mesh, prob.ids, prob.ndof, prob.Ap, prob.Ai, prob.mats)
    h.set_orientations(R, prob.grain)
    st = O.CPState(prob.nqp, mat.g0)
    f = torch.empty(prob.ndof, dtype=torch.float64, device=device)
    vals = torch.empty(int(prob.Ap[-1]), dtype=torch.float64, device=device)
    for s in range(1, 6):
        r, defl = prob.displacement(2e-4 * s, 2e-5, seed=s)
        rd, dd = (torch.from_numpy(np.ascontiguousarray(x)).to(device) for x in (r, defl))
        err = h.residual_tangent(f, vals, rd, defl=dd, dt=1.0)
        fo, vo, erro = prob.assemble(st, r, defl, dt=1.0)
        assert err == erro == 0
        assert rel_inf(f.cpu().numpy(), fo) < TOL
        assert rel_csr_rows(vals.cpu().numpy(), vo, prob.Ap) < TOL
        assert rel_inf(h.get_state(P.STATE_PLASTIC_NP1), st.pF_np1) < TOL
        assert rel_inf(h.get_state(P.STATE_TAU), st.tau) < TOL
        h.commit_step()
        st.commit()
    assert np.abs(st.gdot).max() > 1e-5
    h.close()
