"""A crystal-plasticity pass at displacements that are no numbers fails with nothing of an earlier pass in
its results: the handle that had a good pass before, and the one that had none, return the same."""
import numpy as np
import pytest
import torch

import pgfem3d_amd as P
from problems import CPBoxProblem, fcc_crystal_he

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("law,three_field", [("cubic", False), ("hyperelastic", False), ("hyperelastic", True)])
def test_failed_pass_holds_nothing_of_the_last(device, law, three_field):
    mat = P.fcc_crystal() if law == "cubic" else fcc_crystal_he()
    prob = CPBoxProblem(2, P.PGF_TET10, mat, n_grains=3, seed=5)
    r, defl = prob.displacement(1e-3, 2e-5, seed=1)
    good, dd = torch.from_numpy(r).to(device), torch.from_numpy(defl).to(device)
    bad = good.clone()
    bad[len(r) // 2] = float("nan")
    out = []
    for before in (False, True):
        h = P.Handle(prob.mesh, prob.ids, prob.ndof, prob.Ap, prob.Ai, prob.mats)
        h.set_orientations(prob.R, prob.grain)
        h.set_three_field(three_field)
        f, v = (torch.zeros(n, dtype=torch.float64, device=device) for n in (prob.ndof, h.nnz))
        if before:
            assert h.residual_tangent(f, v, good, defl=dd, dt=1.0) == 0
            h.reset_step()
        err = [h.residual_tangent(f, v, bad, defl=dd, dt=1.0)]
        res = [f.cpu().numpy(), v.cpu().numpy()]
        err.append(h.tangent(v, bad, defl=dd, dt=1.0))
        out.append((err, res + [v.cpu().numpy()]))
        h.close()
    (e0, x0), (e1, x1) = out
    assert e0 == e1 and min(e0) > 0
    for a, b in zip(x0, x1):
        assert np.array_equal(a, b, equal_nan=True)
