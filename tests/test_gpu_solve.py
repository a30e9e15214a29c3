"""The device linear solve (pgf_solve) against a sparse direct solve on the host, at the sizes
where its row ranges end: fewer rows than one 256-row range, ranges that cut a node's rows, and
more ranges than a dot product has partials."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

import pgfem3d_amd as P
from problems import BoxProblem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("etype,n", [(P.PGF_TET4, 1), (P.PGF_TET4, 3), (P.PGF_HEX8, 4), (P.PGF_TET10, 3), (P.PGF_HEX8, 45)])
def test_solution_and_residual(device, etype, n):
    import torch

    prob = BoxProblem(n, etype, P.neo_hookean(70e3, 0.33))
    h = P.Handle(prob.mesh, prob.ids, prob.ndof, prob.Ap, prob.Ai, prob.mats)
    r, defl = prob.displacement(0.01, 0.002 / n, seed=3)
    f = torch.empty(prob.ndof, dtype=torch.float64, device=device)
    vals = torch.empty(h.nnz, dtype=torch.float64, device=device)
    assert h.residual_tangent(f, vals, torch.from_numpy(r).to(device), defl=torch.from_numpy(defl).to(device)) == 0
    K = sp.csr_matrix((vals.cpu().numpy(), prob.Ai, prob.Ap), shape=(prob.ndof, prob.ndof))
    b = np.random.default_rng(1).standard_normal(prob.ndof)
    x = torch.zeros(prob.ndof, dtype=torch.float64, device=device)
    tol = 1e-10
    its, res = h.solve(vals, torch.from_numpy(b).to(device), x, tol=tol, maxit=20000)
    assert res <= tol and its >= 1
    # the recurrence's residual drifts from the true one by rounding only
    true = np.linalg.norm(b - K @ x.cpu().numpy()) / np.linalg.norm(b)
    assert true <= 10 * tol
    if prob.ndof < 5000:
        want = spla.spsolve(K.tocsc(), b)
        # |dx| / |x| <= cond |r| / |b|
        assert np.linalg.norm(x.cpu().numpy() - want) <= np.linalg.cond(K.toarray()) * 10 * tol * np.linalg.norm(want)
    # from the solution the solve stops before its first iteration; a zero load gives zero
    assert h.solve(vals, torch.from_numpy(b).to(device), x, tol=100 * tol, maxit=10)[0] == 0
    z = torch.zeros_like(x)
    assert h.solve(vals, torch.zeros_like(x), z, tol=tol, maxit=10) == (0, 0.0) and not z.any()
    # the iteration cap: what was reached, and its residual
    its, res = h.solve(vals, torch.from_numpy(b).to(device), z, tol=1e-300, maxit=3)
    assert its == 3 and abs(np.linalg.norm(b - K @ z.cpu().numpy()) / np.linalg.norm(b) - res) <= 1e-10 * res
    h.close()
