"""The device linear solve takes any CSR pattern of the handle's row lengths: a node's rows with their
columns in other orders, and with other columns, give the solution of the matrix that they describe."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla
import torch

import pgfem3d_amd as P
from problems import BoxProblem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["same", "reversed", "other column"])
@pytest.mark.parametrize("etype,n", [(P.PGF_TET4, 4), (P.PGF_HEX8, 6)])
def test_rows_of_a_node_with_their_own_columns(device, kind, etype, n):
    prob = BoxProblem(n, etype, P.neo_hookean(70e3, 0.33))
    Ap, Ai = prob.Ap, prob.Ai.copy()
    rng = np.random.default_rng(4)
    full = prob.ids[(prob.ids > 0).all(1)]
    for row in (full[:, 1] - 1 if kind != "same" else []):  # the second of each node's three rows
        lo, hi = Ap[row], Ap[row + 1]
        if kind == "reversed":
            Ai[lo:hi] = Ai[lo:hi][::-1]
        else:
            k = lo + int(np.flatnonzero(Ai[lo:hi] != row)[0])
            Ai[k] = np.setdiff1d(np.arange(prob.ndof), Ai[lo:hi])[0]
    rows = np.repeat(np.arange(prob.ndof), np.diff(Ap))
    vals = rng.standard_normal(len(Ai))
    vals[Ai == rows] = 2.0 * np.diff(Ap).max()  # diagonally dominant
    K = sp.csr_matrix((vals, Ai, Ap), shape=(prob.ndof,) * 2)
    b = rng.standard_normal(prob.ndof)
    want = spla.spsolve(K.tocsc(), b)
    h = P.Handle(prob.mesh, prob.ids, prob.ndof, Ap, Ai, prob.mats)
    x = torch.zeros(prob.ndof, dtype=torch.float64, device=device)
    _, res = h.solve(*(torch.from_numpy(y).to(device) for y in (vals, b)), x, tol=1e-13, maxit=200)
    # a diagonally dominant matrix: |dx| <= 2 |K^-1| |b| res <= 4 |b| / diag * res
    assert res <= 1e-13 and np.abs(x.cpu().numpy() - want).max() <= 1e-12 * np.abs(want).max()
    h.close()
