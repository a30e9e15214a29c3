"""Where the device linear solve stops without converging: every breakdown of the iteration, on one
workgroup and on more row ranges than a dot product has partials.  Each node's first two free DOFs
carry the same 2 x 2 system, for which the iteration's numbers are exact in floating point, so that
the breakdown is met exactly; the other DOFs have no entries and no load."""
import numpy as np
import pytest
import torch

import pgfem3d_amd as P
from problems import BoxProblem

pytestmark = pytest.mark.gpu

# matrix, load, then by hand: iterations, solution, residual over load
BREAKDOWNS = {
    "rh.v = 0": ((-4, -4, 0, 2), (1, 1), 1, (0, 0), 1.0),
    "rh.v = 0, second iteration": ((-4, -4, -4, -4), (1, 0), 2, (-0.25, 0.125), 0.5 ** 0.5),
    "omega = 0": ((-4, -4, -4, 0), (1, 0), 1, (-0.25, 0), 1.0),
}


@pytest.mark.parametrize("kind", BREAKDOWNS)
@pytest.mark.parametrize("n", [2, 9, 45])
def test_breakdowns(device, kind, n):
    (a, b, c, d), load, its, sol, res = BREAKDOWNS[kind]
    prob = BoxProblem(n, P.PGF_HEX8, P.neo_hookean(70e3, 0.33))
    first = prob.ids[(prob.ids > 0).sum(1) >= 2]
    i = np.sort(np.where(first > 0, first, 1 << 40), axis=1)[:, :2] - 1
    vals, rhs, x = np.zeros(int(prob.Ap[-1])), np.zeros(prob.ndof), np.zeros(prob.ndof)
    for p, q, v in ((0, 0, a), (0, 1, b), (1, 0, c), (1, 1, d)):
        lo, hi = prob.Ap[i[:, p]], prob.Ap[i[:, p] + 1]
        for k in range(int((hi - lo).max())):
            at = np.minimum(lo + k, hi - 1)
            vals[at[prob.Ai[at] == i[:, q]]] = v
    for p in (0, 1):
        rhs[i[:, p]], x[i[:, p]] = load[p], sol[p]
    h = P.Handle(prob.mesh, prob.ids, prob.ndof, prob.Ap, prob.Ai, prob.mats)
    for _ in range(3):
        got = torch.zeros(prob.ndof, dtype=torch.float64, device=device)
        it, rr = h.solve(*(torch.from_numpy(y).to(device) for y in (vals, rhs)), got, tol=1e-12, maxit=50)
        assert it == its and abs(rr - res) <= 1e-14 and np.array_equal(got.cpu().numpy(), x)
    h.close()
