"""The gather assembly against the coloured one where its loops end: a fan of m tetrahedra around an
axis, whose end nodes have m staging blocks each (the gather takes 64 at a time, in batches of 4, 8
or 16) and whose ring nodes have two, with nodes of one, two and three free DOFs; fused, tangent
and residual passes.

Tolerance: both modes add the same m element entries, in different orders: m eps of the largest
entry, 130 * 1.1e-16 < 2e-14; 1e-13.
"""
import numpy as np
import pytest
import torch

import pgfem3d_amd as P

TOL = 1e-13

pytestmark = pytest.mark.gpu


def _fan(m):
    t = 2 * np.pi * np.arange(m) / m
    X = np.concatenate([[[0, 0, 1.0], [0, 0, -1.0]], np.stack([np.cos(t), np.sin(t), 0 * t], 1)])
    i = np.arange(m)
    conn = np.stack([0 * i + 1, 2 + i, 2 + (i + 1) % m, 0 * i], 1)
    mesh = P.MeshArrays(X=np.ascontiguousarray(X), elem_ptr=np.arange(0, 4 * m + 1, 4, dtype=np.int64),
                        elem_conn=np.ascontiguousarray(conn.reshape(-1), dtype=np.int64),
                        elem_mat=np.zeros(m, dtype=np.int64))
    free = np.ones((m + 2, 3), dtype=bool)
    free[2::4, 0] = free[3::4, :2] = free[4::8, :] = False
    free[2, :] = False
    ids = np.zeros((m + 2, 3), dtype=np.int64)
    ids[free] = 1 + np.arange(free.sum())
    return mesh, ids, int(free.sum())


@pytest.mark.parametrize("batch", [2, 4, 8])
@pytest.mark.parametrize("m", [3, 4, 5, 7, 8, 9, 15, 16, 17, 63, 64, 65, 130])
def test_fan_of_tets(device, m, batch):
    mesh, ids, ndof = _fan(m)
    Ap, Ai = P.psparse_apai(mesh, ids, ndof)
    r = torch.from_numpy(1e-3 * np.random.default_rng(m).standard_normal(ndof)).to(device)
    out = []
    for mode in (P.ASSEMBLY_GATHER, P.ASSEMBLY_COLOURED):
        h = P.Handle(mesh, ids, ndof, Ap, Ai, [P.j2_linear(70e3, 0.33, 250.0, 1000.0)])
        h.set_assembly(mode)
        h.set_tuning(gather_batch=batch)
        fv = [torch.full((k,), np.nan, dtype=torch.float64, device=device) for k in (ndof, int(Ap[-1])) * 2]
        assert h.residual_tangent(fv[0], fv[1], r) == 0
        assert h.residual(fv[2], r, run_integration=True) == 0
        assert h.tangent(fv[3], r) == 0
        out.append([x.cpu().numpy() for x in fv])
        h.close()
    for a, b in zip(*out):
        assert np.abs(a - b).max() <= TOL * np.abs(b).max()


@pytest.mark.parametrize("graph", [False, True])
def test_failure_counts_belong_to_their_pass(device, graph):
    """Inverted elements are counted by the pass that meets them, eager and replayed, and by no
    later one."""
    mesh, ids, ndof = _fan(9)
    Ap, Ai = P.psparse_apai(mesh, ids, ndof)
    good = torch.zeros(ndof, dtype=torch.float64, device=device)
    bad = good.clone()
    bad[int(ids[0, 2]) - 1] = -2.5  # the upper end node below the lower one: all nine inverted
    h = P.Handle(mesh, ids, ndof, Ap, Ai, [P.neo_hookean(200e3, 0.3)])
    h.set_graph(graph)
    f, buf = torch.empty_like(good), good.clone()
    counts = []
    for r in (good, bad, bad, good, bad, good, good):
        buf.copy_(r)
        torch.cuda.synchronize()
        counts.append(h.residual(f, buf, run_integration=True))
    n = counts[1]
    assert n >= 9 and counts == [0, n, n, 0, n, 0, 0]
    h.close()
