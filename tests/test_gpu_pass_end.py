"""The end of a pass: its failure count and its results belong to it alone, whatever the handle did
before.  A pass is given up after its launches are queued when an earlier call of the program has left
a HIP error; the pass that follows waits for it and returns its own count and results, bit for bit
those of an undisturbed pass."""
import numpy as np
import pytest
import torch

import pgfem3d_amd as P
from problems import BoxProblem

pytestmark = pytest.mark.gpu


def _problem(device):
    prob = BoxProblem(11, P.PGF_TET10, P.j2_linear(70e3, 0.33, 250.0, 1000.0))
    h = P.Handle(prob.mesh, prob.ids, prob.ndof, prob.Ap, prob.Ai, prob.mats)
    r, defl = prob.displacement(0.012, 2e-4, seed=3)
    good = torch.from_numpy(r).to(device)
    return prob, h, good, -200.0 * good, torch.from_numpy(defl).to(device)  # the second: inverted elements


def _vectors(h, prob, device):
    f = torch.full((prob.ndof,), np.nan, dtype=torch.float64, device=device)
    return f, torch.full((h.nnz,), np.nan, dtype=torch.float64, device=device)


@pytest.mark.parametrize("mode", ["eager", "graph", "static"])
def test_pass_after_one_given_up(device, mode):
    prob, h, good, bad, defl = _problem(device)  # staging that fits the static form
    h.set_graph(mode == "graph")
    call = h.residual_tangent_static if mode == "static" else h.residual_tangent
    ref, lost, out = (_vectors(h, prob, device) for _ in range(3))
    assert call(*lost, bad, defl=defl) > 0
    assert call(*ref, good, defl=defl) == 0
    assert call(*out, good, defl=defl) == 0
    for x in out:
        x.fill_(np.nan)
    torch.cuda.synchronize()
    assert P.lib().hipSetDevice(1 << 20) != 0  # no such device: the error stays for the next look at it
    with pytest.raises(P.PGFError):
        call(*lost, bad, defl=defl)
    assert call(*out, good, defl=defl) == 0
    for a, b in zip(out, ref):
        assert torch.equal(a, b)
    assert call(*lost, bad, defl=defl) > 0
    h.close()


def test_captured_pass_dropped_after_a_change_of_stream(device):
    """Passes replayed on one stream, the graph then dropped or captured anew from another."""
    prob, h, good, _, defl = _problem(device)
    ref, out = (_vectors(h, prob, device) for _ in range(2))
    assert h.residual_tangent(*ref, good, defl=defl) == 0
    streams = [torch.cuda.Stream() for _ in range(2)]
    for k in range(6):
        h.set_stream(streams[k % 2].cuda_stream)
        h.set_graph(True)
        for x in out:
            x.fill_(np.nan)
        torch.cuda.synchronize()
        for _ in range(3):
            assert h.residual_tangent(*out, good, defl=defl) == 0
            for a, b in zip(out, ref):
                assert torch.equal(a, b)
        h.set_stream(streams[(k + 1) % 2].cuda_stream)
        if k % 3 == 0:
            h.set_graph(False)
        elif k % 3 == 1:
            h.set_assembly(P.ASSEMBLY_COLOURED)
            h.set_assembly(P.ASSEMBLY_GATHER)
        else:
            other = _vectors(h, prob, device)
            assert h.residual_tangent(*other, good, defl=defl) == 0
            assert torch.equal(other[1], ref[1])
    h.set_stream(streams[0].cuda_stream)
    h.close()
