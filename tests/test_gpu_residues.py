"""Residue sums (d2q9_residues) against NumPy at sizes around the 64 columns
a wave takes and with more pieces than workgroups."""
import numpy as np
import pytest
import torch

from pylabolt_amd import cases
from pylabolt_amd.engine import padded_view
from pylabolt_amd.solvers.fluidLB import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("nx,ny", [(12, 9), (70, 63), (70, 64), (33, 65),
                                   (20, 128), (700, 1500)])
def test_residue_sums(nx, ny, storage):
    """A sum of n terms of one sign in any order: relative error below n eps
    (the terms themselves are the same)."""
    s = Solver(simulation=cases.cylinder(nx, ny, diameter=min(nx, ny) // 3),
               storage=storage, verbose=False)
    s.set_backend()
    e = s.engine
    e.advance(2)
    rng = np.random.default_rng(5)
    old = torch.from_numpy(rng.standard_normal(3 * e.plane)).to(e.device,
                                                               e.ctype)
    new = torch.from_numpy(rng.standard_normal(3 * e.plane)).to(e.device,
                                                               e.ctype)
    e.mom[e.i_mom].copy_(new)
    before = old.clone()
    torch.cuda.synchronize()
    got = e.residue_sums(old)
    fluid = torch.from_numpy(e.tables.fluid_pad).to(e.device)

    def field(t, q):
        return padded_view(t, q, nx, ny, e.pitch, e.plane)
    for q in range(3):
        o = field(before, q)[fluid].double().cpu().numpy()
        v = field(new, q)[fluid].double().cpu().numpy()
        want = ((v - o) ** 2).sum(), (o ** 2).sum()
        tol = o.size * 2.3e-16
        assert abs(got[2 * q] / want[0] - 1) <= tol
        assert abs(got[2 * q + 1] / want[1] - 1) <= tol
        assert torch.equal(field(old, q)[fluid], field(new, q)[fluid])
        assert torch.equal(field(old, q)[~fluid], field(before, q)[~fluid])
