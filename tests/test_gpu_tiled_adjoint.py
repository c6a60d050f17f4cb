"""Reverse steps in regions (d2q9_adjoint_steps) and the forward passes of a
rollout against the step-by-step kernels, at the edges of launches, segments
and lattices."""
import numpy as np
import pytest
import torch

from pylabolt_amd import cases
from pylabolt_amd.adjoint import FlowRollout
from tests.test_host_tiled import _box

pytestmark = pytest.mark.gpu


def _channel(nx, ny, forcing):
    return cases.poiseuille_channel(nx, ny, model="BGK", forcing=forcing)


def _walled(nx, ny, forcing):
    """Bounce-back on every side."""
    sim = cases.lid_driven_cavity(nx, ny)
    sim.boundary_dict["lid"]["fluid"] = {"type": "bounce_back"}
    sim.collision_dict["fluid"]["forcing_model"] = forcing
    return sim


def _circle(nx, ny, forcing):
    sim = _box(nx, ny)
    sim.collision_dict["fluid"]["forcing_model"] = forcing
    return sim


@pytest.mark.parametrize("case", [_channel, _walled, _circle])
@pytest.mark.parametrize("forcing", ["guo_linear", "guo_second_order"])
@pytest.mark.parametrize("size,steps,mode", [
    ((70, 33), 1, "sqrt"), ((37, 70), 5, "sqrt"), ((65, 64), 23, "sqrt"),
    ((40, 26), 11, "moments"), ((20, 18), 40, "sqrt")])
def test_rollout_equals_single_steps(case, forcing, size, steps, mode):
    """The same arithmetic per cell and step, in the same order: equal."""
    rng = np.random.default_rng(5)
    force = torch.tensor(rng.normal(0, 1e-5, (*size, 2)), device="cuda")
    u0 = torch.tensor(rng.normal(0, 0.01, (*size, 2)), device="cuda")
    seed = torch.tensor(rng.normal(0, 1, (*size, 2)), device="cuda")
    got = []
    for tiled in (True, False):
        r = FlowRollout(case(*size, forcing), steps, checkpoint=mode)
        assert r.eng.tiled is not None
        if not tiled:
            r.eng.tiled = None
        for _ in range(2):      # the second pass replays the graphs
            u = r.forward(force, u0)
            gf, gu = r.backward(seed)
        fluid = r.fluid_pad[1:-1, 1:-1]
        got.append([t[fluid] for t in (u, gf, gu)])
        r.close()
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("steps,mode", [(3, "sqrt"), (40, "sqrt"),
                                        (41, "sqrt"), (9, "moments")])
def test_backward_again_and_another_forward(steps, mode):
    """A second reverse pass of the same forward pass gives the same, though
    the first one has replaced the moments of the last segment; so does one
    after another forward pass and back."""
    rng = np.random.default_rng(2)
    force, u0, seed = (torch.tensor(rng.normal(0, s, (30, 40, 2)),
                                    device="cuda") for s in (1e-5, 0.01, 1))
    r = FlowRollout(_channel(30, 40, "guo_linear"), steps, checkpoint=mode)
    u = r.forward(force, u0)
    first = r.backward(seed)
    again = r.backward(seed)
    r.forward(2 * force, u0)
    other = r.backward(seed)
    v = r.forward(force, u0)
    last = r.backward(seed)
    r.close()
    assert torch.equal(u, v)
    for a, b, c, d in zip(first, again, last, other):
        assert torch.equal(a, b) and torch.equal(a, c)
    assert not torch.equal(other[1], first[1])
