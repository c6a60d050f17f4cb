"""16-bit lattices asked for the two-step sweep: what is rounded follows from
the step alone (in the deep interior every second one), not from how many
steps a call or a launch takes."""
import numpy as np
import pytest
import torch

from pylabolt_amd import cases
from pylabolt_amd.solvers.fluidLB import Solver

pytestmark = pytest.mark.gpu

CASES = {
    # no rim; ny of two blocks of either 16-bit form
    "channel": lambda: cases.poiseuille_channel(96, 512),
    # a rim with a moving wall; with pressure ends and a solid
    "cavity": lambda: cases.lid_driven_cavity(100, 400),
    "cylinder": lambda: cases.cylinder(120, 520, diameter=20, xc=40),
    # large enough for strips
    "large_cavity": lambda: cases.lid_driven_cavity(1500, 1300),
}


def _engine(sim, storage):
    s = Solver(simulation=sim(), storage=storage, verbose=False,
               two_step=True)
    f = s.state.fields
    rng = np.random.default_rng(5)
    fluid = ~f.solid & ~f.ghost_node
    f.velocity[fluid] = 0.02 * rng.standard_normal((int(fluid.sum()), 2))
    s.set_backend()
    return s.engine


@pytest.mark.parametrize("storage", ["f16dev", "bf16dev"])
@pytest.mark.parametrize("name", list(CASES))
def test_rounding_does_not_follow_the_calls(name, storage):
    a, b = (_engine(CASES[name], storage) for _ in range(2))
    assert (a.deep_fraction == 1.0) == (name == "channel")
    a.advance(1)
    b.step(True)
    a.advance(13)
    for _ in range(6):
        b.advance(2)
    b.step(True)
    fluid = a.tables.fluid_pad.ravel()
    for x, y in zip((a.pop(), *a.moments_host()), (b.pop(), *b.moments_host())):
        assert np.array_equal(x[fluid], y[fluid]), (name, storage)


@pytest.mark.parametrize("storage", ["f16dev", "f32"])
def test_without_room_for_the_scratch_lattice(monkeypatch, storage):
    """The lattice then advances as with single steps."""
    def sim():
        return (cases.poiseuille_channel(1024, 512) if storage == "f16dev"
                else cases.lid_driven_cavity(200, 300))

    def full(*a, **k):
        raise torch.cuda.OutOfMemoryError("no room")
    engines = []
    for two_step in (False, True):
        s = Solver(simulation=sim(), storage=storage, verbose=False,
                   two_step=two_step)
        with monkeypatch.context() as m:
            if two_step:
                m.setattr(torch, "empty_like", full)
                with pytest.warns(UserWarning, match="no device memory"):
                    s.set_backend()
            else:
                s.set_backend()
        engines.append(s.engine)
    a, b = engines
    assert not b.two_step and not b.runs_pairs
    for n in (1, 7):
        a.advance(n)
        b.advance(n)
        assert np.array_equal(a.pop(), b.pop())
