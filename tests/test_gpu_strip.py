"""Strip sweep (d2q9_strip_steps) against single fused steps, bitwise, at the
edges of strips, chunks and launches."""
import numpy as np
import pytest

from pylabolt_amd import cases
from pylabolt_amd.solvers.fluidLB import Solver
from tests.test_host_tiled import STRIP_CASES, _box

pytestmark = pytest.mark.gpu

STORAGES = ("f64", "f32", "f16dev", "bf16dev")


def _pair(sim, storage, rows, force=None):
    """Two engines of a case from the same perturbed start: the first held to
    the strip sweep with chunks of about ``rows`` rows, the second to single
    steps."""
    out = []
    for strips in (True, False):
        s = Solver(simulation=sim(), storage=storage, verbose=False,
                   two_step=False)
        f = s.state.fields
        rng = np.random.default_rng(3)
        fluid = ~f.solid & ~f.ghost_node
        f.velocity[fluid] = 0.02 * rng.standard_normal((int(fluid.sum()), 2))
        s.backend.create_engine(s.state, s.collision_operator,
                                s.force_operator, force_field=force)
        e = s.engine
        if strips:
            e._setup_strips(rows)
            assert e.strips is not None and e.strips.n_chunks > 0
        else:
            e.tiled = None
        out.append(e)
    return out


def _equal(a, b, what):
    fluid = a.tables.fluid_pad.ravel()
    for x, y in zip((a.pop(), *a.moments_host()), (b.pop(), *b.moments_host())):
        assert np.array_equal(x[fluid], y[fluid]), what


@pytest.mark.parametrize("storage", STORAGES)
@pytest.mark.parametrize("name", list(STRIP_CASES))
def test_strips_equal_single_steps(name, storage):
    a, b = _pair(STRIP_CASES[name], storage, 24)
    # the first step, one launch of 4, 3 and 2 steps, several, one step
    for n in (5, 3, 2, 11, 1):
        a.advance(n)
        b.advance(n)
        _equal(a, b, (name, storage, n))


@pytest.mark.parametrize("ny", [64, 112, 119, 120, 121, 176])
@pytest.mark.parametrize("rows", [1, 17, 1000])
def test_strip_widths_and_chunk_heights(ny, rows):
    a, b = _pair(lambda: cases.poiseuille_channel(
        50, ny, model="BGK", forcing="guo_second_order"), "f64", rows)
    a.advance(10)
    b.advance(10)
    _equal(a, b, (ny, rows))


@pytest.mark.parametrize("ny", [120, 121])
def test_force_field(ny):
    nx = 40
    force = 1e-5 * np.random.default_rng(1).standard_normal(
        ((nx + 2) * (ny + 2), 2))

    def sim():
        s = _box(nx, ny)
        s.collision_dict["fluid"]["forcing_model"] = "guo_linear"
        return s
    a, b = _pair(sim, "f32", 20, force)
    a.advance(9)
    b.advance(9)
    _equal(a, b, ny)


def test_large_lattices_take_the_strips():
    s = Solver(simulation=cases.cylinder(1600, 1100, diameter=64),
               storage="f64", verbose=False)
    s.set_backend()
    assert s.engine.strips is not None and not s.engine.two_step
    ref = Solver(simulation=cases.cylinder(1600, 1100, diameter=64),
                 storage="f64", verbose=False, two_step=False)
    ref.set_backend()
    ref.engine.tiled = None
    for n in (7, 1, 8):
        s.advance(n)
        ref.advance(n)
        assert np.array_equal(s.engine.pop(), ref.engine.pop())
