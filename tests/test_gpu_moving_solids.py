"""Solids that move (their cells carry a velocity), through every sweep such a
lattice can take: the two-step sweep in all storage forms, and single steps."""
import numpy as np
import pytest

from oracle import d2q9_oracle as O
from pylabolt_amd import cases
from pylabolt_amd.solvers.fluidLB import Solver
from tests.helpers import max_rel, oracle_case

pytestmark = pytest.mark.gpu

# |f - f_oracle| after 20 steps, as in the tests of the precision forms
ABS_TOL = {"f32": 2e-6, "f16dev": 1e-4, "bf16dev": 1e-3}


def _sim(nx=120, ny=300):
    return cases.cylinder(nx, ny, diameter=20, xc=40)


def _spin(fields, nx, ny):
    """A cylinder that rotates and drifts, the fluid stirred."""
    i, j = np.divmod(np.arange((nx + 2) * (ny + 2)), ny + 2)
    v = np.stack([0.02 - 0.003 * (j - ny / 2), 0.003 * (i - 40.0) - 0.01], 1)
    fields.velocity[fields.solid] = v[fields.solid]
    fluid = ~fields.solid & ~fields.ghost_node
    fields.velocity[fluid] = 0.02 * np.random.default_rng(7).standard_normal(
        (int(fluid.sum()), 2))


def _solver(storage, two_step, nx=120, ny=300):
    s = Solver(simulation=_sim(nx, ny), storage=storage, verbose=False,
               graph_steps=4, two_step=two_step)
    _spin(s.state.fields, nx, ny)
    s.set_backend()
    return s


def _same(a, b):
    fluid = a.tables.fluid_pad.ravel()
    for x, y in zip((a.pop(), *a.moments_host()), (b.pop(), *b.moments_host())):
        assert np.array_equal(x[fluid], y[fluid])


@pytest.mark.parametrize("two_step", [True, False])
@pytest.mark.parametrize("storage", ["f64", "f32", "f16dev", "bf16dev"])
def test_moving_cylinder_follows_the_oracle(storage, two_step):
    s = _solver(storage, two_step)
    e = s.engine
    assert e.sweep == ("two-step" if two_step else "single")
    case = oracle_case(_sim())
    _spin(s.state.fields, 120, 300)
    case.velocity[:] = s.state.fields.velocity
    O.initialize_pop(case)
    for n in (1, 2, 17):
        s.advance(n)
        O.run(case, n)
    fl = case.fluid
    pop, (_, vel) = e.pop()[fl], e.moments_host()
    if storage == "f64":
        assert max_rel(pop, case.pop[fl]) <= 1e-12
        assert max_rel(vel[fl], case.velocity[fl]) <= 1e-12
    else:
        err = float(np.abs(pop - case.pop[fl]).max())
        err_u = float(np.abs(vel[fl] - case.velocity[fl]).max())
        print(f"[moving] {storage} {two_step}: {err:.2e} {err_u:.2e}",
              flush=True)
        assert err <= ABS_TOL[storage] and err_u <= 10 * ABS_TOL[storage]


def test_two_step_asked_for_where_strips_would_run():
    two = _solver("f64", True, 1600, 1100).engine
    one = _solver("f64", False, 1600, 1100).engine
    assert two.sweep == "two-step" and one.sweep == "single"
    for n in (2, 9):
        two.advance(n)
        one.advance(n)
    _same(two, one)


def test_solids_set_moving_after_the_engine_was_made():
    """initialize() takes up the velocities the fields hold by then."""
    s = Solver(simulation=_sim(), verbose=False, graph_steps=4, two_step=True)
    s.set_backend()
    s.advance(6)
    _spin(s.state.fields, 120, 300)
    s.collision_operator.initialize_pop(s.state, s.backend)
    s.advance(11)
    one = _solver("f64", False)
    one.advance(11)
    _same(s.engine, one.engine)


def test_large_lattices_take_the_two_step_sweep_by_default():
    default = _solver("f64", None, 1600, 1100).engine
    small = _solver("f64", None).engine
    half = _solver("bf16dev", None, 1600, 1100).engine
    assert default.sweep == "two-step"
    assert small.sweep == half.sweep == "single"
    one = _solver("f64", False, 1600, 1100).engine
    for n in (1, 6):
        default.advance(n)
        one.advance(n)
    _same(default, one)
