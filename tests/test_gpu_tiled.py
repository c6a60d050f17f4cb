"""Tiled sweep (several steps per launch, d2q9_tiled_steps) against single
fused steps, bitwise, at the edges of regions, launches and lattices."""
import numpy as np
import pytest
import torch

from pylabolt_amd import _native as nt
from pylabolt_amd import cases
from pylabolt_amd.solvers.fluidLB import Solver
from tests.test_host_tiled import CASES, _box, _two_lids

pytestmark = pytest.mark.gpu

STORAGES = ("f64", "f32", "f16dev", "bf16dev")


def _pair(sim, storage, seed=3):
    """Two solvers of a case from the same perturbed start, the second one
    held to single steps."""
    out = []
    for tiled in (True, False):
        s = Solver(simulation=sim(), storage=storage, verbose=False,
                   two_step=False)
        f = s.state.fields
        rng = np.random.default_rng(seed)
        fluid = ~f.solid & ~f.ghost_node
        f.velocity[fluid] = 0.02 * rng.standard_normal((int(fluid.sum()), 2))
        s.set_backend()
        assert s.engine.tiled is not None
        if not tiled:
            s.engine.tiled = None
        out.append(s.engine)
    return out


def _equal(a, b, what):
    for x, y in zip((a.pop(), *a.moments_host()), (b.pop(), *b.moments_host())):
        fluid = a.tables.fluid_pad.ravel()
        assert np.array_equal(x[fluid], y[fluid]), what


@pytest.mark.parametrize("storage", STORAGES)
@pytest.mark.parametrize("name", list(CASES))
def test_tiled_equals_single_steps(name, storage):
    a, b = _pair(CASES[name], storage)
    K = a.tiled.steps
    # first step after initialisation, one launch, a remainder
    for n in (1, K, 2 * K + 1):
        a.advance(n)
        b.advance(n)
        _equal(a, b, (name, storage, n))


@pytest.mark.parametrize("shape", [(24, 32, 4), (14, 16, 6), (20, 32, 8),
                                   (16, 64, 5), (5, 16, 2), (32, 32, 1)])
@pytest.mark.parametrize("sim", [
    lambda: cases.lid_driven_cavity(64, 48),
    lambda: cases.poiseuille_channel(70, 131),
    lambda: cases.cylinder(90, 129, diameter=12),
    lambda: _box(65, 64)], ids=["cavity", "channel", "cylinder", "box"])
def test_region_shapes(sim, shape):
    a, b = _pair(sim, "f64")
    a.tiled.rows, a.tiled.width, a.tiled.steps = shape
    for n in (shape[2] + 1, 3 * shape[2]):
        a.advance(n)
        b.advance(n)
        _equal(a, b, (shape, n))


@pytest.mark.parametrize("nx,ny", [(2, 2), (3, 70), (129, 4)])
def test_lattices_smaller_than_a_region(nx, ny):
    a, b = _pair(lambda: cases.poiseuille_channel(nx, ny, model="BGK"), "f64")
    a.advance(13)
    b.advance(13)
    _equal(a, b, (nx, ny))


def test_after_materialize_and_single_steps():
    a, b = _pair(lambda: _two_lids(33, 40), "f32")
    for e in (a, b):
        e.advance(5)
        e.materialize()
        e.step(write_moments=True)
        e.advance(7)
    _equal(a, b, "materialize")
    assert a.time_step == b.time_step == 13


def test_moving_solids_keep_single_steps():
    s = Solver(simulation=cases.cylinder(60, 40, diameter=8), verbose=False)
    f = s.state.fields
    f.velocity[f.solid, 0] = 0.01
    s.set_backend()
    assert s.engine.tiled is None


def test_bad_regions_are_refused():
    s = Solver(simulation=cases.lid_driven_cavity(32, 32), verbose=False)
    s.set_backend()
    e = s.engine
    for rows, width, steps in ((24, 48, 4), (8, 32, 4), (64, 32, 4),
                               (24, 16, 8), (24, 32, 0)):
        e.tiled.rows, e.tiled.width, e.tiled.steps = rows, width, steps
        rc = e.lib.d2q9_tiled_steps(
            e._Lp, e._tiled_p, nt.ptr(e.f[0]), nt.ptr(e.f[1]),
            nt.ptr(e.mom[0]), nt.ptr(e.mom[1]), 1, 1, 1, None, 0,
            e._stream_ptr)
        assert rc in (-1, -2), (rows, width, steps)
    torch.cuda.synchronize()
