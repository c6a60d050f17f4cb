"""The tiled and strip sweeps with the two-step sweep's roundings (16-bit
lattices asked for two steps per sweep) against that sweep, bit for bit."""
import numpy as np
import pytest

from pylabolt_amd import _native as nt
from pylabolt_amd import cases, engine
from pylabolt_amd.solvers.fluidLB import Solver
from tests.test_host_tiled import _box, _mixed_ends, _two_lids

pytestmark = pytest.mark.gpu


def _forced(nx, ny, model="MRT", forcing="guo_second_order"):
    sim = cases.poiseuille_channel(nx, ny, model=model, forcing=forcing)
    sim.forcing_dict["gravity"] = [2e-5, 3e-6]
    return sim


CASES = {
    # no rim; the last row of deep tiles moved up (80 = 6 x 12 + 8)
    "channel": lambda: _forced(72, 256),
    "channel_shifted": lambda: _forced(80, 128, "BGK", "guo_linear"),
    # rims: beside a part of a block, moving walls, pressure ends, solids,
    # sides periodic in y, rows that no tile height divides
    "channel_part": lambda: _forced(75, 300),
    "cavity": lambda: cases.lid_driven_cavity(70, 384),
    "two_lids": lambda: _two_lids(61, 400),
    "cylinder": lambda: cases.cylinder(96, 400, diameter=20, xc=30),
    "mixed_ends": lambda: _mixed_ends(70, 384),
    "box": lambda: _box(66, 384, (20.0, 10.0)),
    "box_edge": lambda: _box(66, 384, (0.0, 0.0)),
}


def _pair(monkeypatch, sim, storage):
    out = []
    for cells in (1 << 30, 0):   # below which tiles run
        monkeypatch.setattr(engine, "_PAIRS_TILED_CELLS",
                            {True: cells, False: cells})
        monkeypatch.setattr(engine, "strip_rows", lambda *a, **k: None)
        s = Solver(simulation=sim(), storage=storage, verbose=False,
                   graph_steps=4, two_step=True)
        f = s.state.fields
        rng = np.random.default_rng(3)
        fluid = ~f.solid & ~f.ghost_node
        f.velocity[fluid] = 0.02 * rng.standard_normal((int(fluid.sum()), 2))
        s.set_backend()
        out.append(s.engine)
    assert [e.sweep for e in out] == ["tiled", "two-step"]
    return out


def _equal(a, b, what):
    fluid = a.tables.fluid_pad.ravel()
    for x, y in zip((a.pop(), *a.moments_host()), (b.pop(), *b.moments_host())):
        assert np.array_equal(x[fluid], y[fluid]), what


@pytest.mark.parametrize("storage", ["f16dev", "bf16dev"])
@pytest.mark.parametrize("name", list(CASES))
def test_equals_the_two_step_sweep(monkeypatch, name, storage):
    a, b = _pair(monkeypatch, CASES[name], storage)
    K = a.tiled.steps
    assert a.tiled.pairs == (1 if name.startswith("channel") and
                             name != "channel_part" else 2)
    # the first step alone, a pair, one and a half, whole launches and a rest
    for n in (1, 2, 3, K, 3 * K - 1, 2 * K + 2, 4):
        a.advance(n)
        b.advance(n)
        _equal(a, b, (name, storage, n))


@pytest.mark.parametrize("shape", [(24, 32, 4), (14, 16, 6), (20, 32, 8),
                                   (16, 64, 5), (7, 16, 2), (18, 32, 3)])
@pytest.mark.parametrize("name", ["cylinder", "box_edge", "two_lids"])
def test_region_shapes(monkeypatch, name, shape):
    a, b = _pair(monkeypatch, CASES[name], "bf16dev")
    a.tiled.rows, a.tiled.width, a.tiled.steps = shape
    for n in (6, 17, 8, 2):
        a.advance(n)
        b.advance(n)
        _equal(a, b, (name, shape, n))


@pytest.mark.parametrize("strips", [False, True])
def test_other_tile_rows_move_the_rim(monkeypatch, strips):
    a, b = _pair(monkeypatch, lambda: _forced(70, 256), "f16dev")
    if strips:
        a._setup_strips(9)
        assert a.sweep == "strips"
    for rows, pairs in ((4, 2), (2, 1)):
        a.set_tile_rows(rows)
        b.set_tile_rows(rows)
        assert a.tiled.pairs == pairs
        for n in (4, 7):
            a.advance(n)
            b.advance(n)
            _equal(a, b, (rows, n))


STRIPS = {
    "channel": lambda: _forced(72, 256),
    "channel_shifted": lambda: _forced(80, 128, "BGK", "guo_linear"),
    "cavity": lambda: cases.lid_driven_cavity(150, 512),
    # zero-gradient walls in deep tiles, a solid, pressure ends; a part of a
    # block at the high side; sides periodic in y
    "cylinder": lambda: cases.cylinder(200, 384, diameter=20, xc=60),
    "cylinder_part": lambda: cases.cylinder(160, 450, diameter=20, xc=50),
    "box": lambda: _box(150, 512, (20.0, 10.0)),
}


@pytest.mark.parametrize("storage", ["f16dev", "bf16dev"])
@pytest.mark.parametrize("rows", [9, 40])
@pytest.mark.parametrize("name", list(STRIPS))
def test_strips_equal_the_two_step_sweep(monkeypatch, name, rows, storage):
    a, b = _pair(monkeypatch, STRIPS[name], storage)
    a._setup_strips(rows)
    assert a.sweep == "strips" and a.strips.n_chunks > 0
    assert a.strips.n_tiles > 0 or a.tiled.pairs == 1
    # launches of 4, 2 and 3, a step left over, whole launches
    for n in (1, 4, 2, 3, 9, 15, 8):
        a.advance(n)
        b.advance(n)
        _equal(a, b, (name, rows, storage, n))


@pytest.mark.parametrize("sim,storage,sweep", [
    (lambda: cases.lid_driven_cavity(1500, 1300), "f16dev", "strips"),
    (lambda: cases.cylinder(1400, 2000, diameter=64), "bf16dev", "strips"),
    (lambda: cases.poiseuille_channel(5000, 1024), "f16dev", "strips"),
    (lambda: cases.poiseuille_channel(1500, 1024), "f16dev", "two-step"),
    (lambda: cases.cylinder(2277, 892, diameter=64), "bf16dev", "tiled")])
def test_large_lattices(monkeypatch, sim, storage, sweep):
    """The sweep a large lattice takes, its moments and populations."""
    out = []
    for held in (False, True):
        if held:
            monkeypatch.setattr(engine, "_PAIRS_TILED_CELLS",
                                {True: 0, False: 0})
            monkeypatch.setattr(engine, "strip_rows", lambda *a, **k: None)
        s = Solver(simulation=sim(), storage=storage, verbose=False,
                   two_step=True)
        s.set_backend()
        out.append(s.engine)
    a, b = out
    assert a.sweep == sweep and b.sweep == "two-step"
    for n in (6, 9):
        a.advance(n)
        b.advance(n)
        _equal(a, b, (sweep, n))


def test_bad_pairs_are_refused():
    s = Solver(simulation=cases.lid_driven_cavity(60, 300), storage="f16dev",
               verbose=False, two_step=True)
    s.set_backend()
    e = s.engine
    for pairs, steps in ((3, 4), (-1, 4), (1, 1)):
        e.tiled.pairs, e.tiled.steps = pairs, steps
        assert e.lib.d2q9_tiled_steps(
            e._Lp, e._tiled_p, nt.ptr(e.f[0]), nt.ptr(e.f[1]),
            nt.ptr(e.mom[0]), nt.ptr(e.mom[1]), 4, 0, 0, None, 0,
            e._stream_ptr) == -1
