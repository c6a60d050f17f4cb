"""Strip sweep (d2q9_strip_steps) against single fused steps, bitwise, at the
edges of strips, chunks and launches."""
import numpy as np
import pytest
import torch

from pylabolt_amd import cases
from pylabolt_amd.engine import pop_aos
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


@pytest.mark.parametrize("storage", ["f16dev", "bf16dev"])
@pytest.mark.parametrize("strips", [False, True])
@pytest.mark.parametrize("name", list(STRIP_CASES))
def test_round_last_is_the_float_sweep(name, strips, storage):
    """A launch that rounds only its last step gives the moments of FP32
    storage from the same state bit for bit, and its populations to one unit
    of the 16-bit form's last place (FP16: 2^-10 of the deviation, BF16:
    2^-7, and FP16's smallest number)."""
    one = []
    for st in (storage, "f32"):
        e = _pair(STRIP_CASES[name], st, 24)[0]
        if not strips:
            e.strips = None
        e.advance(1)
        one.append(e)
    a, b = one
    a.tiled.round_last = 1
    fluid = a.tables.fluid_pad.ravel()
    w = np.asarray(a.weights)
    # the whole state, cells outside the fluid too: a cell may pull from them
    scale = np.array([a.L.dev_scale[k] for k in range(9)])
    a.stream.synchronize()
    with torch.cuda.stream(b.stream):
        buf, nx, ny, B, nbj = b.f[b.i_pop], b.nx, b.ny, b.B, b.nbj
        aos = pop_aos(a.f[a.i_pop], nx, ny, B, nbj).float() / torch.tensor(
            scale, dtype=torch.float32, device=b.device)
        rows = buf.reshape(nx + 2, nbj, 9, B).permute(0, 2, 1, 3).reshape(
            nx + 2, 9, nbj * B).clone()
        rows[:, :, B - 1:B - 1 + ny + 2] = aos.reshape(
            nx + 2, ny + 2, 9).permute(0, 2, 1)
        buf.copy_(rows.reshape(nx + 2, 9, nbj, B).permute(0, 2, 1, 3).reshape(
            -1))
        b.mom[b.i_mom].copy_(a.mom[a.i_mom])
    b.stream.synchronize()
    n = 4 if strips else a.tiled.steps
    a.advance(n)
    b.advance(n)
    for x, y in zip(a.moments_host(), b.moments_host()):
        assert np.array_equal(x[fluid], y[fluid])
    x, y = a.pop()[fluid], b.pop()[fluid]
    bits, least = (10, 2.0 ** -24) if storage == "f16dev" else (7, 2.0 ** -120)
    lim = np.abs(y - w) * 2.0 ** -bits + least / scale + 1e-16
    assert (np.abs(x - y) <= lim).all()


def test_two_step_request_in_16_bits():
    """A 16-bit lattice asked for the two-step sweep rounds the last step of
    a launch, by strips or tiles; small lattices in other storage forms run
    that sweep."""
    def engine(sim, storage):
        s = Solver(simulation=sim, storage=storage, verbose=False,
                   two_step=True)
        s.set_backend()
        assert s.engine.two_step
        return s.engine
    e = engine(cases.cylinder(400, 300, diameter=30), "bf16dev")
    assert e.tiled.round_last == 1 and e.strips is None
    e.step2(True)
    assert e.time_step == 2 and e.moments_host()[0].size
    e.set_tile_rows(2)
    assert e.tiled.round_last == int(e.two_step)
    assert engine(cases.lid_driven_cavity(1500, 1300),
                  "f16dev").strips is not None
    assert engine(cases.poiseuille_channel(512, 256),
                  "f16dev").tiled.round_last == 1
    e = engine(cases.cylinder(400, 300, diameter=30), "f32")
    assert e.tiled is None and e._deep is not None
