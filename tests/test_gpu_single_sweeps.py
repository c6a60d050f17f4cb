"""Single sweeps and their graphs, forks and tile modes, on lattices held to
them (or without tables for the sweeps of several steps per launch)."""
import threading

import numpy as np
import pytest

from oracle import d2q9_oracle as O
from pylabolt_amd import cases
from pylabolt_amd.solvers.fluidLB import Solver
from tests.helpers import max_rel, oracle_case
from tests.test_gpu_solid_tiles import CYLINDERS
from tests.test_host_tiled import _box

pytestmark = pytest.mark.gpu


def _engine(sim, storage="f64", sweep="single", **kw):
    s = Solver(simulation=sim, storage=storage, verbose=False, **kw)
    s.set_backend()
    if sweep == "single" and s.engine.sweep != "single":
        s.engine.tiled = None
    assert s.engine.sweep == sweep
    return s.engine


def _against(case, e, n):
    O.run(case, n)
    fl = case.fluid
    rho, vel = e.moments_host()
    assert max_rel(e.pop()[fl], case.pop[fl]) <= 1e-12
    assert max_rel(e.pop_new()[fl], case.pop_new[fl]) <= 1e-12
    assert max_rel(rho[fl], case.density[fl]) <= 1e-12
    assert max_rel(vel[fl], case.velocity[fl]) <= 1e-12


@pytest.mark.parametrize("name", sorted(CYLINDERS))
def test_solids_as_fix_up_cells(name):
    case = oracle_case(CYLINDERS[name]())
    O.initialize_pop(case)
    e = _engine(CYLINDERS[name](), graph_steps=4, two_step=False,
                solid_tiles="cells")
    assert e.tables.n_general == 0
    for n in (1, 6, 13):
        e.advance(n)
        _against(case, e, n)


@pytest.mark.parametrize("storage", ["f32", "f16dev", "bf16dev"])
@pytest.mark.parametrize("name", ["cylinder_wide", "cylinder_two_blocks"])
def test_solid_tile_modes_are_bitwise_equal(name, storage):
    a, b = (_engine(CYLINDERS[name](), storage, graph_steps=4,
                    two_step=False, solid_tiles=mode)
            for mode in ("sweep", "cells"))
    assert a.tables.n_general > 0 and b.tables.n_general == 0
    for n in (1, 9, 10):
        a.advance(n)
        b.advance(n)
        for x, y in zip((a.pop(), a.pop_new(), *a.moments_host()),
                        (b.pop(), b.pop_new(), *b.moments_host())):
            assert np.array_equal(x, y)


def test_graph_replays_of_a_periodic_box():
    def sim():
        s = _box(70, 300)
        s.obstacle_dict = {"options": {}}
        s.collision_dict["fluid"]["forcing_model"] = "guo_second_order"
        s.forcing_dict = {"gravity": [1e-5, -2e-6]}
        s.initial_fields_dict["default"]["fluid"]["velocity"] = {
            "type": "func", "func": lambda i, j: (0.01 * np.sin(j / 7.0),
                                                  0.02 * np.cos(i / 5.0))}
        return s
    case = oracle_case(sim())
    O.initialize_pop(case)
    e = _engine(sim(), graph_steps=8, two_step=False)
    assert (e.tables.tile_class == 0).any()
    e.advance(41)
    assert len(e._graphs) == 1
    _against(case, e, 41)


@pytest.mark.parametrize("storage,two_step", [("f64", False), ("f64", True),
                                              ("f16dev", True)])
def test_more_boundary_elements_than_the_tiled_sweep_takes(storage, two_step):
    def sim():
        s = cases.lid_driven_cavity(80, 520)
        lid = s.boundary_dict.pop("lid")
        (a, b), = lid["segments"]
        for k in range(40):
            s.boundary_dict[f"lid{k}"] = {
                "wall": True, "segments": [[[a[0] + 2 * k, a[1]],
                                            [a[0] + 2 * k + 1, b[1]]]],
                "fluid": {"type": "fixed_velocity",
                          "value": [0.05 + 1e-3 * k, 0.0]}}
        return s
    case = oracle_case(sim())
    O.initialize_pop(case)
    e = _engine(sim(), storage, "two-step" if two_step else "single",
                graph_steps=4, two_step=two_step)
    assert e.tiled is None
    e.advance(20)
    if storage == "f64":
        _against(case, e, 20)
    else:
        O.run(case, 20)
        fl = case.fluid
        assert np.abs(e.pop()[fl] - case.pop[fl]).max() <= 1e-4


def _drive(e, barrier=None):
    if barrier is not None:
        barrier.wait()
    for _ in range(12):
        # eager steps and graph replays, each with forks and joins
        e.advance(2, use_graph=False)
        e.advance(9)


def test_two_threads_on_two_streams():
    def engines():
        return [_engine(cases.cylinder(44, 130, diameter=10, xc=14),
                        graph_steps=4, two_step=False),
                _engine(cases.cylinder(120, 300, diameter=20, xc=40),
                        sweep="two-step", graph_steps=4, two_step=True)]
    alone = engines()
    for e in alone:
        _drive(e)
        assert e._graphs
    both = engines()
    barrier, errors = threading.Barrier(2), []

    def run(e):
        try:
            _drive(e, barrier)
        except Exception as err:  # reported below
            errors.append(err)
    threads = [threading.Thread(target=run, args=(e,)) for e in both]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for a, b in zip(alone, both):
        for x, y in zip((a.pop(), *a.moments_host()),
                        (b.pop(), *b.moments_host())):
            assert np.array_equal(x, y)
