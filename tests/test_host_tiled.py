"""Host tables of the tiled sweep: where every special cell's populations
stream from, against the oracle's streaming and boundary passes (CPU)."""

import numpy as np
import pytest

from oracle import d2q9_oracle as O
from pylabolt_amd import _native as nt
from pylabolt_amd import cases
from pylabolt_amd.engine import (CX, CY, INV, CaseTables,
                                 elements_from_boundary, strip_rows,
                                 tiled_shape)
from pylabolt_amd.base.state import State
from tests.helpers import oracle_case


def _box(nx, ny, circle=None):
    sim = cases.cylinder(nx, ny, diameter=8)
    sim.boundary_dict = {
        "options": {},
        "ends": {"wall": False, "segments": [[[0, 0], [0, ny - 1]],
                                             [[nx - 1, 0], [nx - 1, ny - 1]]],
                 "fluid": {"type": "periodic"}},
        "sides": {"wall": False, "segments": [[[0, 0], [nx - 1, 0]],
                                              [[0, ny - 1], [nx - 1, ny - 1]]],
                  "fluid": {"type": "periodic"}}}
    sim.obstacle_dict["cylinder"]["center"] = list(circle or (nx / 2, ny / 2))
    return sim


def _two_lids(nx, ny):
    """Moving walls on two adjacent sides: cells with two elements."""
    sim = cases.lid_driven_cavity(nx, ny)
    sim.boundary_dict["side"] = {
        "wall": True, "segments": [[[nx - 1, 0], [nx - 1, ny - 1]]],
        "fluid": {"type": "fixed_velocity", "value": [0.0, 0.03]}}
    return sim


def _mixed_ends(nx, ny):
    """Fixed-pressure, moving-wall and bounce-back sides together."""
    sim = cases.cylinder(nx, ny, diameter=6)
    b = sim.boundary_dict
    b["top_bottom"]["fluid"] = {"type": "bounce_back"}
    b["outlet"]["fluid"] = {"type": "fixed_velocity", "value": [0.02, 0.01]}
    return sim


CASES = {
    "cavity": lambda: cases.lid_driven_cavity(11, 9),
    "two_lids": lambda: _two_lids(10, 12),
    "channel": lambda: cases.poiseuille_channel(9, 8),
    "cylinder": lambda: cases.cylinder(40, 26, diameter=8),
    "mixed_ends": lambda: _mixed_ends(30, 20),
    "box": lambda: _box(20, 18),
    # the circle crosses both periodic sides
    "box_edge": lambda: _box(20, 18, (0.0, 0.0)),
}


@pytest.mark.parametrize("name", CASES)
def test_special_codes_stream_as_the_oracle(name):
    case = oracle_case(CASES[name]())
    sim = CASES[name]()
    st = State(sim)
    nx, ny = int(st.domain.Nx_rank), int(st.domain.Ny_rank)
    t = CaseTables(nx, ny, st.fields.solid, elements_from_boundary(st.boundary),
                   st.boundary.x_periodic, st.boundary.y_periodic, 64, 4)
    cells, codes, has_vel, has_pres = t.special_codes()
    O.initialize_pop(case)
    rng = np.random.default_rng(1)
    case.pop_new[:] *= 1.0 + 0.01 * rng.standard_normal(case.pop_new.shape)
    O.run(case, 3)
    shape = (nx + 2, ny + 2)
    pop = case.pop.reshape(*shape, 9).copy()
    pop[0], pop[-1], pop[:, 0], pop[:, -1] = 0, 0, 0, 0
    if t.x_periodic:
        pop[0], pop[-1] = pop[-2], pop[1]
    if t.y_periodic:
        pop[:, 0], pop[:, -1] = pop[:, -2], pop[:, 1]
    solid = case.solid.reshape(shape)
    pop[solid] = 0.0
    rho = case.density.reshape(shape)
    u = case.velocity.reshape(*shape, 2)
    want = case.pop_new.reshape(*shape, 9)
    kinds = set()
    for i, j in np.argwhere(t.fluid_pad):
        flags = int(cells[i, j]) & 0xff
        assert flags == t.flags_pad[i, j]
        got = np.array([pop[i - CX[k], j - CY[k], k] for k in range(9)])
        if flags & (nt.CELL_NEAR_SOLID | nt.CELL_BC):
            rec = [int(v) for v in codes[int(cells[i, j]) >> 8]]
            for d in range(1, 9):
                w = (rec[(d - 1) >> 2] >> (8 * ((d - 1) & 3))) & 0xff
                dr, dc, k = (w & 3) - 1, ((w >> 2) & 3) - 1, w >> 4
                got[d] = pop[i + dr, j + dc, k]
                if not (rec[2] >> (d - 1)) & 1:
                    continue
                elem = (rec[2] >> (24 if (rec[2] >> (d + 7)) & 1 else 16)) & 0xff
                kind, e = t.elems[elem]
                kinds.add(kind)
                o = int(INV[d])
                assert (dr, dc, k) == (0, 0, o)
                if kind == nt.RULE_VEL:
                    got[d] -= 6 * st.lattice.weights[o] * rho[i, j] * (
                        CX[o] * e["vector"][0] + CY[o] * e["vector"][1])
                else:
                    n0, n1 = e["normal"]
                    ue = 1.5 * u[i, j] - 0.5 * u[i + n0, j + n1]
                    cu = CX[o] * ue[0] + CY[o] * ue[1]
                    got[d] = -got[d] + 2 * st.lattice.weights[o] * e["scalar"] * (
                        1 + 4.5 * cu * cu - 1.5 * (ue @ ue))
        np.testing.assert_allclose(got, want[i, j], rtol=0, atol=1e-15)
    assert has_vel == (nt.RULE_VEL in kinds)
    assert has_pres == (nt.RULE_PRES in kinds)


def test_special_codes_refuse_what_they_cannot_express():
    # a zero-gradient side whose inward neighbours are partly solid
    sim = cases.cylinder(40, 26, diameter=8)
    sim.obstacle_dict["cylinder"]["center"] = [20.0, 4.0]
    sim.obstacle_dict["cylinder"]["radius"] = 3.0
    st = State(sim)
    t = CaseTables(40, 26, st.fields.solid, elements_from_boundary(st.boundary),
                   st.boundary.x_periodic, st.boundary.y_periodic, 64, 4)
    assert t.special_codes() is None


def test_special_codes_refuse_many_elements():
    sim = cases.lid_driven_cavity(80, 12)
    walls = sim.boundary_dict["walls"]
    walls["segments"] = walls["segments"][:2] + [
        [[2 * k, 0], [2 * k + 1, 0]] for k in range(40)]
    st = State(sim)
    t = CaseTables(80, 12, st.fields.solid, elements_from_boundary(st.boundary),
                   st.boundary.x_periodic, st.boundary.y_periodic, 64, 4)
    assert len(t.elems) > nt.TILED_MAX_ELEMS
    assert t.special_codes() is None


@pytest.mark.parametrize("nx,ny", [(2, 2), (7, 300), (128, 128), (513, 97),
                                   (4096, 1024), (30000, 3)])
@pytest.mark.parametrize("double", [True, False])
@pytest.mark.parametrize("forced", [True, False])
def test_tiled_shape_fits_a_workgroup(nx, ny, double, forced):
    rows, width, steps = tiled_shape(((nx, ny),), double, forced)
    assert width in (16, 32, 64) and rows * width <= 1024
    assert steps >= 1 and rows > 2 * steps and width > 2 * steps


STRIP_CASES = {
    "channel": lambda: cases.poiseuille_channel(60, 64),
    "channel_wide": lambda: cases.poiseuille_channel(40, 233),
    "cylinder": lambda: cases.cylinder(150, 200, diameter=20),
    "cavity": lambda: cases.lid_driven_cavity(70, 121),
    "box": lambda: _box(45, 119),
    "box_edge": lambda: _box(60, 130, (0.0, 0.0)),
}


@pytest.mark.parametrize("rows", [8, 24, 1000])
@pytest.mark.parametrize("name", STRIP_CASES)
def test_strip_split_covers_with_plain_chunks(name, rows):
    """Every fluid cell is in a chunk or a tile; every cell within 4 of a
    chunk is plain fluid or the stated wall."""
    sim = STRIP_CASES[name]()
    st = State(sim)
    nx, ny = int(st.domain.Nx_rank), int(st.domain.Ny_rank)
    t = CaseTables(nx, ny, st.fields.solid, elements_from_boundary(st.boundary),
                   st.boundary.x_periodic, st.boundary.y_periodic, 64, 4)
    chunks, tiles, share = t.strip_split(4, 56, 8, rows)
    assert share == tiles.shape[0] * 64 / (nx * ny)
    inner = t.flags_pad[1:-1, 1:-1]
    side = t.wall_side_pad[1:-1, 1:-1]
    seen = np.zeros((nx, ny), dtype=bool)
    for i, n, j, cols, walls in chunks:
        assert 1 <= i and i + n - 1 <= nx and 1 <= j and j + cols - 1 <= ny
        assert 8 <= cols <= 56 and n >= 1
        lo, hi = walls & 3, walls >> 2
        seen[i - 1:i - 1 + n, j - 1:j - 1 + cols] = True
        for r in range(i - 5, i + n + 3):
            if not t.x_periodic:
                assert 0 <= r < nx
            for c in range(j - 5, j + cols + 3):
                if not t.y_periodic and not 0 <= c < ny:
                    assert (lo and j == 1) if c < 0 else (
                        hi and j + cols - 1 == ny)
                    continue
                f = inner[r % nx, c % ny]
                if f == nt.CELL_FLUID:
                    continue
                assert f == nt.CELL_FLUID | nt.CELL_BC
                s = side[r % nx, c]
                assert (c == 0 and s == {1: 0, 2: 2}[lo]) or (
                    c == ny - 1 and s == {1: 1, 2: 3}[hi])
    for i, j in tiles:
        seen[i - 1:i + 7, j - 1:j + 7] = True
    assert seen[t.fluid_pad[1:-1, 1:-1]].all()


def test_strip_rows_rule():
    """One row count per case: chunks just fill whole rounds of what the GPU
    holds at once (1536, in FP64 768), or None for small lattices."""
    def rows(nx, strips, double, **kw):
        return strip_rows(np.full(strips, nx), double, **kw)
    assert rows(800, 14, False) is None
    assert rows(1024, 19, False, rounds=True) is None
    assert strip_rows(np.zeros(0, dtype=int), True) is None
    for nx, strips, double in ((2048, 19, False), (1500, 24, False),
                               (1100, 20, True), (900, 17, False)):
        r = rows(nx, strips, double)
        n = strips * max(1, round(nx / r))
        slots = 768 if double else 1536
        assert 0.85 * slots < n <= slots
    assert 40 <= rows(8192, 37, True) <= 160
    assert rows(8192, 37, False, most=32) <= 32
