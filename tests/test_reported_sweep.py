"""The run's log and metadata name the sweep that runs."""
import json
from types import SimpleNamespace

import pytest

from pylabolt_amd import cases
from pylabolt_amd.base.state import State
from pylabolt_amd.solvers.fluidLB import FluidLB, Solver
from pylabolt_amd.utils.io_operator import InputOutputOperator


@pytest.mark.parametrize("pairs", [False, True])
def test_metadata(tmp_path, pairs):
    st = State(cases.lid_driven_cavity(20, 16))
    io = InputOutputOperator(FluidLB(), st, root=str(tmp_path))
    # two_step as the engine has it where strips take the sweep's place
    io.engine = SimpleNamespace(storage_name="f64", two_step=True,
                                runs_pairs=pairs)
    io.dump_metadata(st)
    meta = json.loads((tmp_path / "metadata.json").read_text())
    assert meta["engine"] == {"storage": "f64", "two_step": pairs}


@pytest.mark.gpu
@pytest.mark.parametrize("sim,storage,two_step,want", [
    (lambda: cases.poiseuille_channel(2048, 512), "f64", None, "strip sweep"),
    (lambda: cases.poiseuille_channel(120, 300), "f64", None, "tiled sweep"),
    (lambda: cases.poiseuille_channel(120, 512), "f16dev", True,
     "tiled sweep, in pairs"),
    (lambda: cases.poiseuille_channel(1024, 512), "f16dev", True,
     "two-step sweep, in pairs"),
    (lambda: cases.lid_driven_cavity(120, 512), "bf16dev", None,
     "tiled sweep")])
def test_log_line(capsys, sim, storage, two_step, want):
    s = Solver(simulation=sim(), storage=storage, two_step=two_step,
               verbose=False)
    s.set_backend(verbose=True)
    line = [v for v in capsys.readouterr().out.splitlines()
            if v.startswith("Engine")]
    assert line and line[0].endswith(f"storage {storage}, {want}")
    assert s.engine.two_step == (want != "tiled sweep")
