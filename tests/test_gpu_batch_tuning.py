"""The autotuner times the persistent kernel only for batches that run it."""
import numpy as np
import pytest

from pylabolt_amd import batch as B
from pylabolt_amd import cases
from pylabolt_amd.solvers.fluidLB import Solver

pytestmark = pytest.mark.gpu


def _sims():
    return cases.batch_cases(n=3, seed=2, nx_range=(32, 64),
                             ny_range=(64, 96)) + [
        cases.cylinder(48, 80, diameter=12, xc=16)]


@pytest.fixture
def runs(monkeypatch):
    """Batches that were tuned, in order (one candidate each)."""
    seen = []
    tune = B.BatchAutotuner.tune

    def spy(self, batch):
        seen.append(batch)
        return tune(self, batch)
    monkeypatch.setattr(B.BatchAutotuner, "tune", spy)
    monkeypatch.setattr(B.BatchAutotuner, "candidates",
                        lambda self, batch: [B.BatchConfig(2, 0, None, 1)])
    return seen


def test_tuned_when_the_persistent_kernel_runs(runs):
    batch = B.BatchedLattices(_sims(), storage="f32")
    assert batch.tiled and not runs
    batch.advance(6)
    assert not runs
    # a lattice that starts anew by itself does not tune either
    batch.engines[0].initialize()
    batch.engines[0].advance(6)
    batch.advance(3)
    assert not runs
    # a solid that moves: the lattice has no tables for the tiled sweep
    solo = []
    for s in batch.solvers + [Solver(simulation=v, storage="f32",
                                     verbose=False, two_step=False)
                              for v in _sims()]:
        f = s.state.fields
        f.velocity[f.solid] = [0.01, -0.005]
        if s not in batch.solvers:
            s.set_backend()
            s.engine.tiled = None
            solo.append(s.engine)
        else:
            s.engine.initialize()
    batch.advance(5)
    batch.advance(4)
    assert runs == [batch] and batch.config.tile_i == 2
    for a, b in zip(batch.engines, solo):
        b.advance(9)
        assert np.array_equal(a.pop(), b.pop())
    batch.close()


def test_a_tuner_that_is_given_tunes_at_once(runs):
    batch = B.BatchedLattices(_sims(), storage="f32",
                              tuner=B.BatchAutotuner(reps=1))
    assert runs == [batch]
    batch.close()
