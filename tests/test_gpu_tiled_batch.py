"""Batched tiled sweep against every lattice stepped alone by single sweeps,
and the persistent kernel that serves batches without its tables."""
import numpy as np
import pytest

from pylabolt_amd import cases
from pylabolt_amd.batch import BatchConfig, BatchedLattices
from pylabolt_amd.solvers.fluidLB import Solver
from tests.test_host_tiled import _box, _two_lids

pytestmark = pytest.mark.gpu


def _sims():
    sims = cases.batch_cases(n=4, seed=5, nx_range=(32, 96), ny_range=(64, 320))
    return sims + [cases.cylinder(48, 140, diameter=12, xc=16), _box(20, 18),
                   _two_lids(33, 40),
                   cases.poiseuille_channel(3, 9, model="BGK",
                                            forcing="guo_linear")]


def _single(sim, storage):
    s = Solver(simulation=sim, storage=storage, verbose=False, two_step=False)
    s.set_backend()
    s.engine.tiled = None
    return s.engine


@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("tiled,policy", [(True, 1), (False, 0), (False, 1)])
def test_batch_equals_single_steps(storage, tiled, policy):
    batch = BatchedLattices(_sims(), storage=storage, graph_steps=4,
                            config=BatchConfig(4, policy, None, 2))
    assert batch.tiled
    batch.tiled = tiled
    solo = [_single(s, storage) for s in _sims()]
    K = batch._tiled_region[2]
    for n in (1, K, 2 * K + 1, 1):
        batch.advance(n)
        for l, (a, b) in enumerate(zip(batch.engines, solo)):
            b.advance(n)
            for x, y in zip((a.pop(), *a.moments_host()),
                            (b.pop(), *b.moments_host())):
                assert np.array_equal(x, y), (storage, tiled, l, n)
    # one lattice stepped on its own in between: still in lockstep
    batch.advance_per_lattice(2)
    batch.advance(3)
    for a, b in zip(batch.engines, solo):
        b.advance(5)
        assert np.array_equal(a.pop(), b.pop())
    batch.close()
