"""The two builds of the neighbour lists (a lane per row of cells where the chip is not full, a thread per particle
otherwise) against each other: the same particles alone and in a batch whose second scene fills the chip."""
import numpy as np
import pytest

from vfd_amd import DFSPHBatch, DFSPHSimulation, scenes
from vfd_amd.simulation import DFSPHSimulationDescription

pytestmark = pytest.mark.gpu
R = 0.02


def _lattice(n, spacing, jitter, seed):
    side = int(np.ceil(n ** (1.0 / 3.0)))
    rng = np.random.default_rng(seed)
    x = scenes.lattice_block((0.1, 0.1, 0.1), (side, side, side), spacing * R, jitter * R, rng)[:n]
    return np.ascontiguousarray(x[rng.permutation(n)])


@pytest.mark.parametrize("n,spacing,jitter", [
    (1, 2.0, 0.0), (15, 2.0, 0.1), (17, 2.0, 0.1), (255, 2.0, 0.2), (257, 2.0, 0.0), (3000, 1.8, 0.3),
    (2000, 1.2, 0.3),   # rows past 64 candidates, lists past the cap of 70
    (700, 0.5, 0.2),    # hundreds of candidates a row, every list full
    (2000, 9.0, 4.0),   # scattered
    (128 * 256, 2.0, 0.1),  # the largest of the one build, and one particle more
    (128 * 256 + 1, 2.0, 0.1),
])
def test_both_builds_give_the_same_lists(n, spacing, jitter):
    desc = DFSPHSimulationDescription(ParticleRadius=R, EnableSurfaceTensionSolver=0)
    x = _lattice(n, spacing, jitter, n)
    alone = DFSPHSimulation(desc)
    alone.set_fluid(x, np.zeros_like(x))
    batch = DFSPHBatch([desc, desc])
    filler = _lattice(40_000, 2.0, 0.1, 3)
    for s, p in zip(batch.scenes, (x, filler)):
        s.set_fluid(p, np.zeros_like(p))
    alone.step_until("search")
    batch.scenes[0].step_until("search")
    for a, b in zip(alone.neighbors(), batch.scenes[0].neighbors()):
        assert np.array_equal(a, b)
    da, db = alone.GetDebugInfo(), batch.scenes[0].GetDebugInfo()
    counts = alone.neighbors()[0]
    assert da.TotalNeighborCount == db.TotalNeighborCount == int(np.sum(counts))
    assert da.MaxNeighborCount == db.MaxNeighborCount == int(np.max(counts))
