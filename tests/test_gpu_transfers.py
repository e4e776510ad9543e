"""What passes between the caller and the particles' slots: fields in the caller's order, read and written, and the
scenes' grids, which travel as a kernel argument or, for more scenes than that holds (four), as a copy."""
import numpy as np
import pytest

from vfd_amd import DFSPHBatch, DFSPHSimulation, scenes
from vfd_amd.simulation import DFSPHSimulationDescription, RigidBodyDescription

pytestmark = pytest.mark.gpu


def _scene(n, seed):
    rng = np.random.default_rng(seed)
    r = 0.02
    side = int(np.ceil(n ** (1.0 / 3.0)))
    x = scenes.lattice_block((3 * r, 2.5 * r, 3 * r), (side, side, side), 2 * r, 0.05 * r, rng)[:n]
    x = np.ascontiguousarray(x[rng.permutation(n)])  # far from the slots' order
    v = rng.uniform(-0.5, 0.5, size=x.shape).astype(np.float32)
    w = 2 * r * (side + 4)
    desc = DFSPHSimulationDescription(ParticleRadius=r, EnableSurfaceTensionSolver=0)
    box = RigidBodyDescription("box", center=(w / 2,) * 3, half_extents=(w / 2,) * 3, inverted=True,
                               resolution=(8, 8, 8))
    return desc, (x, v), [box]


def _fill(sim, scene):
    sim.set_fluid(*scene[1])
    sim.SetRigidBodies(scene[2])


@pytest.mark.parametrize("sizes", [(257,), (1, 256, 700, 255), (300, 0, 1, 513, 40)])
def test_scenes_of_a_batch_and_their_fields(sizes):
    parts = [_scene(n, k) for k, n in enumerate(sizes)]
    batch = DFSPHBatch([p[0] for p in parts])
    alone = []
    for s, p in zip(batch.scenes, parts):
        _fill(s, p)
        alone.append(DFSPHSimulation(p[0]))
        _fill(alone[-1], p)
    for s, p in zip(batch.scenes, parts):  # before any step: the baked particles, in the caller's order
        x, v, _ = s.particles()
        assert np.array_equal(x, p[1][0]) and np.array_equal(v, p[1][1])
    for _ in range(2):
        batch.step()
        for a in alone:
            a.OnUpdate()
    for s, a in zip(batch.scenes, alone):
        for b, c in zip(s.particles(), a.particles()):
            assert np.array_equal(b, c)
        if a.GetParticleCount():
            assert s.GetDebugInfo().TotalNeighborCount == a.GetDebugInfo().TotalNeighborCount
    rng = np.random.default_rng(9)
    wrote = {}
    for k, s in enumerate(batch.scenes):  # each scene's own slots, and no others
        n = s.GetParticleCount()
        wrote[k] = (rng.standard_normal((n, 3)).astype(np.float32), rng.standard_normal(n).astype(np.float32))
        s.set_field("velocity", wrote[k][0])
        s.set_field("delta_final_curvature", wrote[k][1])
    for k, s in enumerate(batch.scenes):
        assert np.array_equal(s.field("velocity"), wrote[k][0])
        assert np.array_equal(s.field("delta_final_curvature"), wrote[k][1])
    with pytest.raises(Exception):
        batch.scenes[0].set_field("density", wrote[0][1])
