"""Surface tension where nearly every particle is a surface candidate, against the oracle: where all of a wave's particles are
candidates, with at most 16 samples each, and there are 24 tiles a sample, a thread samples its own candidate, else a wave
does. Sizes and sample counts on both sides of the rule; the layer's last wave is not full."""
import numpy as np
import pytest

from scene_util import make_gpu, make_oracle
from vfd_amd import DFSPHBatch
from vfd_amd.simulation import DFSPHSimulationDescription

pytestmark = pytest.mark.gpu

R = 0.02
FIELDS = ("mc_surface_normal", "mc_surface_curvature", "mc_surface_normal_smooth", "mc_surface_curvature_smooth")


def _sheet(side, samples, seed):
    """A free layer of side x side particles, two radii apart."""
    rng = np.random.default_rng(seed)
    g = np.stack(np.meshgrid(np.arange(side), [0.0], np.arange(side), indexing="ij"), -1).reshape(-1, 3)
    x = (2.0 * R * g + rng.uniform(-0.2, 0.2, g.shape) * R + 10 * R).astype(np.float32)
    x = np.ascontiguousarray(x[rng.permutation(len(x))])
    desc = DFSPHSimulationDescription(ParticleRadius=R, EnableSurfaceTensionSolver=1, SurfaceTension=0.05, CSDFix=samples,
                                      EnableViscositySolver=0)
    return desc, (x, np.zeros_like(x)), []


@pytest.mark.parametrize("side,samples", [
    (3, 1), (40, 16), (76, 1), (78, 1),      # 23 and 24 tiles
    (109, 2), (111, 2), (134, 3), (136, 3),  # 47 and 49, 71 and 73
    (93, 16), (93, 64), (93, 65),
    (313, 16), (314, 16), (325, 17)])        # 383 and 386 tiles; never from 17 samples on
def test_sheet_matches_the_oracle(side, samples):
    d, f, b = _sheet(side, samples, samples)
    gpu, orc = make_gpu([d], [f], [b]), make_oracle([d], [f], [b])
    gpu.step_until("surface_tension")
    orc.step_until("surface_tension")
    for name in FIELDS:
        assert np.array_equal(gpu.field(name), orc.field(name).astype(np.float32)), (side, samples, name)


def test_scenes_of_a_batch_together_and_alone():
    parts = [_sheet(side, samples, k) for k, (side, samples) in enumerate(((110, 2), (40, 5), (7, 1), (63, 31)))]
    batch = DFSPHBatch([p[0] for p in parts])
    for s, p in zip(batch.scenes, parts):
        s.set_fluid(*p[1])
    batch.scenes[0].step_until("surface_tension")
    for s, p in zip(batch.scenes, parts):
        alone = make_gpu([p[0]], [p[1]], [p[2]])  # fewer tiles: another choice
        alone.step_until("surface_tension")
        for name in FIELDS:
            assert np.array_equal(s.field(name), alone.field(name)), name
