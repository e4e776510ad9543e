"""Volume maps of mesh bodies that stand away from the origin, with bricks of nodes that every edge of the map cuts (lanes
without a node), bit for bit against the oracle."""
import numpy as np
import pytest

from scene_util import make_gpu, make_oracle
from vfd_amd.mesh import TriangleMesh
from vfd_amd.simulation import DFSPHSimulationDescription, RigidBodyDescription

pytestmark = pytest.mark.gpu


def _body(level, shift, resolution):
    m = TriangleMesh.icosphere(level, 0.4, 0.2, 5)
    return RigidBodyDescription("mesh", mesh=TriangleMesh(m.vertices + np.asarray(shift, np.float32), m.triangles),
                                resolution=resolution)


@pytest.mark.parametrize("shift", [(50.0, 0.0, 0.0), (-3.0, 7.0, 0.5)])
def test_map_of_a_body_away_from_the_origin(shift):
    desc = DFSPHSimulationDescription(ParticleRadius=0.02)
    x = np.zeros((1, 3), np.float32)
    scene = ([desc], [(x, x)], [[_body(3, shift, (6, 9, 5))]])  # bricks have four nodes a side
    gpu, orc = make_gpu(*scene), make_oracle(*scene)
    for field in (0, 1):
        g, o = gpu.boundary_map(0, field), orc.boundary_map(0, field)[0].astype(np.float32)
        assert np.array_equal(g, o), (shift, field)
