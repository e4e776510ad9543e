"""The volume-map kernels at the sizes where their dispatch changes, bit for bit against the oracle: meshes of one, a few
and many clusters of 64 triangles (one, two and eight waves per brick of nodes), maps of one cell, of bricks cut by the
map's edge, and a support ball that spans one cell or many."""
import numpy as np
import pytest

from scene_util import make_gpu, make_oracle
from vfd_amd.mesh import TriangleMesh
from vfd_amd.simulation import DFSPHSimulationDescription, RigidBodyDescription

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level,res,r", [(0, (1, 1, 1), 0.05), (0, (9, 2, 5), 0.02), (1, (6, 11, 4), 0.03),
                                         (2, (7, 7, 13), 0.02), (3, (12, 5, 9), 0.012)])
def test_mesh_map_at_dispatch_edges(level, res, r):
    mesh = TriangleMesh.icosphere(level, 0.4, 0.2, 5 + level)
    desc = DFSPHSimulationDescription(ParticleRadius=r)
    body = RigidBodyDescription("mesh", mesh=mesh, resolution=res)
    x = np.zeros((1, 3), np.float32)
    scene = ([desc], [(x, x)], [[body]])
    gpu, orc = make_gpu(*scene), make_oracle(*scene)
    for field in (0, 1):
        g, o = gpu.boundary_map(0, field), orc.boundary_map(0, field)[0].astype(np.float32)
        print(level, res, "field", field, len(g), "nodes, max |diff|", float(np.abs(g - o).max()), flush=True)
        assert np.array_equal(g, o)
