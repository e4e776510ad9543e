"""The resident solvers (one launch per solve, vfd_amd/csrc/solve.hip) against the launched iterations they stand for:
the same bits, whatever the number of blocks, tiles and scenes, with staged and gathered groups, and when a barrier's
limit aborts every solve that has to wait."""
import numpy as np
import pytest

from vfd_amd import DFSPHBatch, DFSPHSimulation, scenes
from vfd_amd.simulation import DFSPHSimulationDescription, RigidBodyDescription

pytestmark = pytest.mark.gpu

FIELDS = ("position", "velocity", "acceleration", "density_advection", "factor", "pressure_rho2", "pressure_rho2_v",
          "pressure_residuum", "viscosity_solution", "velocity_difference", "pressure_acceleration")


def _scene(n, seed, visc=1):
    """n particles of a lattice one support radius off a box's corner, falling on its floor."""
    rng = np.random.default_rng(seed)
    r = 0.02
    side = int(np.ceil(n ** (1.0 / 3.0)))
    x = scenes.lattice_block((3 * r, 2.5 * r, 3 * r), (side, side, side), 2 * r, 0.05 * r, rng)[:n]
    v = rng.uniform(-0.5, 0.5, size=x.shape).astype(np.float32)
    v[:, 1] -= 1.0
    w = 2 * r * (side + 4)
    desc = DFSPHSimulationDescription(ParticleRadius=r, Viscosity=0.02, BoundaryViscosity=0.02,
                                      EnableViscositySolver=visc, EnableSurfaceTensionSolver=0,
                                      MinDivergenceSolverIterations=2, MinPressureSolverIterations=2)
    box = RigidBodyDescription("box", center=(w / 2,) * 3, half_extents=(w / 2,) * 3, inverted=True,
                               resolution=(12, 12, 12))
    return desc, (x, v), [box]


def _sim(scene):
    sim = DFSPHSimulation(scene[0])
    sim.set_fluid(*scene[1])
    sim.SetRigidBodies(scene[2])
    return sim


def _same(a, b, what):
    for f in FIELDS:
        assert np.array_equal(a.field(f), b.field(f)), (what, f)
    da, db = a.GetDebugInfo(), b.GetDebugInfo()
    for f in ("DivergenceSolverIterationCount", "PressureSolverIterationCount", "ViscositySolverIterationCount",
              "DivergenceSolverError", "PressureSolverError", "ViscositySolverError", "TimeStepSize"):
        assert getattr(da, f) == getattr(db, f), (what, f)


@pytest.mark.parametrize("n", [1, 255, 257, 1023, 1025, 5000, 66_000])
def test_resident_solves_match_launched_iterations(n):
    scene = _scene(n, n)
    ref = _sim(scene)
    ref.set_tuning(UseGraphs=0)  # every iteration launched
    sims = {"staged": _sim(scene), "gathered": _sim(scene)}
    sims["gathered"].set_tuning(HaloLimit=0)
    for k in range(2):
        ref.OnUpdate()
        for name, sim in sims.items():
            sim.OnUpdate()
            print(n, name, "step", k, flush=True)
            _same(sim, ref, (n, name, k))


def test_resident_batch_matches_launched_iterations():
    parts = [_scene(n, k, visc=k % 2) for k, n in enumerate((700, 0, 256, 3001, 1, 5000))]
    batches = []
    for graphs in (1, 0):
        b = DFSPHBatch([p[0] for p in parts])
        for s, p in zip(b.scenes, parts):
            s.set_fluid(*p[1])
            s.SetRigidBodies(p[2])
        b.set_tuning(UseGraphs=graphs)
        batches.append(b)
    for k in range(3):
        for b in batches:
            b.step()
        for s, p in enumerate(parts):
            if len(p[1][0]):
                _same(batches[0].scenes[s], batches[1].scenes[s], (s, k))
        print("batch step", k, flush=True)


def test_aborted_solves_are_taken_again(monkeypatch):
    """With no time to wait at a barrier every solve of several blocks is aborted (each wave still leaves its launch) and
    the step runs again with launched iterations; the results are the same and the simulation goes on."""
    scene = _scene(5000, 3)
    ref = _sim(scene)
    ref.set_tuning(UseGraphs=0)
    monkeypatch.setenv("VFD_RESIDENT_WAIT_US", "0")
    sim = _sim(scene)
    for k in range(3):
        ref.OnUpdate()
        sim.OnUpdate()
        _same(sim, ref, k)
        print("aborted step", k, flush=True)
