"""The launched solver loops with graphs on - the path of every simulation too large for resident solves, and of batches of
many scenes - under each run-time knob: how the step runs changes, not what it computes."""
import numpy as np
import pytest

from vfd_amd import DFSPHBatch, DFSPHSimulation, scenes
from vfd_amd.simulation import DFSPHSimulationDescription, RigidBodyDescription

pytestmark = pytest.mark.gpu

KNOBS = [dict(HaloLimit=0), dict(HaloLimit="split"), dict(SolverCheckInterval=1), dict(SolverCheckInterval=7, HaloLimit=0),
         dict(PredictIterations=1), dict(PredictIterations=1, SolverCheckInterval=2, HaloLimit="split"),
         dict(UseGraphs=0), dict(UseGraphs=0, HaloLimit=0), dict(UseGraphs=0, HaloLimit="split", SolverCheckInterval=3)]
FIELDS = ("position", "velocity", "density", "factor", "pressure_rho2", "pressure_rho2_v", "viscosity_solution")


def _scene(dims, seed, nu=0.02):
    rng = np.random.default_rng(seed)
    r = 0.01
    x = scenes.lattice_block((3 * r, 2.5 * r, 3 * r), dims, 2 * r, 0.05 * r, rng)
    v = rng.uniform(-0.3, 0.3, size=x.shape).astype(np.float32)
    half = tuple(r * (d + 4) for d in dims)
    desc = DFSPHSimulationDescription(ParticleRadius=r, Viscosity=nu, BoundaryViscosity=nu, EnableSurfaceTensionSolver=0,
                                      MinDivergenceSolverIterations=3, MinPressureSolverIterations=2,
                                      MaxViscositySolverError=0.001)
    box = RigidBodyDescription("box", center=half, half_extents=half, inverted=True, resolution=(12, 12, 12))
    return desc, (x, v), [box]


def _fill(sim, scene):
    sim.set_fluid(*scene[1])
    sim.SetRigidBodies(scene[2])


def _state(sim):
    d = sim.GetDebugInfo()
    return [sim.field(f) for f in FIELDS] + [np.array([
        d.DivergenceSolverIterationCount, d.PressureSolverIterationCount, d.ViscositySolverIterationCount])]


def _knobs(knobs, largest):
    return {k: max(1, largest - 1) if v == "split" else v for k, v in knobs.items()}


def _check_halos(knobs, d):
    if knobs.get("HaloLimit") == 0:
        assert d.StagedGroupCount == 0 and d.GatheredGroupCount > 0
    if knobs.get("HaloLimit") == "split":
        assert d.StagedGroupCount > 0 and d.GatheredGroupCount > 0


def test_knobs_never_change_a_large_scene():
    scene = _scene((65, 64, 64), 1)  # 266,240 particles: more than 1024 for each of 256 CUs

    def run(**knobs):
        sim = DFSPHSimulation(scene[0])
        _fill(sim, scene)
        if knobs:
            sim.set_tuning(**knobs)
        for _ in range(3):
            sim.OnUpdate()
        return sim
    ref = run()
    want, largest = _state(ref), ref.GetDebugInfo().MaxHaloSize
    ref.set_profiling(True)
    ref.OnUpdate()
    assert "div_accel" in ref.profile() and "div_solve" not in ref.profile()
    del ref
    for knobs in KNOBS:
        sim = run(**_knobs(knobs, largest))
        _check_halos(knobs, sim.GetDebugInfo())
        for f, a, b in zip(FIELDS + ("iterations",), _state(sim), want):
            assert np.array_equal(a, b), (knobs, f)
        print(knobs, "the same", flush=True)


def test_knobs_never_change_a_batch_of_many_scenes():
    parts = [_scene((3 + k % 7, 4 + k % 5, 5 + k % 11), k, 0.02 * (1 + k % 9)) for k in range(66)]

    def run(**knobs):
        batch = DFSPHBatch([p[0] for p in parts])
        for s, p in zip(batch.scenes, parts):
            _fill(s, p)
        if knobs:
            batch.set_tuning(**knobs)
        for _ in range(3):
            batch.step()
        return batch
    ref = run()
    want, largest = [_state(s) for s in ref.scenes], ref.scenes[0].GetDebugInfo().MaxHaloSize
    ref.set_profiling(True)
    ref.step()
    assert "div_accel" in ref.profile() and "div_solve" not in ref.profile()
    for knobs in KNOBS:
        batch = run(**_knobs(knobs, largest))
        _check_halos(knobs, batch.scenes[0].GetDebugInfo())
        for k, s in enumerate(batch.scenes):
            for f, a, b in zip(FIELDS + ("iterations",), _state(s), want[k]):
                assert np.array_equal(a, b), (knobs, k, f)
        print(knobs, "the same", flush=True)
