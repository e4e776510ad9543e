"""Resident solves where their variants differ - groups of one, two and four tiles, staged, gathered and mixed, lists longer
than the pairs a thread holds in registers - and steps whose solves are given up: alone, in a batch, recorded, partial,
and past the pause that follows. Always the bits of the launched iterations."""
import numpy as np
import pytest

from vfd_amd import DFSPHBatch, DFSPHSimulation, scenes
from vfd_amd.simulation import DFSPHSimulationDescription, RigidBodyDescription

pytestmark = pytest.mark.gpu

FIELDS = ("position", "velocity", "acceleration", "density_advection", "factor", "pressure_rho2", "pressure_rho2_v",
          "pressure_residuum", "viscosity_solution", "velocity_difference", "pressure_acceleration")
COUNTS = ("DivergenceSolverIterationCount", "PressureSolverIterationCount", "ViscositySolverIterationCount",
          "DivergenceSolverError", "PressureSolverError", "ViscositySolverError", "TimeStepSize")


def _scene(n, seed, spacing=2.0, **kw):
    """n particles of a lattice of `spacing` radii in a box with a floor, moving downwards."""
    rng = np.random.default_rng(seed)
    r = 0.01
    side = int(np.ceil(n ** (1.0 / 3.0)))
    x = scenes.lattice_block((3 * r, 2.5 * r, 3 * r), (side, side, side), spacing * r, 0.05 * r, rng)[:n]
    v = rng.uniform(-0.2, 0.2, size=x.shape).astype(np.float32)
    v[:, 1] -= 0.5
    half = (0.5 * spacing * r * (side + 4),) * 3
    desc = DFSPHSimulationDescription(ParticleRadius=r, Viscosity=0.02, BoundaryViscosity=0.02,
                                      EnableSurfaceTensionSolver=0, MinDivergenceSolverIterations=2,
                                      MinPressureSolverIterations=2, **kw)
    box = RigidBodyDescription("box", center=half, half_extents=half, inverted=True, resolution=(12, 12, 12))
    return desc, (x, v), [box]


def _sim(scene, **tuning):
    sim = DFSPHSimulation(scene[0])
    sim.set_fluid(*scene[1])
    sim.SetRigidBodies(scene[2])
    if tuning:
        sim.set_tuning(**tuning)
    return sim


def _same(a, b, what, fields=FIELDS):
    for f in fields:
        x, y = a.field(f), b.field(f)
        assert np.isfinite(y).all() and np.array_equal(x, y), (what, f)
    da, db = a.GetDebugInfo(), b.GetDebugInfo()
    for f in COUNTS:
        assert getattr(da, f) == getattr(db, f), (what, f)


@pytest.mark.parametrize("n,spacing,longest", [
    (4000, 1.5, 70),       # one tile a group: every list at the cap
    (70_000, 1.75, 45),    # two tiles: lists past the 44 pairs held in registers
    (131_073, 2.0, 20),    # four tiles: the fewest particles of that size,
    (262_144, 2.0, 20),    # and a block for every CU
])
def test_group_sizes_match_launched_iterations(n, spacing, longest):
    scene = _scene(n, n, spacing)
    ref = _sim(scene, UseGraphs=0)
    ref.OnUpdate()
    d = ref.GetDebugInfo()
    assert d.MaxNeighborCount >= longest
    staged = _sim(scene)
    staged.set_profiling(True)
    staged.OnUpdate()
    assert staged.profile()["div_solve"][0] == 1 and "div_accel" not in staged.profile()
    e = staged.GetDebugInfo()
    assert e.StagedGroupCount > 0
    sims = {"staged": staged, "mixed": _sim(scene, HaloLimit=max(1, e.MaxHaloSize - 1)), "gathered": _sim(scene, HaloLimit=0)}
    for k in range(2):
        for name, sim in sims.items():
            if k or name != "staged":
                sim.OnUpdate()
            print(n, name, "step", k, flush=True)
            _same(sim, ref, (n, name, k))
        if k == 0:
            m = sims["mixed"].GetDebugInfo()  # (the limit is this step's largest halo less one)
            assert m.GatheredGroupCount > 0 and m.StagedGroupCount > 0
            ref.OnUpdate()


def _given_up(sim):
    """Whether a resident solve was given up in the steps profiled: solves and launched iterations both."""
    p = sim.profile()
    return p.get("div_solve", (0,))[0] > 0 and p.get("div_accel", (0,))[0] > 0


@pytest.mark.parametrize("n", [5000, 40_000, 150_000])  # 20 blocks at one word, 157 and 147 at two levels
def test_solves_given_up_are_taken_again(monkeypatch, n):
    scene = _scene(n, 3)
    ref = _sim(scene, UseGraphs=0)
    monkeypatch.setenv("VFD_RESIDENT_WAIT_US", "0")
    sim = _sim(scene)
    sim.set_profiling(True)
    for k in range(3):
        ref.OnUpdate()
        sim.OnUpdate()
        _same(sim, ref, (n, k))
    assert _given_up(sim)


@pytest.mark.parametrize("us", [1, 4, 5, 6, 7, 16])
def test_whichever_solve_is_given_up(monkeypatch, us):
    """Limits about as long as the waits of a step: the divergence solve may pass and a later one not."""
    scene = _scene(40_000, 5)
    ref = _sim(scene, UseGraphs=0)
    monkeypatch.setenv("VFD_RESIDENT_WAIT_US", str(us))
    sim = _sim(scene)
    sim.set_profiling(True)
    for k in range(3):
        ref.OnUpdate()
        sim.OnUpdate()
        _same(sim, ref, (us, k))
    print(us, "us:", {k: v[0] for k, v in sim.profile().items() if k in ("div_solve", "visc_solve", "pres_solve",
                                                                         "div_accel")}, flush=True)


def test_given_up_in_a_batch(monkeypatch):
    parts = [_scene(n, k, EnableViscositySolver=k % 2) for k, n in enumerate((700, 256, 3001, 1, 9000))]

    def batch(**tuning):
        b = DFSPHBatch([p[0] for p in parts])
        for s, p in zip(b.scenes, parts):
            s.set_fluid(*p[1])
            s.SetRigidBodies(p[2])
        b.set_tuning(**tuning)
        return b
    ref = batch(UseGraphs=0)
    monkeypatch.setenv("VFD_RESIDENT_WAIT_US", "0")
    b = batch(UseGraphs=1)
    b.set_profiling(True)
    for k in range(3):
        ref.step()
        b.step()
        for i, (s, t) in enumerate(zip(b.scenes, ref.scenes)):
            _same(s, t, (i, k))
    assert _given_up(b)


def test_given_up_while_recorded(monkeypatch):
    """The viscosity solve of a recorded step is given up: the step is recorded once, and its adjoint is the same."""
    scene = _scene(20_000, 7)
    rng = np.random.default_rng(8)
    lx = rng.standard_normal(scene[1][0].shape).astype(np.float32)

    def run(**tuning):
        sim = _sim(scene, **tuning)
        sim.set_profiling(True)
        sim.tape(True)
        for _ in range(3):
            sim.OnUpdate()
        return sim, sim.adjoint(lx)
    ref, want = run(UseGraphs=0)
    monkeypatch.setenv("VFD_RESIDENT_WAIT_US", "0")
    sim, got = run()
    p = sim.profile()
    assert p["visc_solve"][0] > 0 and p["cg_matvec"][0] > 0  # given up, and taken again
    _same(sim, ref, "recorded")
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("phase", ["divergence", "viscosity", "pressure"])
def test_given_up_in_a_partial_step(monkeypatch, phase):
    scene = _scene(40_000, 9)
    ref = _sim(scene, UseGraphs=0)
    monkeypatch.setenv("VFD_RESIDENT_WAIT_US", "0")
    sim = _sim(scene)
    sim.set_profiling(True)
    fields = ("position", "velocity", "factor", "pressure_rho2_v", "density")
    for k in range(2):
        ref.step_until(phase)
        sim.step_until(phase)
        for f in fields:
            assert np.array_equal(sim.field(f), ref.field(f)), (phase, k, f)
    assert _given_up(sim)
    ref.OnUpdate()
    sim.OnUpdate()
    _same(sim, ref, phase)


def test_resident_solves_are_tried_again_after_the_pause(monkeypatch):
    scene = _scene(5000, 11)
    ref = _sim(scene, UseGraphs=0)
    monkeypatch.setenv("VFD_RESIDENT_WAIT_US", "0")
    sim = _sim(scene)
    sim.set_profiling(True)
    for _ in range(70):
        ref.OnUpdate()
        sim.OnUpdate()
    _same(sim, ref, "past the pause")
    assert sim.profile()["div_solve"][0] == 2  # the first step, 64 without, one more, 128 without
