"""Simulations whose resident solves want the same CUs: two threads, a simulation each, more than half of the chip's blocks
each. A solve that cannot get its blocks is given up and taken again, with the same results as alone."""
import threading
import time

import numpy as np
import pytest

from vfd_amd import DFSPHSimulation, scenes
from vfd_amd.simulation import DFSPHSimulationDescription, RigidBodyDescription

pytestmark = pytest.mark.gpu
STEPS = 40


def _sim(seed):
    rng = np.random.default_rng(seed)
    r = 0.01
    x = scenes.lattice_block((3 * r, 2.5 * r, 3 * r), (56, 56, 56), 2 * r, 0.05 * r, rng)  # 175,616: 172 blocks
    v = rng.uniform(-0.2, 0.2, size=x.shape).astype(np.float32)
    desc = DFSPHSimulationDescription(ParticleRadius=r, Viscosity=0.02, BoundaryViscosity=0.02,
                                      EnableSurfaceTensionSolver=0, MinDivergenceSolverIterations=2,
                                      MinPressureSolverIterations=2)
    box = RigidBodyDescription("box", center=(0.65,) * 3, half_extents=(0.65,) * 3, inverted=True, resolution=(12,) * 3)
    sim = DFSPHSimulation(desc)
    sim.set_fluid(x, v)
    sim.SetRigidBodies([box])
    sim.set_frame_capture(False)
    sim.OnUpdate()
    return sim


def test_two_simulations_on_two_threads_end_as_alone():
    alone = [_sim(k) for k in range(2)]
    t0 = time.perf_counter()
    for s in alone:
        s.advance(STEPS)
    print("one after the other: %.1f ms" % (1e3 * (time.perf_counter() - t0)), flush=True)
    both = [_sim(k) for k in range(2)]
    errors = []

    def run(s):
        try:
            s.advance(STEPS)
        except Exception as e:  # noqa: BLE001 (reported below, in the test's own thread)
            errors.append(e)
    threads = [threading.Thread(target=run, args=(s,)) for s in both]
    t0 = time.perf_counter()
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    print("at once: %.1f ms" % (1e3 * (time.perf_counter() - t0)), flush=True)
    assert not errors, errors
    for a, b in zip(alone, both):
        for f in ("position", "velocity", "density", "pressure_rho2", "viscosity_solution"):
            assert np.array_equal(a.field(f), b.field(f)), f
