"""Solvers in threads of their own on one GPU, with timing on as by default: the frames are those of the solvers
alone, bit for bit. One solve at a time takes the PCG's one-launch form, the others' run as launches beside it."""
import threading

import numpy as np
import pytest

from luisacomputesimulator_amd import NewtonSolver, pcg_form_counts, scenes

pytestmark = pytest.mark.gpu

MAKE = [lambda: scenes.square_cloth(65), lambda: scenes.cloth_on_sphere(48, 0.02, -0.01, seed=4, height=0.3015),
        lambda: scenes.cylinder_tube(rings=96, per_ring=96, cyl_radius=0.1084, cyl_segments=96, cyl_rings=5),
        lambda: scenes.square_cloth(33)]


def test_solvers_in_threads(require_gpu):
    frames = 4
    alone = []
    for make in MAKE:
        s = NewtonSolver.from_scene(make())
        s.physics_step_gpu(frames)
        alone.append(s.get_simulation_results())
    solvers, before, errors = [NewtonSolver.from_scene(m()) for m in MAKE], pcg_form_counts(), []

    def run(s):
        try:
            for _ in range(frames):
                s.physics_step_gpu(1)
        except Exception as e:  # reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=run, args=(s,)) for s in solvers]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    print(f"[gpu-threads] forms before {before}, after {pcg_form_counts()}", flush=True)
    assert not errors
    for k, (s, x) in enumerate(zip(solvers, alone)):
        assert np.array_equal(s.get_simulation_results(), x), k
        assert s.kernel_times()["pcg"][1] > 0
