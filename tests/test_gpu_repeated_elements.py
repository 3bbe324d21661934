"""Contacts with a collider mesh that lists a triangle twice, has an edge of three triangles and triangles that
name a vertex twice, as mesh files have them: contacts of one row then have equal vertex ids, or one contact
names a row twice. The contact gradient and Hessian against the oracle, and the same bits in two solvers."""
import numpy as np
import pytest

import oracle
from luisacomputesimulator_amd import NewtonSolver, scenes

pytestmark = pytest.mark.gpu


def scene():
    sc = scenes.small_two_sheets(9, gap=0.7e-3)
    collider, cloth = sc.meshes
    collider.fixed = [scenes.FixedPoints("All")]
    t = collider.tris
    collider.tris = np.concatenate([t, [[i, i, i + 1] for i in (12, 20, 32, 40, 49)], t[60:64], [[30, 31, 50]]]).astype(np.int32)
    cloth.verts = cloth.verts + np.array([-0.003, 0.0, 0.006], np.float32)  # its edges pass over the collider's vertices
    cloth.fixed = [scenes.FixedPoints("LeftBack", 0.001)]
    sc.meshes = [cloth, collider]  # an edge pair is kept from the earlier edge: the collider's come later
    return sc


def test_contacts_of_repeated_elements(require_gpu):
    solvers = [NewtonSolver.from_scene(scene()) for _ in range(2)]
    o = oracle.Oracle(scene(), 32)
    for s in ("frame_begin", "predict", "iter_begin", "material", "update_contacts", "contact_assemble"):
        for h in (*solvers, o):
            h.stage(s)
    idx, typ = o.get("contact_idx").reshape(-1, 4), o.get("contact_type").reshape(-1, 1)
    twice = sum(len(set(c.tolist())) < 4 for c in idx)
    key, count = np.unique(np.concatenate([typ, idx], 1), axis=0, return_counts=True)
    print(f"[gpu-repeats] {len(idx)} contacts, {twice} name a row twice, {np.count_nonzero(count > 1)} keys are shared",
          flush=True)
    assert twice > 0 and np.count_nonzero(count > 1) > 0
    a, b = solvers
    own = np.concatenate([a.read("contact_type").reshape(-1, 1), a.read("contact_idx").reshape(-1, 4)], 1)
    assert np.array_equal(np.unique(own, axis=0), key) and len(own) == len(idx)
    free = np.flatnonzero(o.get("is_fixed") == 0)  # (a pinned row's own terms hide the contact's)
    # sums of up to 30 FP32 terms in another order, barrier terms within a few ulps
    for name, width in (("cgB", 3), ("diag", 9)):
        got, ref = a.read(name).reshape(-1, width)[free], o.get(name).reshape(-1, width)[free]
        err = np.abs(got - ref).max() / np.abs(ref).max()
        print(f"[gpu-repeats] {name}: {err:.2e}", flush=True)
        assert err < 2e-5
        assert np.array_equal(a.read(name), b.read(name))
    for frame in range(4):
        for g in solvers:
            g.physics_step_gpu(1)
        assert np.isfinite(a.get_simulation_results()).all()
        assert np.array_equal(a.get_simulation_results(), b.get_simulation_results())
    b.set_graphs(False)  # the launches against the one-launch form
    for frame in range(2):
        for g in solvers:
            g.physics_step_gpu(1)
        assert np.array_equal(a.get_simulation_results(), b.get_simulation_results())
