"""When the broad phase walks the solver's own hierarchies (host setup, no GPU needed): not for the edges or faces of
scenes with more than 64 blocks over several separate pieces, nor for batches of more than 64 blocks that are less
than a quarter full."""
import numpy as np
import pytest

from luisacomputesimulator_amd import LcsxError, NewtonSolver, scenes
from test_gpu_cluster_query import patches


def use(scs):
    s = NewtonSolver(scs[0].params)
    for k, sc in enumerate(scs):
        if k:
            s.begin_scene()
        for m in sc.meshes:
            mid = s.register_mesh(m.name, m.verts, m.tris, m.material)
            for fp in m.fixed:
                s.add_fixed_points(mid, fp.method, fp.range, fp.anim)
    try:
        s.init_solver()
    except LcsxError as e:
        if "error 7" not in str(e):  # LCSX_ERR_NO_GPU on a CPU-only host
            raise
    return s.read("cluster_use").tolist()


@pytest.mark.parametrize("name,want", [("tube", [1, 1]), ("boxes", [1, 1]), ("batch", [1, 1])])
def test_the_repositorys_workloads_walk_the_hierarchies(name, want):
    scs = {"tube": lambda: [scenes.cylinder_tube()], "boxes": lambda: [scenes.cloth_rigid_coupling(33, 24)],
           "batch": lambda: scenes.sphere_batch(80, 0, 17, 40)}[name]()
    assert use(scs) == want


def test_separate_pieces():
    # 16 edges and 8 faces a piece: 64 blocks of edges, one more with two pieces in it, then of faces
    assert use([patches(4096)]) == [1, 1]
    assert use([patches(4098)]) == [1, 0]
    assert use([patches(8192)]) == [1, 0]
    assert use([patches(8194)]) == [0, 0]
    # as one mesh each (the blocks are the same)
    sc = patches(4098)
    m = sc.meshes[0]
    sc.meshes = [scenes.Mesh(f"p{k}", m.verts[9 * k:9 * k + 9], m.tris[:8], m.material, []) for k in range(4098)]
    assert use([sc]) == [1, 0]


def test_tiny_scenes():
    assert use([scenes.square_cloth(3, seed=k) for k in range(64)]) == [1, 1]
    assert use([scenes.square_cloth(3, seed=k) for k in range(65)]) == [0, 0]
    assert use([scenes.square_cloth(11, seed=k) for k in range(65)]) == [0, 1]  # 200 faces, 320 edges
    assert use([scenes.square_cloth(13, seed=k) for k in range(65)]) == [1, 1]
