"""The PCG in one launch (k_pcg_grid) against the same iterations as three launches each: the sums
are taken over the same partition in the same order, so positions and iteration counts are equal bit
for bit, frame by frame, without and in contact, in every precision. set_graphs(False) selects the
launches; a solver left alone takes the one-launch form wherever the system fits it."""
import numpy as np
import pytest

from luisacomputesimulator_amd import BsrSystem, LcsxError, NewtonSolver, pcg_form_counts, pcg_solve_bsr, scenes

pytestmark = pytest.mark.gpu


def boxes():
    sc = scenes.cloth_rigid_coupling(n=17, boxes=2, seed=3, box_region=((-0.25, 0.25), (0.32, 0.5), (-0.25, 0.25)))
    for m in sc.meshes[1:]:
        m.verts[:, 1] -= np.float32(m.verts[:, 1].min() - (0.2 + 1.3e-3))
    return sc


def spring():
    sc = scenes.square_cloth(21)
    sc.meshes[0].material.stretch_model = "Spring"
    return sc


def tube_on_ring():
    """A tube in contact with a short piece of its cylinder: a few thousand contact slots."""
    sc = scenes.cylinder_tube(rings=96, per_ring=96, cyl_radius=0.1084, cyl_segments=96, cyl_rings=5)
    n = len(sc.meshes[0].verts)
    sc.meshes[1].verts[:, 0] *= np.float32(0.05)
    sc.initial_position[n:, 0] *= np.float32(0.05)
    return sc


def irregular(n):
    """A cloth of randomly moved grid points and their Delaunay triangles on a sphere: rows of up to 20 blocks."""
    from scipy.spatial import Delaunay

    sc = scenes.cloth_on_sphere(n, 0.02, -0.01, seed=4, sphere_subdiv=3, height=0.3015)
    m, rng = sc.meshes[0], np.random.default_rng(0)
    g = np.stack(np.meshgrid(np.arange(n), np.arange(n), indexing="ij"), -1).reshape(-1, 2).astype(float)
    inner = ((g > 0) & (g < n - 1)).all(1)
    g[inner] += rng.uniform(-0.48, 0.48, size=(int(inner.sum()), 2))
    v, t = m.verts.copy(), Delaunay(g).simplices.astype(np.int32)
    v[:, 0], v[:, 2] = g[:, 1] / (n - 1) - 0.5, g[:, 0] / (n - 1) - 0.5
    a, b = g[t[:, 1]] - g[t[:, 0]], g[t[:, 2]] - g[t[:, 0]]
    area = np.abs(a[:, 0] * b[:, 1] - a[:, 1] * b[:, 0])
    m.verts, m.tris = v.astype(np.float32), t[area > 1e-6]
    return sc


# rows: less than one 64-row chunk, one row past it, several workgroups, many, and above 65,536 rows (two row
# blocks per workgroup) without and with contacts
CASES = {
    "square_7": (lambda: scenes.square_cloth(7), 3),
    "square_33": (lambda: scenes.square_cloth(33), 3),
    "square_65x": (lambda: scenes.twisting_sheet(65), 2),
    "spring_21": (spring, 3),
    "sphere_24": (lambda: scenes.cloth_on_sphere(24, 0.02, -0.01, seed=4, sphere_subdiv=2, height=0.3015), 5),
    "tube_41x48": (lambda: scenes.cylinder_tube(rings=41, per_ring=48, cyl_segments=24, cyl_rings=9), 5),
    "tube_contact": (tube_on_ring, 2),
    "boxes": (boxes, 4),
    "square_257": (lambda: scenes.square_cloth(257), 1),
    "sphere_257": (lambda: scenes.cloth_on_sphere(257, 0.02, -0.01, seed=4, sphere_subdiv=2, height=0.3015), 2),
}


@pytest.mark.parametrize("precision", ["fp32", "mixed", "mixed_bf16"])
@pytest.mark.parametrize("name", list(CASES))
def test_one_launch_equals_launches(require_gpu, name, precision):
    make, frames = CASES[name]

    def solver():
        sc = make()
        sc.params.precision = precision
        return NewtonSolver.from_scene(sc)

    one, launches = solver(), solver()
    launches.set_graphs(False)
    contacts = 0
    for f in range(frames):
        _, form = counted(lambda: one.physics_step_gpu(1))
        launches.physics_step_gpu(1)
        assert set(form) <= {"one_launch"}
        # (the tubes' later frames have more contacts than it takes)
        assert form == {"one_launch": one.stats()["newton_iters"]} or (name in ("tube_41x48", "tube_contact") and f > 0)
        a, b = one.stats(), launches.stats()
        contacts = max(contacts, a["num_contacts"])
        print(f"[gpu-grid] {name} {precision} frame {f}: Newton {a['newton_iters']}/{b['newton_iters']}, "
              f"PCG {a['pcg_iters_total']}/{b['pcg_iters_total']}, contacts {a['num_contacts']}", flush=True)
        assert a["newton_iters"] == b["newton_iters"] and a["pcg_iters_total"] == b["pcg_iters_total"]
        assert a["pcg_rel"] == b["pcg_rel"]
        assert np.array_equal(one.get_simulation_results(), launches.get_simulation_results())
        assert np.array_equal(one.get_velocities(), launches.get_velocities())
    assert one.kernel_times()["pcg_grid"][1] > 0 and "pcg_grid" not in launches.kernel_times()
    if name in ("tube_contact", "sphere_24", "boxes", "sphere_257"):
        assert contacts > 0


def batch(sizes):
    return [scenes.square_cloth(n, seed=k) if k % 2 else
            scenes.cloth_on_sphere(n, 0.02, -0.01, seed=k, sphere_subdiv=2, height=0.3015) for k, n in enumerate(sizes)]


# rows of 17 to 32 blocks: in contact up to 20 row blocks, or 64 of 16-bit blocks
@pytest.mark.parametrize("n,precision,one", [(33, "fp32", True), (33, "mixed", True), (112, "fp32", False),
                                             (112, "mixed_bf16", True)])
def test_rows_of_an_irregular_mesh(require_gpu, n, precision, one):
    def solver(collide=True):
        sc = irregular(n)
        sc.params.precision, sc.params.use_self_collision = precision, collide
        return NewtonSolver.from_scene(sc)

    a, b, c = solver(), solver(), solver(False)
    csr = a.read("csr").astype(np.int64)
    width = int(np.diff(csr[:a.num_verts + 1]).max())
    assert 16 < width <= 32
    b.set_graphs(False)
    forms = {}
    for f in range(2):
        _, form = counted(lambda: a.physics_step_gpu(1))
        b.physics_step_gpu(1)
        forms = {k: forms.get(k, 0) + v for k, v in form.items()}
        assert a.stats()["pcg_iters_total"] == b.stats()["pcg_iters_total"]
        assert np.array_equal(a.get_simulation_results(), b.get_simulation_results())
    print(f"[gpu-grid] irregular {n} {precision}: rows of {width}, {a.stats()['num_contacts']} contacts, {forms}", flush=True)
    assert a.stats()["num_contacts"] > 0
    assert set(forms) == ({"one_launch"} if one else set())
    assert set(counted(lambda: c.physics_step_gpu(1))[1]) == {"one_launch"}  # without contacts, whatever the size


def test_forms_of_the_launches_and_back(require_gpu):
    """set_graphs and set_spmv_shape choose the launches, before or after the solver is initialised, and
    set_one_launch the default form again; with graphs the solves that fit run in one launch all the same."""
    def forms(g):
        return set(counted(lambda: g.physics_step_gpu(1))[1])

    g = NewtonSolver.from_scene(scenes.square_cloth(17))
    assert forms(g) == {"one_launch"}
    for choose in (lambda: g.set_graphs(False), lambda: g.set_spmv_shape(3), lambda: g.set_one_launch(False),
                   lambda: g.set_graphs(True)):
        choose()
        assert forms(g) == set()
        g.set_one_launch()
        assert forms(g) == {"one_launch"}
    sc = scenes.square_cloth(17)
    h = NewtonSolver(sc.params)
    mid = h.register_mesh("square", sc.meshes[0].verts, sc.meshes[0].tris, sc.meshes[0].material)
    h.set_graphs(False)
    h.init_solver()
    assert mid == 0 and forms(h) == set()
    with pytest.raises(LcsxError):
        g.set_one_launch(2)


@pytest.mark.parametrize("name", ["square_33", "tube_contact", "square_257"])
def test_a_wait_that_runs_out_starts_over(require_gpu, name):
    """One workgroup of the first solve is not launched, so the others' waits for it run out and they end (about
    0.14 s); the solve is the launches' then, bit for bit, and the next ones run in one launch again."""
    a, b = (NewtonSolver.from_scene(CASES[name][0]()) for _ in range(2))
    b.set_graphs(False)
    a.stage("withhold_workgroup")
    (_, forms), _ = counted(lambda: a.physics_step_gpu(1)), b.physics_step_gpu(1)
    assert forms == {"waited": 1, "one_launch": a.stats()["newton_iters"] - 1}
    assert a.kernel_times()["pcg_grid_gave_up"][1] == 1
    assert np.array_equal(a.get_simulation_results(), b.get_simulation_results())


def test_an_iteration_cap_of_all_integers(require_gpu):
    """pcg_iter_count as a program sets it that wants no cap: every solve takes as many epochs of the exchanged
    words as its cap, so they are cleared before the numbers run out. Two solves without contacts, whose numbers
    end a wrap, then one with contacts (words that no solve has written yet), and again."""
    def solver(cap):
        sc = tube_on_ring()
        sc.params.pcg_iter_count, sc.params.pcg_check_every, sc.params.pcg_rel_tol = cap, 1, 1e-3
        return NewtonSolver.from_scene(sc)

    a, b = solver(2 ** 31 - 1), solver(1000)
    b.set_graphs(False)
    for rep in range(3):
        for s in ("frame_begin", "predict", "iter_begin", "material", "pcg", "pcg", "update_contacts", "contact_assemble",
                  "pcg"):
            b.stage(s)
            assert b.stats()["pcg_iters"] < 1000  # so does a, whose iterations are the same
            _, form = counted(lambda: a.stage(s))
            assert form == ({"one_launch": 1} if s == "pcg" else {})
            assert s != "pcg" or np.array_equal(a.read("dx"), b.read("dx")), rep
        contacts = len(b.read("contact_idx")) // 4
        print(f"[gpu-grid] cap 2^31 - 1: {b.stats()['pcg_iters']} iterations, {contacts} contacts", flush=True)
        assert contacts > 0


def test_a_refused_lease_takes_the_launches(require_gpu):
    """While another solve of the process holds the device's one-launch form (its lease is taken here through the
    library's C++ symbols), solvers' and block-CSR solves run as launches, with the same bits."""
    import ctypes as C

    from luisacomputesimulator_amd import load_library

    lib = load_library()
    take, drop = lib._ZN4lcsx9GridLease4takeEi, lib._ZN4lcsx9GridLeaseD1Ev
    take.restype, take.argtypes, drop.restype, drop.argtypes = C.c_bool, [C.c_void_p, C.c_int], None, [C.c_void_p]
    sysm, _, b = banded(1000, 6, 3)
    solve = lambda: pcg_solve_bsr(sysm, b.astype(np.float32), max_iters=60, check_every=1, abs_tol=0.0)
    (x, res), form = counted(solve)
    assert form == {"one_launch": 1}
    g, h = (NewtonSolver.from_scene(CASES["tube_contact"][0]()) for _ in range(2))
    g.physics_step_gpu(1)
    lease = C.c_int(-1)
    assert take(C.byref(lease), 0)
    try:
        (y, launched), form = counted(solve)
        _, forms = counted(lambda: h.physics_step_gpu(1))
    finally:
        drop(C.byref(lease))
    assert form == {"refused": 1} and set(forms) == {"refused"}
    assert np.array_equal(x, y) and res == launched
    assert np.array_equal(g.get_simulation_results(), h.get_simulation_results())


# scenes of unequal sizes in one launch, scenes dealt to two, and more rows than two launches hold
@pytest.mark.parametrize("sizes,one_launch", [((2, 9, 33, 17, 24), True), ((220, 33, 220, 221), True),
                                              ((220,) * 6, False)])
def test_batch_one_launch_equals_launches(require_gpu, sizes, one_launch):
    one, launches = (NewtonSolver.from_scenes(batch(sizes)) for _ in range(2))
    launches.set_graphs(False)
    frames, contacts = 4 if max(sizes) < 100 else 1, 0
    for f in range(frames):
        one.physics_step_gpu(1)
        launches.physics_step_gpu(1)
        contacts = max(contacts, one.stats()["num_contacts"])
        print(f"[gpu-grid] batch {sizes} frame {f}: {one.stats()['pcg_iters_total']}, {contacts} contacts", flush=True)
        assert one.stats()["pcg_iters_total"] == launches.stats()["pcg_iters_total"]
        assert np.array_equal(one.get_simulation_results(), launches.get_simulation_results())
    assert contacts > 0 and ("pcg_grid" in one.kernel_times()) == one_launch


def banded(n, half, seed):
    """A diagonally dominant block-CSR system: row i has the columns i - half .. i + half but itself."""
    rng = np.random.default_rng(seed)
    i = np.repeat(np.arange(n), 2 * half)
    c = i + np.tile(np.concatenate([np.arange(-half, 0), np.arange(1, half + 1)]), n)
    keep = (c >= 0) & (c < n)
    i, c = i[keep], c[keep]
    lo, hi = np.minimum(i, c), np.maximum(i, c)
    v = np.stack([np.sin(lo * 12.9898 + hi * 78.233 + k) for k in range(3)], -1)
    blocks = -(v[:, :, None] * v[:, None, :]).astype(np.float32)
    diag = np.zeros((n, 3, 3))
    np.add.at(diag, i, -blocks.astype(np.float64))
    diag += 0.05 * np.eye(3)
    ptr = np.concatenate([[0], np.cumsum(np.bincount(i, minlength=n))])
    return BsrSystem(ptr, c, blocks, diag.astype(np.float32)), (i, c, blocks, diag), rng.normal(size=(n, 3))


def counted(fn):
    """fn's result, and the forms of the PCG that it was counted in."""
    before = pcg_form_counts()
    out = fn()
    return out, {k: v - before[k] for k, v in pcg_form_counts().items() if v != before[k]}


def widened(ptr, cols, blocks, diag):
    """The same system with 40 zero blocks more in its last row: wider than any one-launch shape, so the solve
    takes the launches, where a zero block adds nothing."""
    extra = np.arange(40) % (len(ptr) - 1)
    ptr = ptr.copy()
    ptr[-1] += len(extra)
    return BsrSystem(ptr, np.concatenate([cols, extra]), np.concatenate([blocks, np.zeros((40, 3, 3), np.float32)]), diag)


# one row, around a row block's and a workgroup's edge, two row blocks per workgroup (above 65536), and
# rows wider than any shape holds (24 blocks a row above 65536 rows, 40 below)
@pytest.mark.parametrize("n,half", [(1, 1), (255, 2), (256, 6), (257, 6), (1000, 6), (1025, 11), (65536, 6), (65537, 6),
                                    (131072, 3), (70000, 12), (3000, 20)])
def test_block_csr_solve(require_gpu, n, half):
    """The residual of 100 iterations against the FP64 recurrence's own, and the solution against the
    64-bit iterate (1e-4: 100 FP32 iterations of a system of condition below 1e3). The form that ran, and the
    launches' bits."""
    sysm, (i, c, blocks, diag), b = banded(n, half, n)
    b = b.astype(np.float32)
    (x, res), form = counted(lambda: pcg_solve_bsr(sysm, b, max_iters=100, check_every=25, abs_tol=0.0))
    # (the shapes are for a mean of up to 24 blocks a row, or 12 above 65,536 rows)
    one = len(c) <= (24 if n <= 65536 else 12) * n
    assert form == ({"one_launch": 1} if one else {})
    if one:
        ptr = np.concatenate([[0], np.cumsum(np.bincount(i, minlength=n))])
        wide = widened(ptr, c, blocks, diag.astype(np.float32))
        (y, launched), form = counted(lambda: pcg_solve_bsr(wide, b, max_iters=100, check_every=25, abs_tol=0.0))
        # (40 blocks more in a tiny matrix are more than any shape's mean)
        assert form == ({"unfit": 1} if len(c) + 40 <= (24 if n <= 65536 else 12) * n else {})
        assert np.array_equal(x, y) and res == launched
    B, D, inv = blocks.astype(np.float64), diag.astype(np.float32).astype(np.float64), None
    inv = np.linalg.inv(D)

    def mul(p):
        y = np.einsum("nij,nj->ni", D, p)
        q = np.einsum("nij,nj->ni", B, p[c])
        for d in range(3):
            y[:, d] += np.bincount(i, weights=q[:, d], minlength=n)
        return y

    xr, r, p, old = np.zeros((n, 3)), b.astype(np.float64), np.zeros((n, 3)), None
    for _ in range(100):
        z = np.einsum("nij,nj->ni", inv, r)
        rz = float((r * z).sum())
        p = z + (0.0 if old is None or old < 1e-10 else rz / old) * p
        q = mul(p)
        pq = float((p * q).sum())
        a = 0.0 if pq < 1e-10 else rz / pq
        xr, r, old = xr + a * p, r - a * q, rz
    err = np.linalg.norm(x - xr) / np.linalg.norm(xr)
    print(f"[gpu-grid] block CSR n {n}, {2 * half} blocks a row: {res}, error against 64 bits {err:.2e}", flush=True)
    assert res["iters"] == 100 and err < 1e-4


def named_rows(ptr, cols, rows):
    """The most rows outside its own that the columns of one workgroup (of `rows` rows) name."""
    n, most = len(ptr) - 1, 0
    for r in range(0, n, rows):
        c = np.unique(cols[ptr[r]:ptr[min(r + rows, n)]])
        most = max(most, int(np.count_nonzero((c < r) | (c >= r + rows))))
    return most


# columns all over the matrix: a workgroup of 256 rows holds p of 3,840 others, one of 512 rows (above 65,536
# rows) of 3,584; the last two fit
@pytest.mark.parametrize("n,width,fits", [(60000, 20, False), (100000, 10, False), (20000, 14, True), (70000, 6, True)])
def test_block_csr_scattered_columns(require_gpu, n, width, fits):
    """A workgroup that names more rows than it can hold gives up before it reads any of them, and the solve is
    the launches'. Bit for bit against the launches, and against the dominance of the diagonal."""
    rng = np.random.default_rng(n + width)
    i = np.repeat(np.arange(n), width)
    c = rng.integers(0, n, size=i.size)
    c = np.where(c == i, (c + 1) % n, c)
    ptr = np.arange(n + 1) * width
    room = 3840 if n <= 65536 else 3584
    named = named_rows(ptr, c, 4096 - room)
    print(f"[gpu-grid] scattered n {n}, {width} blocks a row: {named} rows named, room for {room}", flush=True)
    assert (named <= room) == fits
    blocks = np.tile(-0.01 * np.eye(3, dtype=np.float32), (i.size, 1, 1))
    blocks *= (1.0 + 0.5 * np.sin(np.arange(i.size, dtype=np.float32)))[:, None, None]
    diag = np.tile(np.eye(3, dtype=np.float32), (n, 1, 1))
    b = rng.normal(size=(n, 3)).astype(np.float32)
    opt = dict(max_iters=4, check_every=4, abs_tol=0.0)
    (x, res), form = counted(lambda: pcg_solve_bsr(BsrSystem(ptr, c, blocks, diag), b, **opt))
    assert form == ({"one_launch": 1} if fits else {"unfit": 1})
    assert res["iters"] == 4 and np.isfinite(x).all()
    y, launched = pcg_solve_bsr(widened(ptr, c, blocks, diag), b, **opt)
    assert np.array_equal(x, y) and res == launched
    # the matrix is not symmetric: only that four iterations reduce the residual as the dominance says
    r = b - x.astype(np.float64)
    for d in range(3):
        r[:, d] -= np.bincount(i, weights=blocks[:, d, d].astype(np.float64) * x[c, d], minlength=n)
    assert np.linalg.norm(r) < 0.02 * np.linalg.norm(b)


def test_shuffled_cloth_takes_the_launches(require_gpu):
    """A cloth whose vertices are numbered at random, as a mesh file may have them: the one-launch form gives up
    in its first solve, and the frame is the launches', bit for bit."""
    def solver():
        sc = scenes.square_cloth(257)
        m, perm = sc.meshes[0], np.random.default_rng(7).permutation(257 * 257)
        place = np.empty_like(perm)
        place[perm] = np.arange(len(perm))
        m.verts, m.tris = m.verts[perm], place[m.tris].astype(np.int32)
        return NewtonSolver.from_scene(sc)

    one, launches = solver(), solver()
    csr = one.read("csr").astype(np.int64)
    n = 257 * 257
    named = named_rows(csr[:n + 1] - (n + 1), csr[n + 1:], 512)
    print(f"[gpu-grid] shuffled cloth: {named} rows named", flush=True)
    assert named > 3584
    launches.set_graphs(False)
    for g in (one, launches):
        g.physics_step_gpu(1)
    assert one.stats()["pcg_iters_total"] == launches.stats()["pcg_iters_total"]
    assert one.kernel_times()["pcg_grid"][1] == 1 and one.kernel_times()["pcg_grid_gave_up"][1] == 1
    assert np.array_equal(one.get_simulation_results(), launches.get_simulation_results())


def test_block_csr_bad_index_in_the_middle(require_gpu):
    sysm, _, b = banded(2000, 4, 1)
    ok = sysm._dev[1].host.copy()
    bad = BsrSystem(sysm._dev[0].host, np.where(np.arange(len(ok)) == 8003, 2000, ok), sysm._dev[2].host,
                    sysm._dev[3].host)
    with pytest.raises(LcsxError, match="outside the matrix"):
        pcg_solve_bsr(bad, b.astype(np.float32))
