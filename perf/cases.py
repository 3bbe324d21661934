"""The work that users of this framework have it do, as cases that can be timed and compared.

Kinds of cases, each through public entry points:

  spmv      y = A x on a caller's own block-CSR matrix (lcsx_spmv_bsr): a solver of the caller's.
  pcg       a caller's own block system solved by the block-Jacobi PCG (lcsx_pcg_solve_bsr).
  sweep     continuous collision of moving meshes outside the solver: tree construction, refit on the
            swept boxes, the query and the CCD step bound (lcsx_lbvh_*, lcsx_ccd_pairs), vertices
            against faces or edges against edges; the pairs are sorted, as a program does that needs
            them in an order that does not change from run to run.
  frame     one simulated frame from a state that the program sets (NewtonSolver.set_state,
            physics_step_gpu, get_simulation_results): cloth, tube, or a batch of scenes.
  newton    one Newton iteration in contact from a set state through the stage entry points: the unit
            that a frame repeats 3 to 100 times.

Sizes are those of the repository's workloads (33 x 33 cloth, 297 x 297 tube around a cylinder,
cloth-on-sphere scenes with n in 17..161, 129 x 129 cloth with boxes, twisting sheets up to
513 x 513) and the odd sizes between them.
"""
import ctypes
import math
import weakref

import numpy as np
import torch

import luisacomputesimulator_amd as lcsx
from luisacomputesimulator_amd import NewtonSolver, scenes

DEV = "cuda"


# ------------------------------------------------------------------ cases
def listed():
    return [
        # the product of a caller's solver on the largest sheet (513 x 513): streaming the matrix
        {"name": "spmv_513", "kind": "spmv", "n": 513},
        # the smallest solve (33 x 33 cloth, relative test on every iteration): latency and launches
        {"name": "pcg_33", "kind": "pcg", "n": 33, "check": 1, "rel": 1e-4},
        # a solve of the tube's size that runs to the cap of 100 iterations, tested every 25
        {"name": "pcg_297", "kind": "pcg", "n": 297, "check": 25, "rel": 0.0},
        # vertices against faces of the tube closing in on its cylinder
        {"name": "sweep_vf_tube_297", "kind": "sweep", "mesh": "tube", "n": 297, "edges": False},
        # edges against edges of a small cloth moving onto a sphere
        {"name": "sweep_ee_sphere_65", "kind": "sweep", "mesh": "sphere", "n": 65, "edges": True},
        # the smallest frame: a 33 x 33 cloth in free fall
        {"name": "frame_cloth_33", "kind": "frame", "scene": "cloth", "n": 33, "precision": "fp32"},
        # an ordinary frame in contact: a cloth arriving on a sphere, 16-bit blocks (FP16), FP64 collision
        {"name": "frame_sphere_97_fp16", "kind": "frame", "scene": "sphere", "n": 97, "precision": "mixed"},
        # the benchmark's frame: the 297 x 297 tube spinning with its ends
        {"name": "frame_tube_297", "kind": "frame", "scene": "tube", "n": 297, "precision": "fp32"},
        # a batch of scenes of mixed sizes arriving on their spheres, stepped together
        {"name": "frame_batch_24", "kind": "frame", "scene": "batch", "n": 161, "count": 24, "precision": "fp32"},
        # the benchmark's contact frames: the whole tube within the contact band of its cylinder
        {"name": "newton_tube_297", "kind": "newton", "scene": "tube", "n": 297, "precision": "fp32"},
        # cloth and affine bodies: 24 boxes with a corner each in contact with a 129 x 129 cloth
        {"name": "newton_boxes_129", "kind": "newton", "scene": "boxes", "n": 129, "count": 24, "precision": "fp32"},
        # a large sheet twisted at its edges, 16-bit blocks (BF16), FP64 collision
        {"name": "newton_sheet_385_bf16", "kind": "newton", "scene": "sheet", "n": 385, "precision": "mixed_bf16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["spmv", "pcg", "sweep", "frame", "frame", "newton", "newton"])
    if kind == "spmv":
        return {"kind": kind, "n": _log_int(rng, 17, 513)}
    if kind == "pcg":
        if rng.random() < 0.5:
            return {"kind": kind, "n": _log_int(rng, 17, 129), "check": 1, "rel": 1e-4}
        return {"kind": kind, "n": _log_int(rng, 150, 400), "check": 25, "rel": 0.0}
    if kind == "sweep":
        mesh = rng.choice(["tube", "sphere"])
        n = _log_int(rng, 64, 297) if mesh == "tube" else _log_int(rng, 17, 161)
        return {"kind": kind, "mesh": mesh, "n": n, "edges": rng.random() < 0.5}
    precision = rng.choice(["fp32", "fp32", "fp32", "mixed", "mixed_bf16"])
    if kind == "frame":
        scene = rng.choice(["cloth", "sphere", "tube", "batch"])
        if scene == "tube":
            return {"kind": kind, "scene": scene, "n": _log_int(rng, 64, 297), "precision": "fp32"}
        if scene != "cloth" and precision == "mixed_bf16":
            precision = "mixed"  # BF16 blocks leave a whole frame in contact open to a few percent
        if scene == "batch":
            return {"kind": kind, "scene": scene, "n": _log_int(rng, 33, 161), "count": _log_int(rng, 4, 24),
                    "precision": precision}
        return {"kind": kind, "scene": scene, "n": _log_int(rng, 17, 161), "precision": precision}
    scene = rng.choice(["tube", "boxes", "sheet"])
    if scene == "tube":
        return {"kind": kind, "scene": scene, "n": _log_int(rng, 64, 297), "precision": precision}
    if scene == "boxes":
        return {"kind": kind, "scene": scene, "n": _log_int(rng, 33, 161), "count": rng.randint(4, 25),
                "precision": precision}
    return {"kind": kind, "scene": scene, "n": _log_int(rng, 33, 385), "precision": precision}


# ------------------------------------------------------------------ block systems
def _grid_links(n):
    """Neighbour pairs (i < j) of a cloth's Hessian on an n x n grid: the edges with both diagonals and
    the vertices two apart (hinges), up to 12 blocks in a row."""
    ids = np.arange(n * n, dtype=np.int64).reshape(n, n)
    out = []
    for dr, dc in ((0, 1), (1, 0), (1, 1), (1, -1), (0, 2), (2, 0)):
        a = ids[:n - dr, max(0, -dc):n - max(0, dc)]
        b = ids[dr:, max(0, dc):n + min(0, dc)]
        out.append(np.stack([a.reshape(-1), b.reshape(-1)], 1))
    return np.concatenate(out)


def _system(n, seed):
    """Block-CSR system of a rippled n x n cloth of 1 x 1 m (membrane stiffness 10 N/m, 0.2 kg/m^2,
    dt 1/60 s): stiff along each link, 3% across it, with the lumped mass over dt^2 on the diagonal.
    FP32 arrays on the GPU: row_ptr, col (int32), blocks (nnz, 9), diag (n, 9), b (n, 3)."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    links = torch.from_numpy(_grid_links(n)).to(DEV)
    nv = n * n
    h = 1.0 / (n - 1)
    r, c = torch.meshgrid(torch.arange(n, device=DEV), torch.arange(n, device=DEV), indexing="ij")
    x = torch.stack([c * h, torch.zeros_like(c) * h, r * h], -1).reshape(nv, 3).double()
    x = x + 0.2 * h * torch.randn(nv, 3, generator=g, device=DEV, dtype=torch.float64)
    d = x[links[:, 1]] - x[links[:, 0]]
    d = d / d.norm(dim=1, keepdim=True)
    k = 10.0 * (0.5 + torch.rand(len(links), 1, 1, generator=g, device=DEV, dtype=torch.float64))
    blk = (k * (d[:, :, None] * d[:, None, :] + 0.03 * torch.eye(3, device=DEV, dtype=torch.float64))).float()
    mass = 0.2 * h * h * 3600.0
    diag = torch.zeros(nv, 3, 3, device=DEV, dtype=torch.float64)
    diag += mass * torch.eye(3, device=DEV, dtype=torch.float64)
    order = torch.cat([links[:, 0] * nv + links[:, 1], links[:, 1] * nv + links[:, 0]])
    both = torch.cat([links[:, 0], links[:, 1]])
    order, at = order.sort()  # by row, then column: the block-CSR order, and a fixed order of the sums
    row, col = both[at], order % nv
    blocks = -torch.cat([blk, blk])[at]
    ptr = torch.zeros(nv + 1, device=DEV, dtype=torch.int64)
    ptr[1:] = torch.bincount(row, minlength=nv).cumsum(0)
    run = torch.zeros(len(row) + 1, 9, device=DEV, dtype=torch.float64)
    run[1:] = blocks.double().reshape(-1, 9).cumsum(0)
    diag = (diag.reshape(nv, 9) - (run[ptr[1:]] - run[ptr[:-1]])).float()
    # a load with a smooth part (gravity, wind) and a rough one (elastic forces of one vertex)
    b = mass * torch.tensor([0.0, -9.8 / 3600.0, 0.0], device=DEV, dtype=torch.float64)
    b = b + mass * 1e-3 * torch.randn(nv, 3, generator=g, device=DEV, dtype=torch.float64)
    return {"ptr": ptr.int(), "col": col.int().contiguous(), "blocks": blocks.reshape(-1, 9).contiguous(),
            "diag": diag.contiguous(), "b": b.float().contiguous()}


def _bsr(m):
    return lcsx.lcsx_bsr(len(m["ptr"]) - 1, len(m["col"]), m["ptr"].data_ptr(), m["col"].data_ptr(),
                         m["blocks"].data_ptr(), m["diag"].data_ptr())


def _ok(code):
    if code != 0:
        raise lcsx.LcsxError(lcsx.load_library().lcsx_last_error().decode(errors="replace"))


def _mul64(m, x):
    """A x in 64 bits: the row sums as differences of one running sum would cancel, so by index_add."""
    row = torch.repeat_interleave(torch.arange(len(m["ptr"]) - 1, device=DEV), (m["ptr"][1:] - m["ptr"][:-1]).long())
    y = (m["diag"].double().reshape(-1, 3, 3) @ x[:, :, None])[:, :, 0]
    return y.index_add(0, row, (m["blocks"].double().reshape(-1, 3, 3) @ x[m["col"].long()][:, :, None])[:, :, 0])


def _pcg64(m, iters):
    """x of the block-Jacobi PCG after `iters` iterations from x = 0, in 64 bits; iters None: to 1e-13."""
    inv = torch.linalg.inv(m["diag"].double().reshape(-1, 3, 3))
    x = torch.zeros_like(m["b"], dtype=torch.float64)
    r = m["b"].double()
    p, rz_old, rz0 = torch.zeros_like(x), None, None
    for k in range(iters if iters is not None else 3000):
        z = (inv @ r[:, :, None])[:, :, 0]
        rz = (r * z).sum()
        rz0 = rz if rz0 is None else rz0
        if iters is None and k % 20 == 0 and float(rz) <= 1e-26 * float(rz0):
            break
        p = z + (0.0 if rz_old is None else rz / rz_old) * p
        q = _mul64(m, p)
        alpha = rz / (p * q).sum()
        x, r, rz_old = x + alpha * p, r - alpha * q, rz
    return x


# ------------------------------------------------------------------ meshes and states
def _ripple(x, rng, amplitude, wave):
    """A smooth vector field over points x: three random plane waves of about the given wavelength."""
    out = np.zeros_like(x)
    for _ in range(3):
        k = rng.normal(size=3) * 2.0 * np.pi / wave
        out += np.sin(x @ k + rng.uniform(0, 2 * np.pi))[:, None] * rng.normal(size=3)
    return amplitude * out / 3.0


def _tube_scene(n, gap, gravity=(0.0, 0.0, 0.0)):
    """The tube of n rings of n vertices around its cylinder, `gap` metres apart."""
    return scenes.cylinder_tube(rings=n, per_ring=n, radius=0.11, cyl_radius=0.11 - gap, gravity=gravity)


def _sphere_scene(n, ox, oz, seed):
    """A cloth 1.5 mm above the top of its sphere: within the contact band from the first iteration."""
    return scenes.cloth_on_sphere(n, ox, oz, seed=seed, height=0.3015)


def _spin_targets(solver, scene, x, angle_of_mesh):
    """Pinned targets of each mesh: its pinned vertices at x turned about the x axis by angle_of_mesh."""
    fixed = solver.read("fixed_verts").astype(np.int64)
    at = 0
    for mid, mesh in enumerate(scene.meshes):
        ids = fixed[(fixed >= at) & (fixed < at + len(mesh.verts))]
        at += len(mesh.verts)
        if len(ids):
            p = x[ids].astype(np.float64)
            a = angle_of_mesh(mid, p) if callable(angle_of_mesh) else angle_of_mesh
            c, s = np.cos(a), np.sin(a)
            solver.set_pinned_targets(mid, np.stack([p[:, 0], c * p[:, 1] - s * p[:, 2], s * p[:, 1] + c * p[:, 2]], -1))


def _boxes_scene(n, count, seed):
    """`count` affine boxes on an n x n cloth, one corner of each 1.2 mm above it (inside the contact
    band), in the cells of a 5 x 5 grid, with random orientations."""
    rng = np.random.default_rng(seed)
    sc = scenes.cloth_rigid_coupling(n, boxes=0, seed=seed)
    cloth = sc.meshes[0]
    mat = scenes.Material(thickness=cloth.material.thickness, density=500.0, d_hat=cloth.material.d_hat,
                          body="rigid_solid", rigid_stiffness=1e8)
    cells = rng.permutation(25)[:count]
    top = float(cloth.verts[:, 1].max())
    for k, cell in enumerate(cells):
        center = np.array([-0.36 + 0.18 * (cell % 5), 0.0, -0.36 + 0.18 * (cell // 5)])
        v, t = scenes.box_mesh(center, 0.1, scenes.rotation_matrix(rng.uniform(0.0, 2.0 * np.pi, size=3)))
        v = v + np.array([0.0, top + 1.2e-3 - v[:, 1].min(), 0.0], dtype=np.float32)
        sc.meshes.append(scenes.Mesh(f"box{k}", v.astype(np.float32), t, mat, []))
    return sc


def _solver_state(case, seed):
    """A solver and the state (positions, velocities) it is set to before each pass."""
    rng = np.random.default_rng(seed)
    scene, n = case["scene"], case["n"]
    if scene == "batch":
        # the sizes belong to the case: every seed's batch has the same rows
        ns = np.random.default_rng(case["count"]).integers(max(17, n // 4), n + 1, size=case["count"])
        ns[0] = n
        off = rng.uniform(-0.1, 0.1, size=(case["count"], 2))
        scs = [_sphere_scene(int(ns[k]), *off[k], seed=seed + k) for k in range(case["count"])]
    elif scene == "sphere":
        scs = [_sphere_scene(n, *rng.uniform(-0.1, 0.1, size=2), seed=seed)]
    elif scene == "cloth":
        scs = [scenes.square_cloth(n, seed=seed)]
    elif scene == "tube":
        # frame: 10 mm apart (the benchmark's start); newton: the tube in the contact band all around
        scs = [_tube_scene(n, 0.01 if case["kind"] == "frame" else 1.6e-3)]
    elif scene == "boxes":
        scs = [_boxes_scene(n, case["count"], seed)]
    else:
        scs = [scenes.twisting_sheet(n)]
    for sc in scs:
        sc.params.precision = case["precision"]
        if scene in ("batch", "sphere"):
            # a fixed three Newton iterations, as an interactive program runs: where the loop ends by its
            # tolerance, a rounding can add an iteration, and the frame then differs by that step
            sc.params.newton_tol = 1e-5
    solver = NewtonSolver.from_scenes(scs) if len(scs) > 1 else NewtonSolver.from_scene(scs[0])
    x = solver.get_simulation_results().astype(np.float64)
    v = solver.get_velocities().astype(np.float64)
    free = np.ones(len(x), dtype=bool)
    free[solver.read("fixed_verts").astype(np.int64)] = False
    dt = scs[0].params.implicit_dt
    if scene == "tube":
        w = 2.0 * np.pi
        v[free] += _ripple(x, rng, 0.05, 0.3)[free]
        if case["kind"] == "newton":
            x[free] += _ripple(x, rng, 1e-4, 0.1)[free]
        _spin_targets(solver, scs[0], x, w * dt)
    elif scene == "sheet":
        # the edges turn against each other by one frame's 3 degrees; the sheet follows in between
        v[:, 1] -= 2.0 * np.pi * x[:, 0] * x[:, 2]
        v[:, 2] += 2.0 * np.pi * x[:, 0] * x[:, 1]
        v[free] += _ripple(x, rng, 0.05, 0.3)[free]
        _spin_targets(solver, scs[0], x, lambda mid, p: np.where(p[:, 0] < 0.0, np.pi, -np.pi) * dt)
    elif scene == "boxes":
        bodies = np.arange(solver.num_verts - 4 * case["count"], solver.num_verts)
        v[bodies[::4], 1] -= 0.2 + 0.1 * rng.random(case["count"])  # translation rows
        cloth = free.copy()
        cloth[n * n:] = False
        v[cloth] += _ripple(x, rng, 0.02, 0.3)[cloth]
    elif scene == "cloth":
        v[free] += _ripple(x, rng, 0.3, 0.5)[free]
    else:
        for k in range(len(scs)):  # cloths coming down on their spheres
            a, m = solver.scene_range(k) if len(scs) > 1 else (0, len(x))
            mine = np.zeros(len(x), dtype=bool)
            mine[a:a + m] = free[a:a + m]
            v[mine] += np.array([0.0, -0.2, 0.0]) + _ripple(x, rng, 0.05, 0.5)[mine]
    return {"solver": solver, "x": x.astype(np.float32), "v": v.astype(np.float32), "bodies": scene == "boxes"}


def _sweep_state(case, seed):
    """Device arrays of a mesh pair moving together: primitives, start and end positions, per-vertex
    offset and query padding, query boxes, the tree and the output list."""
    rng = np.random.default_rng(seed)
    if case["mesh"] == "tube":
        sc = _tube_scene(case["n"], 1.6e-3)
    else:
        sc = _sphere_scene(case["n"], *rng.uniform(-0.1, 0.1, size=2), seed=seed)
    x0 = np.concatenate([m.verts for m in sc.meshes]).astype(np.float64)
    at = np.cumsum([0] + [len(m.verts) for m in sc.meshes])
    tris = np.concatenate([m.tris.astype(np.int64) + o for m, o in zip(sc.meshes, at)])
    move = _ripple(x0, rng, 1.5e-3, 0.2)
    move[at[1]:] = 0.0  # the cylinder or sphere stands still
    x1 = x0 + move
    dev = lambda a, t: torch.from_numpy(np.ascontiguousarray(a)).to(DEV).to(t)  # noqa: E731
    s = {"x0": dev(x0, torch.float32).contiguous(), "x1": dev(x1, torch.float32).contiguous(), "nv": len(x0),
         "edges": bool(case["edges"])}
    if case["edges"]:
        e = np.sort(np.concatenate([tris[:, [0, 1]], tris[:, [1, 2]], tris[:, [2, 0]]]), 1)
        prims = np.unique(e, axis=0)
    else:
        prims = tris
    s["prims"] = dev(prims.astype(np.int32), torch.int32).contiguous()
    offset, d_hat = 0.5e-3, 1e-3
    s["offset"] = torch.full((len(x0),), offset, device=DEV)
    pts = torch.stack([s["x0"], s["x1"]], 0)  # (2, nv, 3)
    if case["edges"]:
        pts = pts[:, s["prims"].long()].transpose(0, 1).reshape(len(prims), 4, 3).transpose(0, 1)
    s["boxes"] = torch.cat([pts.amin(0) - (offset + d_hat), pts.amax(0) + (offset + d_hat)], 1).contiguous()
    cap = 40 * len(s["boxes"])
    s["pairs"] = torch.empty(cap, 2, device=DEV, dtype=torch.int32)
    s["sorted"] = torch.empty(cap, device=DEV, dtype=torch.int64)  # (leaf, query) keys, -1 past the last
    s["count"] = torch.zeros(1, device=DEV, dtype=torch.int32)
    s["toi"] = torch.zeros(1, device=DEV)
    lib = lcsx.load_library()
    h = ctypes.c_void_p()
    torch.cuda.synchronize()
    _ok(lib.lcsx_lbvh_create(2 if case["edges"] else 3, s["prims"].data_ptr(), len(prims), ctypes.byref(h)))
    s["tree"] = h
    holder = torch.nn.Module()  # gives the tree back with the state
    weakref.finalize(holder, lib.lcsx_lbvh_destroy, h)
    s["holder"] = holder
    return s


# ------------------------------------------------------------------ the cases' parts
def prepare(case, seed):
    kind = case["kind"]
    if kind in ("spmv", "pcg"):
        m = _system(case["n"], seed)
        m["bsr"], m["kind"] = _bsr(m), kind
        m["out"] = torch.empty_like(m["b"])
        if kind == "pcg":
            # tested by the relative test alone or not at all, so the solve does the same work anywhere
            m["opt"] = lcsx.lcsx_pcg_options(100, case["check"], case["rel"], 0.0)
        torch.cuda.synchronize()
        return m
    if kind == "sweep":
        return dict(_sweep_state(case, seed), kind=kind)
    return dict(_solver_state(case, seed), kind=kind)


def run(state):
    kind = state["kind"]
    lib = lcsx.load_library()
    if kind == "spmv":
        _ok(lib.lcsx_spmv_bsr(ctypes.byref(state["bsr"]), state["b"].data_ptr(), state["out"].data_ptr(), None))
        return state["out"]
    if kind == "pcg":
        res = lcsx.lcsx_pcg_result()
        _ok(lib.lcsx_pcg_solve_bsr(ctypes.byref(state["bsr"]), state["b"].data_ptr(), state["out"].data_ptr(),
                                   ctypes.byref(state["opt"]), None, ctypes.byref(res)))
        return state["out"]
    if kind == "sweep":
        s = state
        s["count"].zero_()
        _ok(lib.lcsx_lbvh_construct(s["tree"], s["x0"].data_ptr(), s["nv"], None))
        _ok(lib.lcsx_lbvh_refit(s["tree"], s["x0"].data_ptr(), s["x1"].data_ptr(), s["offset"].data_ptr(), None))
        _ok(lib.lcsx_lbvh_query(s["tree"], s["boxes"].data_ptr(), len(s["boxes"]), int(s["edges"]),
                                s["pairs"].data_ptr(), len(s["pairs"]), s["count"].data_ptr(), None))
        found = int(s["count"].item())
        if found > len(s["pairs"]):
            raise lcsx.LcsxError("the pair list is too small")
        _ok(lib.lcsx_ccd_pairs(int(s["edges"]), s["pairs"].data_ptr(), found, s["prims"].data_ptr(),
                               s["x0"].data_ptr(), s["x1"].data_ptr(), s["offset"].data_ptr(), 0,
                               s["toi"].data_ptr(), None))
        s["sorted"].fill_(-1)
        s["sorted"][:found] = s["pairs"][:found].view(torch.int64).reshape(-1).sort().values
        return {"pairs": s["sorted"], "toi": s["toi"]}
    solver = state["solver"]
    solver.set_state(state["x"], state["v"])
    if kind == "frame":
        solver.physics_step_gpu(1)
        return {"x": solver.get_simulation_results(), "v": solver.get_velocities()}
    for stage in ("frame_begin", "predict", "newton_iteration"):
        solver.stage(stage)
    if state["bodies"]:  # the bodies' soft rotations leave FP32's direction open to 1e-2 (its step is in x)
        return {"x": solver.get_simulation_results()}
    return {"x": solver.get_simulation_results(), "dx": solver.read("dx")}


def _scene_counts(case):
    """Rows, faces, edges and blocks (both triangles of the matrix) of a case's scenes, to a few percent."""
    n = case["n"]
    scene = case.get("scene", case.get("mesh"))
    if scene == "batch":
        cloth, other = case["count"] * (0.45 * n * n), case["count"] * 642
    else:
        cloth = n * n
        other = {"tube": 5760, "sphere": 642, "boxes": 12 * case.get("count", 0)}.get(scene, 0)
    return {"rows": cloth + other, "faces": 2 * (cloth + other), "edges": 3 * (cloth + other), "blocks": 12 * cloth}


def work(case):
    """Bytes: each input read once and each output written once; operations: the products of the solves."""
    kind, n = case["kind"], case["n"]
    if kind in ("spmv", "pcg"):
        nv, nnz = n * n, 2 * len(_grid_links(n))
        matrix = 40 * nnz + 36 * nv + 4 * (nv + 1)
        iters = 1 if kind == "spmv" else (100 if case["rel"] == 0.0 else 40)
        return {"bytes": matrix + 24 * nv, "flops": iters * 18 * (nnz + (nv if kind == "spmv" else 2 * nv))}
    c = _scene_counts(case)
    if kind == "sweep":
        prims = c["edges"] * 8 if case["edges"] else c["faces"] * 12
        queries = c["edges"] if case["edges"] else c["rows"]
        pairs = 14 * queries  # found per query, about
        return {"bytes": prims + 24 * c["rows"] + 4 * c["rows"] + 24 * queries + 8 * pairs, "flops": 100.0 * pairs}
    # state in and out, element constants (index, rest shape) and per Newton iteration the system once
    newton = 1 if kind == "newton" else 3
    pcg = 100 if case["scene"] in ("tube", "sheet") else 40
    system = 36 * (c["blocks"] + c["rows"])
    return {"bytes": 48 * c["rows"] + 44 * c["faces"] + 28 * c["edges"] + newton * system,
            "flops": newton * (pcg * 18 * (c["blocks"] + 2 * c["rows"]) + 2000 * c["faces"])}


def tolerance(case):
    """About four times what a build with every sum in another order (wavefront butterflies, block sums,
    the lanes of a row) differs by over a hundred drawn cases, the largest of them."""
    kind = case["kind"]
    if kind == "spmv":  # 13 blocks of 3 terms in FP32: 7e-8 off the 64-bit product
        return {"rel": 4e-7, "max": 4e-6}
    if kind == "pcg":
        # a relative test can end one iteration earlier or later, 1e-4 of the solution; at the cap the
        # FP32 iterates are up to 1e-5 off the 64-bit ones
        return {"rel": 5e-4, "max": 2e-2} if case["rel"] > 0.0 else {"rel": 4e-5, "max": 4e-3}
    if kind == "sweep":  # the pairs exactly; the step bound's last bits
        return {"rel": 1e-6, "max": 1e-6}
    precision = case["precision"]
    if kind == "frame":
        # seen: free fall and the spinning tube 6e-5, contact 4e-4 (max 6e-2, a vertex leaving its contact)
        return {"rel": 2e-4, "max": 4e-3} if case["scene"] in ("cloth", "tube") else {"rel": 2e-3, "max": 0.25}
    if case["scene"] == "sheet":  # seen: FP32 3e-7, FP16 2e-5, BF16 5e-4
        return {"fp32": {"rel": 2e-6, "max": 2e-5}, "mixed": {"rel": 8e-5, "max": 8e-4},
                "mixed_bf16": {"rel": 2e-3, "max": 2e-2}}[precision]
    # seen: tube 5e-5 (max 3e-3), boxes 5e-5 (max 1e-3)
    return {"rel": 2e-4, "max": 1.2e-2 if case["scene"] == "tube" else 4e-3}


def exact(case, seed):
    """spmv and pcg in 64 bits. A solve that stops by its relative test is compared with the solution
    itself (it stops 1e-4 away), one that runs to the cap with the 64-bit iterate after as many
    iterations. The sweeps give whole numbers and ACCD's bound, which is where its loop stops and has
    no other value in 64 bits; a frame or a Newton iteration in plain numpy (contact search, assembly
    and solve of up to 148,225 rows) is far beyond 20 seconds."""
    if case["kind"] == "spmv":
        m = _system(case["n"], seed)
        return _mul64(m, m["b"].double())
    if case["kind"] == "pcg":
        m = _system(case["n"], seed)
        return _pcg64(m, None if case["rel"] > 0.0 else 100)
    return None
