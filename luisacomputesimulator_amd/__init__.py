"""MI355X-native Newton step for IPC cloth simulation (LuisaComputeSimulator's hot path).

Python front end over the C ABI in ``include/lcsx.h`` (``liblcsx.so``, HIP for gfx950). The
class surface follows the reference's pybind module ``lcs_solver_py``
(``PythonBindings/python_bindings.cpp:303-359``): ``NewtonSolver.register_mesh``,
``init_solver``, ``physics_step_gpu`` and ``get_simulation_results``, plus the per-stage entry
points of the reference's NewtonSolver / LBVH / NarrowPhasesDetector / ConjugateGradientSolver
classes for parity checks and measurement.

There is no CPU fallback: if ``liblcsx.so`` is missing or no GPU is present, calls raise.
"""
from __future__ import annotations

import ctypes as C
import os
from typing import Dict, List, Optional

import numpy as np

from . import scenes  # noqa: F401
from .scenes import BODY_TYPES, FIXED_METHODS, STRETCH_MODELS, Anim, Material, Params, Scene

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "liblcsx.so")
_LIB: Optional[C.CDLL] = None


class LcsxError(RuntimeError):
    pass


class lcsx_material(C.Structure):
    _fields_ = [("thickness", C.c_float), ("youngs_modulus", C.c_float), ("poisson_ratio", C.c_float),
                ("area_bending_stiffness", C.c_float), ("density", C.c_float), ("mass", C.c_float),
                ("d_hat", C.c_float), ("body", C.c_int), ("rigid_stiffness", C.c_float),
                ("stretch_spring", C.c_int)]


class lcsx_fixed_anim(C.Structure):
    _fields_ = [("use_translate", C.c_int), ("translate", C.c_float * 3), ("use_scale", C.c_int),
                ("scale", C.c_float * 3), ("use_rotate", C.c_int), ("rot_center", C.c_float * 3),
                ("rot_axis", C.c_float * 3), ("rot_deg_per_s", C.c_float)]


class lcsx_params(C.Structure):
    _fields_ = [("implicit_dt", C.c_float), ("nonlinear_iter_count", C.c_int), ("newton_max_iters", C.c_int),
                ("pcg_iter_count", C.c_int), ("pcg_check_every", C.c_int), ("pcg_rel_tol", C.c_float),
                ("pcg_abs_tol", C.c_float), ("gravity", C.c_float * 3), ("use_floor", C.c_int),
                ("use_self_collision", C.c_int), ("use_ccd_linesearch", C.c_int), ("floor_y", C.c_float),
                ("stiffness_collision", C.c_float), ("stiffness_dirichlet", C.c_float), ("damping_cloth", C.c_float),
                ("bending_scaling", C.c_float), ("newton_tol", C.c_float), ("precision", C.c_int),
                ("use_energy_linesearch", C.c_int),
                ("contact_energy_type", C.c_int), ("post_dist_check", C.c_int)]


class lcsx_stats(C.Structure):
    _fields_ = [("frame", C.c_int), ("newton_iters", C.c_int), ("pcg_iters", C.c_int), ("pcg_iters_total", C.c_int),
                ("toi", C.c_float), ("max_dx", C.c_float), ("pin_delta", C.c_float), ("pcg_rel", C.c_float),
                ("num_pairs_vf", C.c_int), ("num_pairs_ee", C.c_int), ("num_contacts", C.c_int),
                ("converged", C.c_int), ("broadphase_overflow", C.c_int), ("pcg_rz_true", C.c_double),
                ("min_gap", C.c_double), ("num_penetrating", C.c_int), ("gap_pairs", C.c_int),
                ("toi_min", C.c_float), ("num_ccd_pairs", C.c_int)]


class lcsx_bsr(C.Structure):
    _fields_ = [("n_rows", C.c_int), ("nnz", C.c_int), ("row_ptr", C.c_void_p), ("col", C.c_void_p),
                ("blocks", C.c_void_p), ("diag", C.c_void_p)]


class lcsx_pcg_options(C.Structure):
    _fields_ = [("max_iters", C.c_int), ("check_every", C.c_int), ("rel_tol", C.c_float), ("abs_tol", C.c_float)]


class lcsx_pcg_result(C.Structure):
    _fields_ = [("iters", C.c_int), ("converged", C.c_int), ("rz0", C.c_float), ("rz", C.c_float)]


# Every exported symbol of include/lcsx.h with its ctypes signature.
_SIGS = {
    "lcsx_last_error": (C.c_char_p, []),
    "lcsx_version": (C.c_char_p, []),
    "lcsx_device_count": (C.c_int, []),
    "lcsx_params_default": (None, [C.POINTER(lcsx_params)]),
    "lcsx_material_default": (None, [C.POINTER(lcsx_material)]),
    "lcsx_solver_create": (C.c_int, [C.POINTER(lcsx_params), C.c_int, C.POINTER(C.c_void_p)]),
    "lcsx_solver_destroy": (C.c_int, [C.c_void_p]),
    "lcsx_solver_add_mesh": (C.c_int, [C.c_void_p, C.POINTER(C.c_float), C.c_int, C.POINTER(C.c_int32), C.c_int,
                                       C.POINTER(lcsx_material), C.POINTER(C.c_int)]),
    "lcsx_solver_add_fixed_points": (C.c_int, [C.c_void_p, C.c_int, C.c_int, C.c_float, C.POINTER(lcsx_fixed_anim),
                                               C.POINTER(C.c_int)]),
    "lcsx_solver_load_scene_json": (C.c_int, [C.c_void_p, C.c_char_p, C.c_char_p]),
    "lcsx_solver_init": (C.c_int, [C.c_void_p]),
    "lcsx_solver_step": (C.c_int, [C.c_void_p, C.c_int]),
    "lcsx_solver_get_positions": (C.c_int, [C.c_void_p, C.POINTER(C.c_float), C.c_size_t]),
    "lcsx_solver_get_velocities": (C.c_int, [C.c_void_p, C.POINTER(C.c_float), C.c_size_t]),
    "lcsx_solver_set_state": (C.c_int, [C.c_void_p, C.POINTER(C.c_float), C.POINTER(C.c_float), C.c_size_t]),
    "lcsx_solver_set_pinned_targets": (C.c_int, [C.c_void_p, C.c_int, C.POINTER(C.c_float), C.c_int]),
    "lcsx_solver_get_stats": (C.c_int, [C.c_void_p, C.POINTER(lcsx_stats)]),
    "lcsx_solver_num_verts": (C.c_int, [C.c_void_p]),
    "lcsx_solver_begin_scene": (C.c_int, [C.c_void_p, C.POINTER(C.c_int)]),
    "lcsx_solver_num_scenes": (C.c_int, [C.c_void_p]),
    "lcsx_solver_scene_range": (C.c_int, [C.c_void_p, C.c_int, C.POINTER(C.c_int), C.POINTER(C.c_int)]),
    "lcsx_solver_get_scene_stats": (C.c_int, [C.c_void_p, C.c_int, C.POINTER(lcsx_stats)]),
    "lcsx_solver_run_stage": (C.c_int, [C.c_void_p, C.c_char_p]),
    "lcsx_solver_read": (C.c_int, [C.c_void_p, C.c_char_p, C.c_void_p, C.c_size_t, C.POINTER(C.c_size_t)]),
    "lcsx_solver_write": (C.c_int, [C.c_void_p, C.c_char_p, C.c_void_p, C.c_size_t]),
    "lcsx_solver_kernel_times": (C.c_int, [C.c_void_p, C.c_char_p, C.c_size_t, C.c_int]),
    "lcsx_solver_set_timing": (C.c_int, [C.c_void_p, C.c_int]),
    "lcsx_solver_set_graphs": (C.c_int, [C.c_void_p, C.c_int]),
    "lcsx_solver_set_one_launch": (C.c_int, [C.c_void_p, C.c_int]),
    "lcsx_solver_set_query_shape": (C.c_int, [C.c_void_p, C.c_int]),
    "lcsx_solver_set_spmv_shape": (C.c_int, [C.c_void_p, C.c_int]),
    "lcsx_solver_save_state": (C.c_int, [C.c_void_p, C.c_char_p]),
    "lcsx_solver_load_state": (C.c_int, [C.c_void_p, C.c_char_p, C.c_int]),
    "lcsx_solver_save_obj": (C.c_int, [C.c_void_p, C.c_char_p]),
    "lcsx_solver_autotune": (C.c_int, [C.c_void_p, C.c_char_p, C.c_size_t]),
    "lcsx_lbvh_create": (C.c_int, [C.c_int, C.c_void_p, C.c_int, C.POINTER(C.c_void_p)]),
    "lcsx_lbvh_destroy": (C.c_int, [C.c_void_p]),
    "lcsx_lbvh_set_query_shape": (C.c_int, [C.c_void_p, C.c_int]),
    "lcsx_lbvh_construct": (C.c_int, [C.c_void_p, C.c_void_p, C.c_int, C.c_void_p]),
    "lcsx_lbvh_refit": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p]),
    "lcsx_lbvh_query": (C.c_int, [C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_void_p, C.c_uint32, C.c_void_p,
                                  C.c_void_p]),
    "lcsx_lbvh_read": (C.c_int, [C.c_void_p, C.c_char_p, C.c_void_p, C.c_size_t]),
    "lcsx_pcg_options_default": (None, [C.POINTER(lcsx_pcg_options)]),
    "lcsx_pcg_solve_bsr": (C.c_int, [C.POINTER(lcsx_bsr), C.c_void_p, C.c_void_p, C.POINTER(lcsx_pcg_options),
                                     C.c_void_p, C.POINTER(lcsx_pcg_result)]),
    "lcsx_pcg_solve_bsr_noalloc": (C.c_int, [C.POINTER(lcsx_bsr), C.c_void_p, C.c_void_p,
                                             C.POINTER(lcsx_pcg_options), C.c_void_p, C.POINTER(lcsx_pcg_result)]),
    "lcsx_pcg_form_counts": (C.c_int, [C.c_int, C.POINTER(C.c_uint64)]),
    "lcsx_spmv_bsr": (C.c_int, [C.POINTER(lcsx_bsr), C.c_void_p, C.c_void_p, C.c_void_p]),
    "lcsx_pcg_solve_op": (C.c_int, [C.c_int, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p,
                                    C.POINTER(lcsx_pcg_options), C.c_void_p, C.POINTER(lcsx_pcg_result)]),
    "lcsx_ccd_pairs": (C.c_int, [C.c_int, C.c_void_p, C.c_uint32, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p,
                                 C.c_int, C.c_void_p, C.c_void_p]),
    "lcsx_dcd_pairs": (C.c_int, [C.c_int, C.c_void_p, C.c_uint32, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p,
                                 C.c_void_p, C.c_void_p, C.c_float, C.c_int, C.c_int, C.c_void_p, C.c_void_p,
                                 C.c_void_p, C.c_void_p, C.c_uint32, C.c_void_p, C.c_void_p]),
}

# lcsx_spmv_fn: the product callback of lcsx_pcg_solve_op (user, device p, device q, stream)
SPMV_FN = C.CFUNCTYPE(None, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p)


def load_library(path: str = LIB_PATH) -> C.CDLL:
    """Loads liblcsx.so (raises if it has not been built)."""
    global _LIB
    if _LIB is not None:
        return _LIB
    if not os.path.exists(path):
        raise LcsxError(f"{path} is missing: build it with `python -m luisacomputesimulator_amd.build`")
    lib = C.CDLL(path)
    for name, (res, args) in _SIGS.items():
        fn = getattr(lib, name)
        fn.restype = res
        fn.argtypes = args
    _LIB = lib
    return lib


def _check(code: int) -> None:
    if code != 0:
        msg = load_library().lcsx_last_error().decode(errors="replace")
        raise LcsxError(f"lcsx error {code}: {msg}")


def params_to_c(p: Params) -> lcsx_params:
    c = lcsx_params()
    c.implicit_dt = p.implicit_dt
    c.nonlinear_iter_count = p.nonlinear_iter_count
    c.newton_max_iters = p.newton_max_iters
    c.pcg_iter_count = p.pcg_iter_count
    c.pcg_check_every = p.pcg_check_every
    c.pcg_rel_tol = p.pcg_rel_tol
    c.pcg_abs_tol = p.pcg_abs_tol
    c.gravity[:] = list(p.gravity)
    c.use_floor = int(p.use_floor)
    c.use_self_collision = int(p.use_self_collision)
    c.use_ccd_linesearch = int(p.use_ccd_linesearch)
    c.floor_y = p.floor_y
    c.stiffness_collision = p.stiffness_collision
    c.stiffness_dirichlet = p.stiffness_dirichlet
    c.damping_cloth = p.damping_cloth
    c.bending_scaling = p.bending_scaling
    c.newton_tol = p.newton_tol
    c.precision = {"fp32": 0, "mixed": 1, "mixed_bf16": 2}[p.precision]
    c.use_energy_linesearch = int(p.use_energy_linesearch)
    c.contact_energy_type = int(p.contact_energy_type)
    c.post_dist_check = int(getattr(p, "post_dist_check", True))
    return c


def material_to_c(m: Material) -> lcsx_material:
    c = lcsx_material()
    c.thickness, c.youngs_modulus, c.poisson_ratio = m.thickness, m.youngs_modulus, m.poisson_ratio
    c.area_bending_stiffness, c.density, c.mass, c.d_hat = m.area_bending_stiffness, m.density, m.mass, m.d_hat
    c.body = BODY_TYPES[m.body]
    c.rigid_stiffness = m.rigid_stiffness
    c.stretch_spring = STRETCH_MODELS[m.stretch_model]
    return c


def anim_to_c(a: Anim) -> lcsx_fixed_anim:
    c = lcsx_fixed_anim()
    c.use_translate, c.use_scale, c.use_rotate = int(a.use_translate), int(a.use_scale), int(a.use_rotate)
    c.translate[:] = list(a.translate)
    c.scale[:] = list(a.scale)
    c.rot_center[:] = list(a.rot_center)
    c.rot_axis[:] = list(a.rot_axis)
    c.rot_deg_per_s = a.rot_deg_per_s
    return c


_NP = {"f": np.float32, "u": np.uint32, "q": np.uint64, "b": np.uint8, "d": np.float64}
# dtype of each readable buffer (see lcsx_solver_read)
_DTYPES: Dict[str, str] = {n: "u" for n in ("faces", "edges", "hinges", "csr", "stretch_faces", "bending_hinges",
                                            "stretch_springs",
                                             "fixed_verts", "cluster_use", "pairs_vf", "pairs_ee", "contact_idx", "contact_type",
                                             "ccd_rest_vf", "ccd_rest_ee", "contact_triplets")}
_DTYPES["is_fixed"] = "b"
_DTYPES["energy"] = "d"


def _dtype_of(name: str):
    if name.endswith(".morton_sorted"):
        return np.uint64
    if name.endswith((".sorted_to_orig", ".parent", ".children", ".object_idx")):
        return np.uint32
    return _NP[_DTYPES.get(name, "f")]


class NewtonSolver:
    """GPU Newton solver for a cloth scene (reference NewtonSolver + lcs_solver_py.NewtonSolver)."""

    def __init__(self, params: Optional[Params] = None, device: int = 0):
        self.lib = load_library()
        self.params = params or Params()
        h = C.c_void_p()
        p = params_to_c(self.params)
        _check(self.lib.lcsx_solver_create(C.byref(p), device, C.byref(h)))
        self.h = h
        self.mesh_names: List[str] = []
        self._inited = False

    @classmethod
    def from_scene(cls, scene: Scene, device: int = 0) -> "NewtonSolver":
        s = cls(scene.params, device)
        for m in scene.meshes:
            mid = s.register_mesh(m.name, m.verts, m.tris, m.material)
            for fp in m.fixed:
                s.add_fixed_points(mid, fp.method, fp.range, fp.anim)
        s.init_solver()
        if scene.initial_position is not None or scene.initial_velocity is not None:
            s.set_state(scene.initial_position, scene.initial_velocity)
        return s

    @classmethod
    def from_scenes(cls, scenes: List[Scene], device: int = 0) -> "NewtonSolver":
        """The batched form: every scene of the list in one solver (the first scene's params apply
        to all), stepped together with one launch per stage."""
        s = cls(scenes[0].params, device)
        for k, sc in enumerate(scenes):
            if k:
                s.begin_scene()
            for m in sc.meshes:
                mid = s.register_mesh(m.name, m.verts, m.tris, m.material)
                for fp in m.fixed:
                    s.add_fixed_points(mid, fp.method, fp.range, fp.anim)
        s.init_solver()
        if any(sc.initial_position is not None or sc.initial_velocity is not None for sc in scenes):
            x = np.concatenate([np.asarray(sc.initial_position if sc.initial_position is not None else
                                           np.concatenate([m.verts for m in sc.meshes]), np.float32).reshape(-1, 3)
                                for sc in scenes])
            v = np.concatenate([np.asarray(sc.initial_velocity if sc.initial_velocity is not None else
                                           np.zeros((sc.num_verts, 3)), np.float32).reshape(-1, 3) for sc in scenes])
            s.set_state(x, v)
        return s

    def begin_scene(self) -> int:
        sid = C.c_int()
        _check(self.lib.lcsx_solver_begin_scene(self.h, C.byref(sid)))
        return sid.value

    @property
    def num_scenes(self) -> int:
        return int(self.lib.lcsx_solver_num_scenes(self.h))

    def scene_range(self, scene: int) -> tuple:
        a, n = C.c_int(), C.c_int()
        _check(self.lib.lcsx_solver_scene_range(self.h, scene, C.byref(a), C.byref(n)))
        return a.value, n.value

    def scene_stats(self, scene: int) -> dict:
        s = lcsx_stats()
        _check(self.lib.lcsx_solver_get_scene_stats(self.h, scene, C.byref(s)))
        return {f: getattr(s, f) for f, _ in lcsx_stats._fields_}

    def __del__(self):
        try:
            if getattr(self, "h", None):
                self.lib.lcsx_solver_destroy(self.h)
                self.h = None
        except Exception:
            pass

    # -- lcs_solver_py surface ------------------------------------------------------------
    def register_mesh(self, name: str, vertices, triangles, material: Optional[Material] = None) -> int:
        v = np.ascontiguousarray(vertices, dtype=np.float32).reshape(-1, 3)
        t = np.ascontiguousarray(triangles, dtype=np.int32).reshape(-1, 3)
        mid = C.c_int()
        mat = material_to_c(material or Material())
        _check(self.lib.lcsx_solver_add_mesh(self.h, v.ctypes.data_as(C.POINTER(C.c_float)), len(v),
                                             t.ctypes.data_as(C.POINTER(C.c_int32)), len(t), C.byref(mat), C.byref(mid)))
        self.mesh_names.append(name)
        return mid.value

    def add_fixed_points(self, mesh_id: int, method: str, range_: float = 0.001, anim: Optional[Anim] = None) -> int:
        n = C.c_int()
        a = anim_to_c(anim or Anim())
        _check(self.lib.lcsx_solver_add_fixed_points(self.h, mesh_id, FIXED_METHODS[method], range_, C.byref(a),
                                                     C.byref(n)))
        return n.value

    def load_scene_json(self, path: str, mesh_dir: str = "") -> None:
        _check(self.lib.lcsx_solver_load_scene_json(self.h, path.encode(), mesh_dir.encode()))

    def num_meshes(self) -> int:
        return len(self.mesh_names)

    def get_mesh_names(self) -> List[str]:
        return list(self.mesh_names)

    def init_solver(self) -> None:
        _check(self.lib.lcsx_solver_init(self.h))
        self._inited = True

    def physics_step_gpu(self, frames: int = 1) -> None:
        _check(self.lib.lcsx_solver_step(self.h, frames))

    def get_simulation_results(self) -> np.ndarray:
        n = self.num_verts
        out = np.empty((n, 3), dtype=np.float32)
        _check(self.lib.lcsx_solver_get_positions(self.h, out.ctypes.data_as(C.POINTER(C.c_float)), out.size))
        return out

    def get_velocities(self) -> np.ndarray:
        out = np.empty((self.num_verts, 3), dtype=np.float32)
        _check(self.lib.lcsx_solver_get_velocities(self.h, out.ctypes.data_as(C.POINTER(C.c_float)), out.size))
        return out

    def set_state(self, x=None, v=None) -> None:
        n = 3 * self.num_verts
        xa = None if x is None else np.ascontiguousarray(x, dtype=np.float32).reshape(-1)
        va = None if v is None else np.ascontiguousarray(v, dtype=np.float32).reshape(-1)
        fp = C.POINTER(C.c_float)
        _check(self.lib.lcsx_solver_set_state(self.h, None if xa is None else xa.ctypes.data_as(fp),
                                              None if va is None else va.ctypes.data_as(fp), n))

    def set_pinned_targets(self, mesh_id: int, targets) -> None:
        t = np.ascontiguousarray(targets, dtype=np.float32).reshape(-1, 3)
        _check(self.lib.lcsx_solver_set_pinned_targets(self.h, mesh_id, t.ctypes.data_as(C.POINTER(C.c_float)), len(t)))

    @property
    def num_verts(self) -> int:
        return int(self.lib.lcsx_solver_num_verts(self.h))

    def stats(self) -> dict:
        s = lcsx_stats()
        _check(self.lib.lcsx_solver_get_stats(self.h, C.byref(s)))
        return {f: getattr(s, f) for f, _ in lcsx_stats._fields_}

    # -- per-stage entry points -----------------------------------------------------------
    def stage(self, name: str) -> None:
        _check(self.lib.lcsx_solver_run_stage(self.h, name.encode()))

    def read(self, name: str) -> np.ndarray:
        cnt = C.c_size_t()
        _check(self.lib.lcsx_solver_read(self.h, name.encode(), None, 0, C.byref(cnt)))
        a = np.empty(cnt.value, dtype=_dtype_of(name))
        _check(self.lib.lcsx_solver_read(self.h, name.encode(), a.ctypes.data_as(C.c_void_p), a.nbytes, None))
        return a

    def write(self, name: str, value) -> None:
        a = np.ascontiguousarray(value, dtype=np.float32).reshape(-1)
        _check(self.lib.lcsx_solver_write(self.h, name.encode(), a.ctypes.data_as(C.c_void_p), a.nbytes))

    def set_timing(self, level: int) -> None:
        _check(self.lib.lcsx_solver_set_timing(self.h, level))

    def save_state(self, path: str) -> None:
        """Writes the reference's ".state" checkpoint (positions, velocities, body q / qv)."""
        _check(self.lib.lcsx_solver_save_state(self.h, os.fspath(path).encode()))

    def load_state(self, path: str, frame: Optional[int] = None) -> None:
        """Reads a ".state" checkpoint; with frame, also sets the frame counter."""
        _check(self.lib.lcsx_solver_load_state(self.h, os.fspath(path).encode(), -1 if frame is None else int(frame)))

    def save_obj(self, path: str) -> None:
        """Writes the current positions as one OBJ with an object per mesh."""
        _check(self.lib.lcsx_solver_save_obj(self.h, os.fspath(path).encode()))

    def set_graphs(self, on: bool) -> None:
        """Replay captured hipGraphs of the PCG iterations, or launch each kernel (the default)."""
        _check(self.lib.lcsx_solver_set_graphs(self.h, int(on)))

    def set_one_launch(self, on: bool = True) -> None:
        """The PCG in one launch where the system fits (the default; takes back the choice of the launches by
        set_graphs and set_spmv_shape), or launches only."""
        _check(self.lib.lcsx_solver_set_one_launch(self.h, int(on)))

    def set_query_shape(self, shape: int) -> None:
        """Broad-phase traversal shape (0..3 binary steps, 4..6 four-wide steps of the LBVH with
        different LDS stack entries and per-wavefront pair staging; 7..9 the solver's own
        hierarchies, 16 queries per wavefront, or as 4 in scenes of thousands of pieces and batches of
        tiny scenes; every shape finds the same pairs)."""
        _check(self.lib.lcsx_solver_set_query_shape(self.h, int(shape)))

    def set_spmv_shape(self, shape: int) -> None:
        """PCG SpMV mapping (0..2: three blocks per pass with unconditional loads, three with
        predicated loads, two with unconditional loads; 3..5: the same with the contact chunks
        launched first; every shape gives the same bits)."""
        _check(self.lib.lcsx_solver_set_spmv_shape(self.h, int(shape)))

    def autotune(self) -> Dict[str, object]:
        """Times the runtime mappings on the current state and keeps the fastest (results are
        unchanged by any of them); returns the timings (ms) and the chosen settings."""
        buf = C.create_string_buffer(4096)
        _check(self.lib.lcsx_solver_autotune(self.h, buf, len(buf)))
        out: Dict[str, object] = {}
        for item in buf.value.decode().split(";"):
            if item.startswith("chosen:"):
                out["chosen"] = {k: int(v) for k, v in (kv.split("=") for kv in item[7:].split(","))}
            elif "=" in item:
                k, v = item.rsplit("=", 1)
                out[k] = float(v)
        return out

    def kernel_times(self, reset: bool = False) -> Dict[str, tuple]:
        buf = C.create_string_buffer(8192)
        _check(self.lib.lcsx_solver_kernel_times(self.h, buf, len(buf), int(reset)))
        out = {}
        for item in buf.value.decode().split(";"):
            if "=" in item:
                k, v = item.split("=")
                ms, n = v.split(",")
                out[k] = (float(ms), int(n))
        return out


def device_count() -> int:
    return int(load_library().lcsx_device_count())


class BsrSystem:
    """A block system in device memory for the standalone PCG (lcsx_pcg_solve_bsr): row_ptr (n + 1)
    and col (nnz) int32, blocks (nnz x 3 x 3) and diag (n x 3 x 3) float32, row-major blocks."""

    def __init__(self, row_ptr, col, blocks, diag):
        from . import hiprt

        self.n = int(len(row_ptr) - 1)
        self.nnz = int(len(col))
        self._dev = [hiprt.DeviceArray(np.asarray(row_ptr, dtype=np.int32)),
                     hiprt.DeviceArray(np.asarray(col, dtype=np.int32)),
                     hiprt.DeviceArray(np.asarray(blocks, dtype=np.float32).reshape(-1)),
                     hiprt.DeviceArray(np.asarray(diag, dtype=np.float32).reshape(-1))]
        self.c = lcsx_bsr(self.n, self.nnz, *(d.ptr for d in self._dev))

    @classmethod
    def from_reference_csr(cls, csr, offdiag, diag):
        """From the reference's CSR layout (init_sim_data.cpp:904-914): csr[0..n] are the absolute
        positions of each row's neighbours in csr itself (after the n + 1 header slots), and
        offdiag holds one block per csr slot."""
        csr = np.asarray(csr, dtype=np.int64)
        n = int(np.asarray(diag).reshape(-1, 9).shape[0])
        row_ptr = csr[:n + 1] - (n + 1)
        blocks = np.asarray(offdiag, dtype=np.float32).reshape(-1, 9)[n + 1:]
        return cls(row_ptr, csr[n + 1:], blocks, diag)


def pcg_solve_bsr(system: "BsrSystem", b, max_iters: int = 100, check_every: int = 25, rel_tol: float = 0.0,
                  abs_tol: float = 1e-10, no_alloc: bool = False):
    """ConjugateGradientSolver::device_solve on a caller's block system (lcsx_pcg_solve_bsr, or with
    no_alloc lcsx_pcg_solve_bsr_noalloc): returns (x as an n x 3 array, result dict)."""
    from . import hiprt

    lib = load_library()
    bd = hiprt.DeviceArray(np.asarray(b, dtype=np.float32).reshape(-1))
    xd = hiprt.DeviceArray(np.zeros(3 * system.n, dtype=np.float32))
    o = lcsx_pcg_options(max_iters, check_every, rel_tol, abs_tol)
    r = lcsx_pcg_result()
    fn = lib.lcsx_pcg_solve_bsr_noalloc if no_alloc else lib.lcsx_pcg_solve_bsr
    _check(fn(C.byref(system.c), bd.ptr, xd.ptr, C.byref(o), None, C.byref(r)))
    return xd.numpy().reshape(-1, 3), {f: getattr(r, f) for f, _ in lcsx_pcg_result._fields_}


def pcg_form_counts(device: int = 0) -> Dict[str, int]:
    """Solves of this process on a device: in one launch to their end, and as launches because the rows did not
    fit it, a wait ran out in it, or another solve held it (lcsx_pcg_form_counts)."""
    c = (C.c_uint64 * 4)()
    _check(load_library().lcsx_pcg_form_counts(device, c))
    return dict(zip(("one_launch", "unfit", "waited", "refused"), map(int, c)))


def spmv_bsr(system: "BsrSystem", x) -> np.ndarray:
    """device_SpMV on a caller's block system (lcsx_spmv_bsr): y = A x as an n x 3 array."""
    from . import hiprt

    lib = load_library()
    xd = hiprt.DeviceArray(np.asarray(x, dtype=np.float32).reshape(-1))
    yd = hiprt.DeviceArray(np.zeros(3 * system.n, dtype=np.float32))
    _check(lib.lcsx_spmv_bsr(C.byref(system.c), xd.ptr, yd.ptr, None))
    return yd.numpy().reshape(-1, 3)


def pcg_solve_op(n: int, diag, spmv, b, max_iters: int = 100, check_every: int = 25, rel_tol: float = 0.0,
                 abs_tol: float = 1e-10):
    """ConjugateGradientSolver::device_solve in its operator form (lcsx_pcg_solve_op): spmv(p_ptr,
    q_ptr, stream) enqueues q = A p on device arrays of 3 floats per row; diag holds the n 3x3
    diagonal blocks (the preconditioner). Returns (x as an n x 3 array, result dict)."""
    from . import hiprt

    lib = load_library()
    dd = hiprt.DeviceArray(np.asarray(diag, dtype=np.float32).reshape(-1))
    bd = hiprt.DeviceArray(np.asarray(b, dtype=np.float32).reshape(-1))
    xd = hiprt.DeviceArray(np.zeros(3 * n, dtype=np.float32))
    cb = SPMV_FN(lambda user, p, q, stream: spmv(p, q, stream))
    o = lcsx_pcg_options(max_iters, check_every, rel_tol, abs_tol)
    r = lcsx_pcg_result()
    _check(lib.lcsx_pcg_solve_op(int(n), dd.ptr, cb, None, bd.ptr, xd.ptr, C.byref(o), None, C.byref(r)))
    return xd.numpy().reshape(-1, 3), {f: getattr(r, f) for f, _ in lcsx_pcg_result._fields_}
