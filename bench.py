#!/usr/bin/env python3
"""Benchmark: Newton steps/s of the cloth Newton step on one MI355X.

Workload (headline): the 297 x 297-vertex cloth tube (88,209 vertices, 175,824 triangles,
r = 0.11 m, length 1 m) around a kinematic cylinder (r = 0.1 m, 5,760 vertices) spinning at
2*pi rad/s, tube ends pinned to the spin, both started in the steady spin; dt = 1/60 s, self
contact with d_hat = 1e-3 m and kappa = 1e9, gravity (0, 0, 0) as in the reference's own
cylinder scenes (cloth_rotation_cylinder_88K.json), FP32. A bench "step" is one simulated frame
(each frame runs >= 3 Newton iterations, each with <= 100 PCG iterations); `value` is Newton
iterations per second over the timed frames, with every input resident on the GPU.

The JSON line carries:
  value         Newton steps/s in FP32 (the reference's precision).
  config        the workload, frames/s, Newton iterations per frame (mean, max, frames at the
                100-iteration cap), the smallest CCD step bound of the timed frames, and the
                zero-penetration check (smallest FP64 gap d - offsets over the candidate pairs
                after every frame, and the count of pairs at or below zero).
  narrow_phase  pairs/s of the swept broad phase + CCD and of the DCD (candidate pairs per Newton
                iteration divided by the kernel groups' device time).
  mixed         the same frames in mixed precision (FP16 off-diagonal blocks with a power-of-two
                scale per block inside the PCG, FP32 vectors with residual replacement every 25
                iterations, FP64 CCD and barrier terms): Newton steps/s and its SpMV figures.
  roofline      the PCG block SpMV k_spmv_pcg of the FP32 run (material blocks and contact
                slots), sampled in the frame after the timed ones (sampling takes the launched form
                of the PCG): algorithmic bytes per launch = 40 B per off-diagonal block (36 B values +
                4 B column) + 64 B per row (36 B diagonal block, 16 B p row, 12 B q written) + 4 B
                per 16-row slice + 24 B per contact slot, divided by the launch's average duration
                from hipEvents attached to the launches (hipExtLaunchKernelGGL) on the solver
                stream; peak = 8 TB/s HBM3E. The 16-bit launch moves 24 B per off-diagonal block
                (20 B packed entries and exponent, 4 B column) and the same per row.
  tube_gravity  the same tube under gravity -9.8 m/s^2 from the first frame: it drapes onto the
                cylinder and from about frame 4 every line search ends at ACCD's 10,001-iteration
                fallback bound (toi 0.001) and the Newton loop runs to its cap; per-frame Newton
                iterations, step bounds, candidate pairs and seconds for a bounded number of frames.
  batched       the batched form on 256 cloth-on-sphere scenes (grid side n ~ U{17..161},
                sphere r = 0.3 m offset U(-0.1, 0.1) m in x and z, seed 0; 2.81M vertices): all
                scenes in one solver (one launch per stage) against the same scenes stepped one by
                one, each from the batch's state after the warm-up frames (the cloths reach the
                spheres at about frame 12). Scene-steps/s = scenes x frames / seconds.
  coupling      cloth-rigid coupling (129 x 129 cloth, 24 affine-body boxes): Newton steps/s in FP32
                and mixed precision over 60 frames, and both trajectories' relative position error
                against the FP64 oracle over the first 24 frames (the first box-cloth contacts
                come at about frame 20).
  cpu_baseline  the CPU oracle (C++ restatement of the reference path) timed on the same work:
                the Newton iteration the GPU timed, from the same state.
"""
import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "Newton steps/s @88K-vert cloth, mixed vs FP32; SpMV HBM GB/s; scene-steps/s"
COUNT_KEYS = ("spmv_slots", "pairs_ccd", "pairs_dcd", "contacts")
HBM_PEAK_GBS = 8000.0


def spmv_bytes(n_rows: int, n_blocks: int, slots: float = 0.0, block_bytes: int = 40) -> float:
    """Algorithmic bytes of one k_spmv_pcg launch: block_bytes per off-diagonal block (40 in FP32:
    36 B values + 4 B column; 24 with 16-bit blocks: 20 B of packed entries and exponent + 4 B
    column) + 64 B per row (36 B diagonal block, 16 B p row, 12 B q written) + 4 B per 16-row
    slice offset, and 24 B per contact slot (16 B coefficient, 4 B row, the contact's 4 B t_c; the
    16 B sum each run of a row's slots writes is not counted)."""
    return block_bytes * n_blocks + 64 * n_rows + 4 * ((n_rows + 15) // 16) + 24 * slots


def traffic_from_profiles():
    """HBM bytes per SpMV launch and the algorithmic bytes of that same launch, from the committed
    rocprofv3 counter summary (lines `hbm_bytes_per_launch:` / `algorithmic_bytes_per_launch:` of
    profiles/k_spmv_pcg_tube88k_counters.md), or (None, None)."""
    path = os.path.join(ROOT, "profiles", "k_spmv_pcg_tube88k_counters.md")
    out = {}
    if os.path.exists(path):
        with open(path) as f:
            for line in f:
                key, _, val = line.strip().partition(":")
                if key in ("hbm_bytes_per_launch", "algorithmic_bytes_per_launch") and val.strip():
                    out[key] = float(val.strip())
    return out.get("hbm_bytes_per_launch"), out.get("algorithmic_bytes_per_launch")


def profile_pcg(g, copy_mib: int = 256) -> None:
    """Counter-run workload (rocprofv3 --pmc): one device-to-device copy of `copy_mib` MiB (the
    calibration kernel of known size) followed by one PCG solve (up to 100 SpMV launches) on the
    system of the last Newton iteration."""
    import numpy as np

    from luisacomputesimulator_amd import hiprt

    src = hiprt.DeviceArray(np.zeros(copy_mib << 18, dtype=np.float32))
    dst = hiprt.DeviceArray(np.zeros(copy_mib << 18, dtype=np.float32))
    hiprt.copy_device(dst, src)
    hiprt.synchronize()
    g.stage("pcg")
    hiprt.synchronize()
    st = g.stats()
    print(f"[bench] profile-pcg: copied {copy_mib} MiB, PCG {st['pcg_iters']} iterations", file=sys.stderr, flush=True)


def batched_leg(args, precision, sequential):
    """Batched vs one-by-one scene-steps/s on the cloth-on-sphere batch."""
    from luisacomputesimulator_amd import NewtonSolver, hiprt, scenes

    scs = scenes.sphere_batch(args.batch_scenes, seed=0)
    for sc in scs:
        sc.params.precision = precision
    t = time.perf_counter()
    b = NewtonSolver.from_scenes(scs)
    print(f"[bench] batch {precision}: {len(scs)} scenes, {b.num_verts} vertices, setup {time.perf_counter() - t:.1f} s",
          file=sys.stderr, flush=True)
    for f in range(args.batch_warmup):
        tw = time.perf_counter()
        b.physics_step_gpu(1)
        st = b.stats()
        print(f"[bench] batch {precision} warmup frame {f}: {st['newton_iters']} scene-Newton, {st['num_contacts']} contacts, "
              f"{time.perf_counter() - tw:.2f} s", file=sys.stderr, flush=True)
    tuned = None
    if args.query_shape >= 0:
        b.set_query_shape(args.query_shape)
    if not args.no_autotune:
        # runtime mappings timed on the warm batch state (results do not depend on them)
        report = b.autotune()
        tuned = report["chosen"]
        print(f"[bench] batch {precision} autotune: {report}", file=sys.stderr, flush=True)
    x0, v0 = b.get_simulation_results(), b.get_velocities()
    ranges = [b.scene_range(g) for g in range(len(scs))]
    hiprt.synchronize()
    newton = 0
    t0 = time.perf_counter()
    for f in range(args.batch_steps):
        b.physics_step_gpu(1)
        newton += b.stats()["newton_iters"]
    hiprt.synchronize()
    el = time.perf_counter() - t0
    out = {"scene_steps_per_s": len(scs) * args.batch_steps / el, "ms_per_frame": 1e3 * el / args.batch_steps,
           "scene_newton_iters": newton, "contacts_last_iter": b.stats()["num_contacts"], "autotuned": tuned}
    print(f"[bench] batch {precision} timed: {out}", file=sys.stderr, flush=True)
    del b
    if sequential:
        total, newton_s = 0.0, 0
        for g, sc in enumerate(scs):
            a, n = ranges[g]
            one = NewtonSolver.from_scene(sc)
            one.set_state(x0[a:a + n], v0[a:a + n])
            one.physics_step_gpu(1)  # warm-up frame (buffer sizes), then back to the batch's state
            one.set_state(x0[a:a + n], v0[a:a + n])
            hiprt.synchronize()
            t0 = time.perf_counter()
            for f in range(args.batch_steps):
                one.physics_step_gpu(1)
                newton_s += one.stats()["newton_iters"]
            hiprt.synchronize()
            total += time.perf_counter() - t0
            del one
            if g % 64 == 63:
                print(f"[bench] one-by-one: {g + 1} scenes, {total:.2f} s", file=sys.stderr, flush=True)
        out["one_by_one_scene_steps_per_s"] = len(scs) * args.batch_steps / total
        out["one_by_one_scene_newton_iters"] = newton_s
        out["speedup_vs_one_by_one"] = out["scene_steps_per_s"] / out["one_by_one_scene_steps_per_s"]
    return out


def coupling_leg(args):
    """Cloth-rigid coupling (129 x 129 cloth pinned at its corners, 24 affine-body boxes): Newton
    steps/s of all frames in FP32 and in mixed precision with FP16 and with BF16 block storage, and
    the position error of each against the FP64 oracle over the first frames (a bounded CPU
    sample)."""
    import numpy as np

    import oracle
    from luisacomputesimulator_amd import NewtonSolver, hiprt, scenes

    out = {"workload": "129x129 cloth pinned at 4 corners + 24 affine-body boxes (0.1 m, solid, density 500, "
                       "stiffness 1e8), seed 0", "frames": args.coupling_frames}
    traj = {}
    for prec in ("fp32", "mixed", "mixed_bf16"):
        sc = scenes.cloth_rigid_coupling(129, 24, seed=0)
        sc.params.precision = prec
        g = NewtonSolver.from_scene(sc)
        nv = sc.num_verts
        hiprt.synchronize()
        newton, xs = 0, []
        t0 = time.perf_counter()
        for f in range(args.coupling_frames):
            g.physics_step_gpu(1)
            newton += g.stats()["newton_iters"]
            if f < args.coupling_oracle_frames:
                xs.append(g.get_simulation_results()[:nv].copy())
        hiprt.synchronize()
        el = time.perf_counter() - t0
        out[prec] = {"newton_steps_per_s": newton / el, "frames_per_s": args.coupling_frames / el,
                     "newton_iters": newton, "contacts_last_iter": g.stats()["num_contacts"]}
        traj[prec] = xs
        print(f"[bench] coupling {prec}: {out[prec]}", file=sys.stderr, flush=True)
    out["mixed_speedup_vs_fp32"] = out["mixed"]["newton_steps_per_s"] / out["fp32"]["newton_steps_per_s"]
    out["mixed_bf16_speedup_vs_fp32"] = out["mixed_bf16"]["newton_steps_per_s"] / out["fp32"]["newton_steps_per_s"]
    if args.coupling_oracle_frames > 0:
        sc = scenes.cloth_rigid_coupling(129, 24, seed=0)
        o64 = oracle.Oracle(sc, 64)
        err = {"fp32": [], "mixed": [], "mixed_bf16": []}
        t0 = time.perf_counter()
        for f in range(args.coupling_oracle_frames):
            o64.step()
            x64 = o64.get("x").reshape(-1, 3)[:sc.num_verts]
            scale = np.abs(x64).max()
            for prec in err:
                err[prec].append(float(np.abs(traj[prec][f] - x64).max() / scale))
            print(f"[bench] coupling FP64 oracle frame {f}: fp32 {err['fp32'][-1]:.2e} mixed {err['mixed'][-1]:.2e} "
                  f"mixed_bf16 {err['mixed_bf16'][-1]:.2e}", file=sys.stderr, flush=True)
        out["rel_error_vs_fp64_per_frame"] = err
        out["oracle_seconds"] = time.perf_counter() - t0
    return out


def spmv_large_leg(args):
    """The PCG SpMV on the 513 x 513 twisting sheet's material system (263,169 rows, about 146 MB of
    FP32 blocks per launch, more than the 256 MB Infinity Cache holds with the rest of the solve):
    one PCG solve of frame 0 with every SpMV launch timed, FP32 and FP16 blocks."""
    from luisacomputesimulator_amd import NewtonSolver, scenes

    out = {"workload": f"twisting sheet {args.n}x{args.n}, frame 0 material system, one PCG solve"}
    for prec in ("fp32", "mixed"):
        sc = scenes.twisting_sheet(args.n)
        sc.params.precision = prec
        g = NewtonSolver.from_scene(sc)
        g.set_timing(3)
        for st in ("frame_begin", "predict", "iter_begin", "material", "update_contacts", "contact_assemble"):
            g.stage(st)
        g.kernel_times(reset=True)
        g.stage("pcg")
        kt = g.kernel_times()
        ms, n = kt.get("spmv", (float("nan"), 0))
        n_rows = g.num_verts
        n_blocks = len(g.read("csr")) - (n_rows + 1)
        nbytes = spmv_bytes(n_rows, n_blocks, kt.get("spmv_slots", (0.0, 0))[0], 40 if prec == "fp32" else 24)
        gbs = nbytes / (ms * 1e-3) / 1e9 if n else None
        out[prec] = {"avg_launch_ms": ms, "launches": n, "bytes_per_launch": nbytes, "achieved_gbs": gbs,
                     "frac": gbs / HBM_PEAK_GBS if gbs else None, "rows": n_rows, "blocks": n_blocks}
        print(f"[bench] spmv_large {prec}: {n} launches, {ms * 1e3:.2f} us, {nbytes / 1e6:.1f} MB, "
              f"{(gbs or 0) / 1e3:.2f} TB/s", file=sys.stderr, flush=True)
        del g
    if out["fp32"]["launches"] and out["mixed"]["launches"]:
        out["mixed_over_fp32_time"] = out["mixed"]["avg_launch_ms"] / out["fp32"]["avg_launch_ms"]
    return out


def twist_error_leg(args):
    """Twisting sheet at a size the FP64 oracle finishes in minutes (n x n, edges turned at -/+ pi
    rad/s, 120 frames): relative position error of the GPU's FP32, mixed (FP16) and mixed (BF16)
    forms, and of the FP32 oracle, against the FP64 oracle at frames 30, 60 and 120."""
    import numpy as np

    import oracle
    from luisacomputesimulator_amd import NewtonSolver, scenes

    n, marks = args.twist_error_n, (30, 60, 120)
    out = {"workload": f"twisting sheet {n}x{n}, edges turned at -/+ pi rad/s, 120 frames", "frames": list(marks)}
    xs = {}
    for prec in ("fp32", "mixed", "mixed_bf16"):
        sc = scenes.twisting_sheet(n)
        sc.params.precision = prec
        g = NewtonSolver.from_scene(sc)
        t0, newton, xs[prec] = time.perf_counter(), 0, {}
        for f in range(1, marks[-1] + 1):
            g.physics_step_gpu(1)
            newton += g.stats()["newton_iters"]
            if f in marks:
                xs[prec][f] = g.get_simulation_results().copy()
        out[prec] = {"newton_iters": newton, "seconds": time.perf_counter() - t0}
        print(f"[bench] twist {n} {prec}: {newton} Newton iterations", file=sys.stderr, flush=True)
    sc = scenes.twisting_sheet(n)
    o64, o32 = oracle.Oracle(sc, 64), oracle.Oracle(sc, 32)
    err = {k: [] for k in ("fp32", "mixed", "mixed_bf16", "oracle_fp32")}
    t0 = time.perf_counter()
    for f in range(1, marks[-1] + 1):
        o64.step()
        o32.step()
        if f in marks:
            x64 = o64.get("x").reshape(-1, 3)
            scale = np.abs(x64).max()
            for prec in ("fp32", "mixed", "mixed_bf16"):
                err[prec].append(float(np.abs(xs[prec][f] - x64).max() / scale))
            err["oracle_fp32"].append(float(np.abs(o32.get("x").reshape(-1, 3) - x64).max() / scale))
            print(f"[bench] twist {n} frame {f} vs FP64: " + ", ".join(f"{k} {v[-1]:.2e}" for k, v in err.items()),
                  file=sys.stderr, flush=True)
    out["rel_error_vs_fp64"] = err
    out["oracle_seconds"] = time.perf_counter() - t0
    return out


def cpu_model() -> str:
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_baseline_same_iteration(g, scene, args, iters: int = 3):
    """The CPU oracle (the C++ restatement of the reference path, FP32, OpenMP) timed on the same
    work as the GPU: from the GPU's state after its timed frames, the next frame's first `iters`
    Newton iterations (frame begin and prediction untimed), on both. The positions after them are
    compared, so the two did the same work."""
    import numpy as np

    import oracle
    from luisacomputesimulator_amd import hiprt

    threads = args.cpu_threads if args.cpu_threads > 0 else min(os.cpu_count() or 1, 16)
    threads = oracle.set_threads(threads)
    x, v, frame = g.get_simulation_results(), g.get_velocities(), g.stats()["frame"]
    # GPU: the same iterations from the same state
    g.set_state(x, v)
    g.stage("frame_begin")
    g.stage("predict")
    hiprt.synchronize()
    t0 = time.perf_counter()
    for _ in range(iters):
        g.stage("newton_iteration")
    hiprt.synchronize()
    gpu_s = time.perf_counter() - t0
    xg = g.read("x").reshape(-1, 3)
    o = oracle.Oracle(scene, 32)
    o.set("x_outer", x)
    o.set("v_outer", v)
    o.set_frame(frame)
    o.stage("frame_begin")
    o.stage("predict")
    t0 = time.perf_counter()
    for _ in range(iters):
        o.stage("newton_iteration")
    cpu_s = time.perf_counter() - t0
    xo = o.get("x").reshape(-1, 3)
    rel = float(np.abs(xg - xo).max() / np.abs(xo).max())
    # per iteration, untimed: position difference and both step bounds (a CCD bound that lands on
    # the other side of a pair's ACCD fallback separates the two by a whole step)
    per_iter = []
    g.set_state(x, v)
    g.stage("frame_begin")
    g.stage("predict")
    o2 = oracle.Oracle(scene, 32)
    o2.set("x_outer", x)
    o2.set("v_outer", v)
    o2.set_frame(frame)
    o2.stage("frame_begin")
    o2.stage("predict")
    for _ in range(iters):
        g.stage("newton_iteration")
        o2.stage("newton_iteration")
        xa, xb = g.read("x").reshape(-1, 3), o2.get("x").reshape(-1, 3)
        per_iter.append({"rel_diff": float(np.abs(xa - xb).max() / np.abs(xb).max()),
                         "toi_gpu": float(g.read("toi")[0]), "toi_cpu": float(o2.scalars()["toi"])})
    oracle.set_threads(1)
    print(f"[bench] cpu_baseline: {iters} Newton iterations from frame {frame}: CPU {cpu_s:.2f} s on {threads} threads, "
          f"GPU {gpu_s * 1e3:.2f} ms, positions differ by {rel:.2e} relative", file=sys.stderr, flush=True)
    return {"value": iters / cpu_s, "unit": "Newton steps/s", "cores": threads, "kind": "port",
            "cpu_model": cpu_model(),
            "sample": f"the first {iters} Newton iterations of frame {frame} of the same {scene.num_verts}-vertex scene "
                      f"from the GPU's state after its timed frames ({cpu_s:.1f} s; C++ oracle, FP32, OpenMP "
                      f"{threads} threads)",
            "gpu_same_iterations_s": gpu_s, "gpu_speedup": cpu_s / gpu_s, "positions_rel_diff": rel,
            "per_iteration": per_iter}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--workload", choices=("tube", "twist"), default="tube",
                    help="tube: the 297 x 297 cloth tube on the spinning cylinder (the headline workload); "
                         "twist: the 513 x 513 sheet twisted by its two pinned edges")
    ap.add_argument("--rings", type=int, default=297, help="tube: rings (= vertices per ring)")
    ap.add_argument("--n", type=int, default=513, help="twist: vertices per side")
    ap.add_argument("--precision", choices=("fp32", "mixed", "both"), default="both",
                    help="fp32: the reference's precision (the headline value); mixed: FP16 blocks in the PCG "
                         "with FP32 residual replacement, FP64 CCD/barrier; both: FP32 headline plus a mixed "
                         "run of the same frames")
    ap.add_argument("--batch-scenes", type=int, default=256, help="batched leg: number of scenes (0: skip)")
    ap.add_argument("--batch-steps", type=int, default=3, help="batched leg: timed frames")
    ap.add_argument("--batch-warmup", type=int, default=16, help="batched leg: frames before timing")
    ap.add_argument("--coupling-frames", type=int, default=60, help="cloth-rigid leg: GPU frames (0: skip)")
    ap.add_argument("--legs", default="tube,tube_gravity,batch,coupling,spmv_large",
                    help="comma list of legs: tube (the headline), tube_gravity, batch, coupling, spmv_large, "
                         "twist_error (not run by default: its FP64 oracle takes minutes)")
    ap.add_argument("--tube-gravity", type=float, default=0.0,
                    help="tube: gravity magnitude of the headline run (m/s^2, default 0 as the reference's "
                         "cylinder scenes)")
    ap.add_argument("--gravity-frames", type=int, default=8, help="tube_gravity leg: frames from the start")
    ap.add_argument("--cpu-threads", type=int, default=0,
                    help="cpu_baseline: OpenMP threads of the CPU oracle (0: all host cores, at most 16)")
    ap.add_argument("--twist-error-n", type=int, default=65, help="twist_error leg: vertices per side")
    ap.add_argument("--no-autotune", action="store_true", help="keep the default runtime mappings")
    ap.add_argument("--query-shape", type=int, default=-1,
                    help="broad-phase traversal shape 0..9 for the tube runs (default: the library's, or the "
                         "autotuner's choice)")
    ap.add_argument("--coupling-oracle-frames", type=int, default=24,
                    help="cloth-rigid leg: frames compared with the FP64 oracle")
    ap.add_argument("--profile-pcg", action="store_true",
                    help="after the warm-up frames run one calibration copy and one PCG solve, then exit "
                         "(workload for rocprofv3 counter runs)")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU: the workload is a single scene on one MI355X and the solver "
              "has no multi-GPU path. Run with --gpus 1.",
              file=sys.stderr)
        sys.exit(2)

    from luisacomputesimulator_amd import NewtonSolver, hiprt, scenes

    def make_scene(gravity=None):
        if args.workload == "tube":
            g = (0.0, -args.tube_gravity, 0.0) if gravity is None else gravity
            return scenes.cylinder_tube(rings=args.rings, per_ring=args.rings, gravity=g)
        return scenes.twisting_sheet(args.n)

    sc = make_scene()
    if args.workload == "tube":
        label = (f"cloth tube {args.rings}x{args.rings} ({sc.meshes[0].verts.shape[0]} verts, "
                 f"{sc.meshes[0].tris.shape[0]} tris) around a spinning kinematic cylinder, dt 1/60 s, kappa 1e9, "
                 f"gravity {-args.tube_gravity:g} m/s^2")
    else:
        label = (f"twisting sheet {args.n}x{args.n} ({sc.num_verts} verts, {sc.num_faces} tris), edges turned "
                 "at -/+ pi rad/s, d_hat 5e-4 m, dt 1/60 s")

    def frame_record(st, t):
        return {"newton": st["newton_iters"], "pcg": st["pcg_iters_total"], "toi_min": st["toi_min"],
                "ccd_pairs": st["num_ccd_pairs"], "contacts": st["num_contacts"], "min_gap": st["min_gap"],
                "penetrating": st["num_penetrating"], "s": round(t, 4)}

    def run(precision):
        """Warm-up and timed frames of a fresh solver in one precision."""
        s = make_scene()
        s.params.precision = precision
        g = NewtonSolver.from_scene(s)
        g.set_timing(1)
        if args.query_shape >= 0:
            g.set_query_shape(args.query_shape)
        tag = precision

        def progress(kind, f, st, t):
            print(f"[bench] {tag} {kind} frame {f}: {st['newton_iters']} Newton, {st['pcg_iters_total']} PCG "
                  f"iterations, min step bound {st['toi_min']:.4g}, {st['num_ccd_pairs']} CCD candidates, "
                  f"{st['num_contacts']} contacts, min gap {st['min_gap']:.3e} m, {st['num_penetrating']} penetrating, "
                  f"{t:.2f} s", file=sys.stderr, flush=True)

        for f in range(args.warmup):
            tw = time.perf_counter()
            g.physics_step_gpu(1)
            progress("warmup", f, g.stats(), time.perf_counter() - tw)
        tuned = None
        if not args.no_autotune:
            # runtime mappings timed on the warm state (results do not depend on them)
            report = g.autotune()
            tuned = report["chosen"]
            print(f"[bench] {tag} autotune: {report}", file=sys.stderr, flush=True)
        if args.profile_pcg:
            profile_pcg(g)
            return None
        g.kernel_times(reset=True)
        hiprt.synchronize()
        newton = pcg = 0
        frames = []
        t0 = time.perf_counter()
        for f in range(args.steps):
            tf = time.perf_counter()
            g.physics_step_gpu(1)
            st = g.stats()
            newton += st["newton_iters"]
            pcg += st["pcg_iters_total"]
            frames.append(frame_record(st, time.perf_counter() - tf))
            progress("timed", f, st, time.perf_counter() - tf)
        hiprt.synchronize()
        elapsed = time.perf_counter() - t0
        kt, st = g.kernel_times(), g.stats()
        # the SpMV's own duration, in the launched form of the PCG, from the frame after the timed ones
        g.set_timing(2)
        g.kernel_times(reset=True)
        g.physics_step_gpu(1)
        kt_spmv = g.kernel_times()
        g.set_timing(1)
        n_rows = g.num_verts
        n_blocks = len(g.read("csr")) - (n_rows + 1)
        spmv_ms, spmv_n = kt_spmv.get("spmv", (float("nan"), 0))
        slots = kt_spmv.get("spmv_slots", (0.0, 0))[0]
        nbytes = spmv_bytes(n_rows, n_blocks, slots, 24 if precision == "mixed" else 40)
        out = {"elapsed": elapsed, "newton": newton, "pcg": pcg, "kt": kt, "st": st, "n_rows": n_rows,
               "tuned": tuned, "frames": frames, "n_blocks": n_blocks, "spmv_ms": spmv_ms, "spmv_n": spmv_n,
               "slots": slots, "nbytes": nbytes,
               "achieved": nbytes / (spmv_ms * 1e-3) / 1e9 if spmv_n else None}
        if precision == "fp32" and not args.no_cpu_baseline:
            out["cpu_baseline"] = cpu_baseline_same_iteration(g, s, args)
        return out

    def frames_summary(frames, max_iters):
        newton = [f["newton"] for f in frames]
        gaps = [f["min_gap"] for f in frames if f["min_gap"] == f["min_gap"]]
        return {"newton_per_frame_mean": sum(newton) / max(len(newton), 1), "newton_per_frame_max": max(newton),
                "frames_at_newton_cap": sum(1 for n in newton if n >= max_iters),
                "toi_min": min(f["toi_min"] for f in frames),
                "min_gap_m": min(gaps) if gaps else None,
                "penetrating_pairs_total": sum(max(f["penetrating"], 0) for f in frames)}

    def narrow_phase_rates(kt):
        """Pairs/s of the swept broad phase and CCD and of the DCD: candidate pairs per Newton
        iteration over the kernel groups' average device time per iteration."""
        def avg(k):
            return kt.get(k, (0.0, 0))[0]
        pc, pd = avg("pairs_ccd"), avg("pairs_dcd")
        out = {"ccd_candidates_per_iter": pc, "dcd_candidates_per_iter": pd, "contacts_per_iter": avg("contacts")}
        for name, pairs, key in (("swept_query", pc, "broadphase_ccd"), ("ccd", pc, "ccd"), ("dcd", pd, "dcd")):
            ms = avg(key)
            out[name + "_ms"] = ms
            out[name + "_pairs_per_s"] = pairs / (ms * 1e-3) if ms > 0 else None
        return out

    def gravity_leg():
        """The tube under gravity from the first frame (bounded frames, per-frame records)."""
        s = make_scene(gravity=(0.0, -9.8, 0.0))
        g = NewtonSolver.from_scene(s)
        frames = []
        for f in range(args.gravity_frames):
            tf = time.perf_counter()
            g.physics_step_gpu(1)
            st = g.stats()
            frames.append(frame_record(st, time.perf_counter() - tf))
            print(f"[bench] tube_gravity frame {f}: {frames[-1]}", file=sys.stderr, flush=True)
        cap = s.params.newton_max_iters
        first = next((i for i, fr in enumerate(frames) if fr["newton"] >= cap), None)
        return {"workload": label.replace(f"gravity {-args.tube_gravity:g}", "gravity -9.8") + ", FP32",
                "frames": frames, "first_frame_at_newton_cap": first, **frames_summary(frames, cap)}

    precisions = {"fp32": ["fp32"], "mixed": ["mixed"], "both": ["fp32", "mixed"]}[args.precision]
    legs = set(args.legs.split(","))
    if "tube" not in legs:
        # a profiling run of the other legs: their JSON objects only
        line = {"metric": METRIC, "value": None, "unit": "Newton steps/s", "n_gpus": 1, "legs": sorted(legs)}
        if "batch" in legs and args.batch_scenes > 0:
            line["batched"] = {"fp32": batched_leg(args, precisions[0], sequential=False)}
        if "coupling" in legs and args.coupling_frames > 0:
            line["coupling"] = coupling_leg(args)
        if "spmv_large" in legs:
            line["spmv_large"] = spmv_large_leg(args)
        if "twist_error" in legs:
            line["twist_error"] = twist_error_leg(args)
        print(json.dumps(line), flush=True)
        return
    res = {}
    for prec in precisions:
        res[prec] = run(prec)
        if res[prec] is None:
            return
    head = res[precisions[0]]
    n_rows, n_blocks, st, kt = head["n_rows"], head["n_blocks"], head["st"], head["kt"]
    traffic = traffic_from_profiles()
    line = {
        "metric": METRIC,
        "value": head["newton"] / head["elapsed"],
        "unit": "Newton steps/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": 1e3 * head["elapsed"] / args.steps,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32" if precisions[0] == "fp32" else "f16/f32/f64 mixed",
        "data": "synthetic",
        "config": {"workload": label + (", FP32" if precisions[0] == "fp32" else ", mixed precision"),
                   "verts_total": n_rows, "material_blocks": n_blocks, "frames": args.steps,
                   "newton_iters": head["newton"], "pcg_iters": head["pcg"],
                   "frames_per_s": args.steps / head["elapsed"],
                   **frames_summary(head["frames"], sc.params.newton_max_iters),
                   "contacts_last_iter": st["num_contacts"],
                   "pairs_last_iter": st["num_pairs_vf"] + st["num_pairs_ee"],
                   "ccd_pairs_last_iter": st["num_ccd_pairs"]},
        "narrow_phase": narrow_phase_rates(kt),
        "frames": head["frames"],
        "roofline": {"bound": "hbm", "achieved": head["achieved"], "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": (head["achieved"] / HBM_PEAK_GBS) if head["achieved"] else None,
                     "traffic": traffic[0] if precisions[0] == "fp32" else None,
                     "traffic_algorithmic_bytes": traffic[1] if precisions[0] == "fp32" else None,
                     "kernel": "k_spmv_pcg", "bytes_per_launch": head["nbytes"], "avg_launch_ms": head["spmv_ms"],
                     "contact_slots_per_launch": head["slots"],
                     "launches": head["spmv_n"]},
        "kernel_ms": {k: round(v[0], 4) for k, v in kt.items() if k not in COUNT_KEYS},
        "autotuned": head["tuned"],
    }
    if "mixed" in res and precisions[0] != "mixed":
        m = res["mixed"]
        line["mixed"] = {"value": m["newton"] / m["elapsed"], "unit": "Newton steps/s",
                         "speedup_vs_fp32": (m["newton"] / m["elapsed"]) / line["value"],
                         "ms_per_step": 1e3 * m["elapsed"] / args.steps,
                         "newton_iters": m["newton"], "pcg_iters": m["pcg"],
                         **frames_summary(m["frames"], sc.params.newton_max_iters),
                         "spmv_avg_launch_ms": m["spmv_ms"], "spmv_bytes_per_launch": m["nbytes"],
                         "spmv_achieved_gbs": m["achieved"],
                         "pcg_ms": round(m["kt"].get("pcg", (float("nan"), 0))[0], 4)}
    if "tube_gravity" in legs and args.workload == "tube" and args.gravity_frames > 0:
        line["tube_gravity"] = gravity_leg()
    if "batch" in legs and args.batch_scenes > 0:
        line["batched"] = {"workload": f"{args.batch_scenes} cloth-on-sphere scenes, n ~ U{{17..161}}, seed 0",
                           "unit": "scene-steps/s", "frames": args.batch_steps, "warmup_frames": args.batch_warmup,
                           "fp32": batched_leg(args, "fp32", sequential=True)}
        if "mixed" in precisions:
            line["batched"]["mixed"] = batched_leg(args, "mixed", sequential=False)
    if "coupling" in legs and args.coupling_frames > 0:
        line["coupling"] = coupling_leg(args)
    if "spmv_large" in legs:
        line["spmv_large"] = spmv_large_leg(args)
    if "twist_error" in legs:
        line["twist_error"] = twist_error_leg(args)
    if "cpu_baseline" in head:
        line["cpu_baseline"] = head["cpu_baseline"]
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
