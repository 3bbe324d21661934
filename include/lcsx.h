/*
 * lcsx: MI355X-native Newton step for IPC cloth simulation (C ABI).
 *
 * This is the drop-in boundary for the reference's per-Newton-step subsystems. The reference
 * exposes C++ classes, not a C ABI; every entry point below names the reference interface it
 * replaces (paths relative to the reference repository root):
 *
 *   NewtonSolver / SolverInterface   Solver/SimulationSolver/newton_solver.h:29-51,
 *                                    Solver/SimulationSolver/solver_interface.h:71-108
 *   Python binding (lcs_solver_py)   PythonBindings/python_bindings.cpp:303-359
 *   LBVH                             Solver/CollisionDetector/lbvh.h:183-223
 *   NarrowPhasesDetector             Solver/CollisionDetector/narrow_phase.h:54-201
 *   ConjugateGradientSolver          Solver/LinearSolver/precond_cg.h:38-47
 *
 * Conventions: plain pointers and sizes, no C++ or torch types. Host arrays unless the name
 * says "device". Positions are packed float triples (12 bytes per vertex). Every call returns
 * an lcsx_status; lcsx_last_error() gives a message for the last failure on the calling thread.
 * Errors are reported, never aborted on: the reference's LUISA_ERROR paths become
 * LCSX_ERR_NAN / LCSX_ERR_STATE, and its resize-and-retry on buffer overflow is done inside
 * the library (LCSX_ERR_CAPACITY only if growth is impossible).
 */
#ifndef LCSX_H
#define LCSX_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef enum lcsx_status
{
    LCSX_OK           = 0,
    LCSX_ERR_ARG      = 1, /* invalid argument or size                                    */
    LCSX_ERR_STATE    = 2, /* call out of order (e.g. step before init)                    */
    LCSX_ERR_HIP      = 3, /* a HIP runtime call failed                                    */
    LCSX_ERR_CAPACITY = 4, /* a contact buffer could not be grown                          */
    LCSX_ERR_NAN      = 5, /* NaN/Inf in the Newton system or the step (reference: LUISA_ERROR) */
    LCSX_ERR_IO       = 6, /* file could not be read or parsed                             */
    LCSX_ERR_NO_GPU   = 7  /* no HIP device available                                      */
} lcsx_status;

typedef struct lcsx_solver lcsx_solver;

/* ClothMaterial, Solver/SimulationCore/physical_material.h:45-63 (same field meaning). */
typedef struct lcsx_material
{
    float thickness;              /* m; contact offset per vertex is thickness / 2          */
    float youngs_modulus;         /* Pa                                                     */
    float poisson_ratio;
    float area_bending_stiffness;
    float density;                /* kg/m^3; mass = area * thickness * density when mass==0 */
    float mass;                   /* total mesh mass, 0 = from density                      */
    float d_hat;                  /* barrier activation distance, m                         */
    int   body;                   /* 0 cloth; 1 rigid shell (affine body, surface mass); 2 rigid
                                     solid (affine body of a closed surface, contact thickness 0)
                                     (RigidMaterial, physical_material.h:69-77)              */
    float rigid_stiffness;        /* RigidMaterial::stiffness: orthogonality kappa          */
    int   stretch_spring;         /* cloth stretch model: 0 Baraff-Witkin FEM (FEM_BW98, the
                                     reference's default), 1 a spring on every edge with stiffness
                                     thickness * E / (2 (1 + nu)) (ConstitutiveStretchModelCloth::
                                     Spring, physical_material.h:10-15, init_sim_data.cpp:205-370) */
} lcsx_material;

/* FixedPointAnimationInfo, Solver/Initializer/init_mesh_data.h:39-93. */
typedef struct lcsx_fixed_anim
{
    int   use_translate;
    float translate[3];
    int   use_scale;
    float scale[3];
    int   use_rotate;
    float rot_center[3];
    float rot_axis[3];
    float rot_deg_per_s;
} lcsx_fixed_anim;

/* SceneParams fields that the Newton step reads (Solver/SimulationCore/scene_params.h:15-182). */
typedef struct lcsx_params
{
    float implicit_dt;          /* s                                                         */
    int   nonlinear_iter_count; /* minimum Newton iterations per frame (reference default 3) */
    int   newton_max_iters;     /* hard cap (reference: 100)                                 */
    int   pcg_iter_count;       /* PCG iteration cap (reference default 100)                 */
    int   pcg_check_every;      /* PCG convergence test interval (reference: 25)             */
    float pcg_rel_tol;          /* also stop when r.z <= tol^2 * r0.z0 (0: off, reference)   */
    float pcg_abs_tol;          /* ... or r.z < abs_tol (reference: 1e-10)                   */
    float gravity[3];
    int   use_floor;
    int   use_self_collision;
    int   use_ccd_linesearch;
    float floor_y;
    float stiffness_collision;  /* kappa                                                     */
    float stiffness_dirichlet;  /* pinned-vertex inertia multiplier (reference: 1e9)         */
    float damping_cloth;        /* velocity damping, v *= exp(-damping * dt)                 */
    float bending_scaling;      /* stiffness_bending_ui                                      */
    float newton_tol;           /* converged when max|dx| < newton_tol * dt                  */
    int   precision;            /* 0: FP32 (the reference's path); 1: mixed precision: FP16 block
                                   storage with per-block power-of-two scale in the PCG SpMV inside
                                   FP32 iterative refinement, FP64 CCD, distances and barrier;
                                   2: the same with BF16 block storage                          */
    int   use_energy_linesearch; /* 1: after the CCD bound, halve the step (at most 20 times) while
                                   the energy does not decrease (newton_solver.cpp:3803-3856)  */
    int   contact_energy_type;  /* 1: IPC log barrier (the reference's default); 0: quadratic
                                   penalty 1/2 kappa area C^2, C = thickness + d_hat - d
                                   (SceneParams::contact_energy_type, scene_params.h:89)        */
    int   post_dist_check;      /* 1 (default): after every frame, the smallest gap d - (offset_a +
                                   offset_b) over the candidate pairs at the final positions, in
                                   FP64, and the count of pairs at or below 0 (lcsx_stats.min_gap,
                                   num_penetrating; NewtonSolver::device_post_dist_check,
                                   newton_solver.cpp:3364-3375)                                 */
} lcsx_params;

/* Scalars of the last Newton iteration / frame. */
typedef struct lcsx_stats
{
    int   frame;
    int   newton_iters;       /* iterations of the last frame                               */
    int   pcg_iters;          /* PCG iterations of the last Newton iteration                */
    int   pcg_iters_total;    /* summed over the last frame                                 */
    float toi;                /* CCD step bound (alpha) of the last iteration, in (0, 1]    */
    float max_dx;             /* max vertex |dx| of the last iteration                      */
    float pin_delta;          /* max |x - x_tilde| over pinned vertices                     */
    float pcg_rel;            /* sqrt(r.z / r0.z0) at PCG exit                              */
    int   num_pairs_vf;       /* broad-phase candidates (DCD query of the last iteration)   */
    int   num_pairs_ee;
    int   num_contacts;       /* active barrier contacts                                    */
    int   converged;
    int   broadphase_overflow;/* a 32-entry traversal stack overflowed (reference: silent)  */
    double pcg_rz_true;       /* mixed precision: r.z of the last true residual (compensated
                                 sum), -1 when the last PCG replaced none                    */
    double min_gap;           /* post_dist_check: smallest d - (offset_a + offset_b) over the
                                 frame's final candidate pairs (FP64 distance), and y - floor -
                                 offset over free vertices with the floor on; +inf with none,
                                 NaN when the check did not run                               */
    int   num_penetrating;    /* post_dist_check: pairs / vertices with gap <= 0 (-1: not run) */
    int   gap_pairs;          /* post_dist_check: pairs and vertices checked (-1: not run)     */
    float toi_min;            /* smallest CCD step bound over the last frame's iterations     */
    int   num_ccd_pairs;      /* swept-box candidate pairs (VF + EE) of the last line search  */
} lcsx_stats;

/* ---------------------------------------------------------------- library */
const char* lcsx_last_error(void);
const char* lcsx_version(void);
/* Number of HIP devices visible (0 on a host without a GPU). */
int lcsx_device_count(void);

/* ------------------------------------------------------- NewtonSolver API */
/* Replaces NewtonSolver construction + lcs::get_scene_params() setup. params may be NULL
 * (reference defaults). device selects the HIP device (ordinal). */
lcsx_status lcsx_solver_create(const lcsx_params* params, int device, lcsx_solver** out);
lcsx_status lcsx_solver_destroy(lcsx_solver* s);
/* Default parameters (scene_params.h defaults; PCG stops on r.z < 1e-10 tested every 25 iterations). */
void lcsx_params_default(lcsx_params* p);
void lcsx_material_default(lcsx_material* m);

/* NewtonSolver::register_mesh (python_bindings.cpp:259) + WorldData material: world-space
 * vertices (n_verts x 3 floats) and triangles (n_tris x 3 int32). mesh_id receives the index. */
lcsx_status lcsx_solver_add_mesh(lcsx_solver* s, const float* verts, int n_verts, const int32_t* tris, int n_tris,
                                 const lcsx_material* material, int* mesh_id);
/* WorldData::load_fixed_points (init_mesh_data.cpp:117-240): method is a FixedPointsType value
 * (3 Left, 4 Right, 5 Front, 6 Back, 7 Up, 8 Down, 9..20 corner combinations, 21 All),
 * range in normalised mesh coordinates. anim may be NULL (static pins). */
lcsx_status lcsx_solver_add_fixed_points(lcsx_solver* s, int mesh_id, int method, float range,
                                         const lcsx_fixed_anim* anim, int* num_selected);
/* Demo::Simulation::load_scene_params_from_json (app_simulation_demo_config.cpp:49-766):
 * scene keys, shells with model_name (OBJ, resolved against mesh_dir), translation, rotation,
 * scale, Cloth material and fixed_points. */
lcsx_status lcsx_solver_load_scene_json(lcsx_solver* s, const char* json_path, const char* mesh_dir);
/* NewtonSolver::init_solver (newton_solver.h:31-51): topology, masses, CSR, device buffers. */
lcsx_status lcsx_solver_init(lcsx_solver* s);
/* physics_step_GPU (newton_solver.cpp:4051-4345) for `frames` frames, each preceded by the
 * pinned-target update of app_simulation.cpp:114-123 at time frame * dt. */
lcsx_status lcsx_solver_step(lcsx_solver* s, int frames);
/* NewtonSolver::get_simulation_results / SolverInterface::get_simulation_results_to_host. */
lcsx_status lcsx_solver_get_positions(lcsx_solver* s, float* out, size_t n_floats);
lcsx_status lcsx_solver_get_velocities(lcsx_solver* s, float* out, size_t n_floats);
/* SolverInterface state restore (load_state positions/velocities, solver_interface.cpp:291-412). */
lcsx_status lcsx_solver_set_state(lcsx_solver* s, const float* x, const float* v, size_t n_floats);
/* Checkpoints in the reference's ".state" text format (SolverInterface::
 * save_current_frame_state_to_host / load_saved_state_from_host, solver_interface.cpp:206-410):
 * "o position" and "o velocity" with one "v x y z" line per mesh vertex (registration order),
 * then "o q" and "o qv" with four lines per affine body (p, a0, a1, a2). Values are written with
 * 9 significant digits, so a save/load round trip is exact; files written by the reference (6
 * digits) load too. load_state with frame >= 0 also sets the frame counter that drives the
 * pinned-vertex animation; the file path is the caller's (the reference builds
 * "<resources>/SimulationState/frame_<n>.state"). */
lcsx_status lcsx_solver_save_state(lcsx_solver* s, const char* path);
lcsx_status lcsx_solver_load_state(lcsx_solver* s, const char* path, int frame);
/* The current positions as one OBJ file, an "o mesh_<i>" object per registered mesh with its
 * triangles (SimMesh::saveToOBJ_combined, mesh_reader.cpp:681-750). */
lcsx_status lcsx_solver_save_obj(lcsx_solver* s, const char* path);
/* SolverInterface::update_pinned_verts_information (solver_interface.h:95-108): explicit targets
 * for the pinned vertices of one mesh (in selection order), replacing the animation. */
lcsx_status lcsx_solver_set_pinned_targets(lcsx_solver* s, int mesh_id, const float* targets, int n_pinned);
lcsx_status lcsx_solver_get_stats(lcsx_solver* s, lcsx_stats* out);
int         lcsx_solver_num_verts(lcsx_solver* s);

/* ------------------------------------------------------- batched form
 * No counterpart in the reference (one scene per NewtonSolver): one solver handle steps a batch
 * of independent scenes together, every stage one launch over all of them. Meshes added (or
 * scene files loaded) after lcsx_solver_begin_scene belong to a new scene; meshes added before
 * the first call form scene 0. All scenes share the parameters (dt, stiffnesses, tolerances).
 * Each scene keeps its own LBVH (a segment of the shared forest), its own PCG scalars and
 * convergence test, its own CCD step bound and its own Newton loop; a scene whose loop has
 * stopped keeps its positions while the others iterate. Positions and velocities of all scenes
 * are concatenated in scene order; lcsx_solver_scene_range gives each scene's vertex range.
 * lcsx_solver_get_stats returns batch totals (iteration counts summed over scenes, the smallest
 * step bound, the largest |dx|); lcsx_solver_get_scene_stats one scene's. */
lcsx_status lcsx_solver_begin_scene(lcsx_solver* s, int* scene_id);
int         lcsx_solver_num_scenes(lcsx_solver* s);
lcsx_status lcsx_solver_scene_range(lcsx_solver* s, int scene, int* first_vertex, int* num_verts);
lcsx_status lcsx_solver_get_scene_stats(lcsx_solver* s, int scene, lcsx_stats* out);

/* ----------------------------------------------- per-stage entry points
 * The reference's subsystem methods, applied to the solver's own device buffers. Used for
 * parity checks and per-kernel measurement. stage is one of:
 *   "frame_begin"      pinned targets + LBVH::reduce_*_tree_aabb + LBVH::construct_tree (x2)
 *   "predict"          fn_predict_position (newton_solver.cpp:577-608)
 *   "iter_begin"       x_iter_start = x
 *   "material"         inertia, ground, stretch, bending evaluation + assembly (newton_solver.cpp:705-1172)
 *   "broad_phase_dcd"  LBVH::update_*_leave_aabb + refit + broad_phase_query_from_{verts,edges} on (x, x)
 *   "broad_phase_ccd"  the same on the swept boxes (x_iter_start, x)
 *   "dcd"              NarrowPhasesDetector::vf/ee_dcd_query_repulsion
 *   "update_contacts"  broad_phase_dcd + dcd
 *   "contact_assemble" device_perPair_evaluate_gradient_hessian (narrow_phase.cpp:2550-2676)
 *   "pcg"              ConjugateGradientSolver::device_solve (precond_cg.cpp:626-771)
 *   "ccd"              ground + VF + EE CCD on (x_iter_start, x) -> toi
 *   "line_search"      NewtonSolver::line_search (newton_solver.cpp:3685-3884), CCD variant
 *   "newton_iteration" one full iteration of the Newton loop
 *   "frame_end"        fn_update_velocity + frame counter
 *   "step"             one full frame
 *   "spmv_dx"          dx <- A dx (the system matrix applied to the dx buffer)
 *   "spmv_dx_lp"       the same with the mixed form's 16-bit off-diagonal blocks (FP32 blocks
 *                      when the solver runs in FP32)
 *   "post_dist_check"  NewtonSolver::device_post_dist_check (newton_solver.cpp:3364-3375): smallest
 *                      FP64 gap over the DCD candidates at x into lcsx_stats.min_gap / num_penetrating
 *   "shrink_lists"     pair and contact lists back to 1024 entries (the next iteration grows them
 *                      and redoes itself: exercises the growth path)
 */
lcsx_status lcsx_solver_run_stage(lcsx_solver* s, const char* stage);
/* Named solver buffers, converted to a canonical host layout: float arrays are FP32, index
 * arrays uint32, morton keys uint64, energies double. Off-diagonal blocks are returned in the reference's CSR slot
 * order (row-major 3x3 per block). count_out receives the element count; with out == NULL only
 * the count is reported. Names:
 *   state      x, v, x_step, x_iter, x_tilde, dx, cgB, diag, offdiag, toi
 *   setup      rest_x, faces, edges, hinges, csr, stretch_faces, bending_hinges, fixed_verts,
 *              is_fixed, face_area, edge_area, vert_area, vert_mass, offset, dhat, sf_Dm, sf_area,
 *              sf_mu, sf_lambda, bh_angle, bh_hbar, bh_k (readable after a failed init for want
 *              of a device, since the host setup is built first)
 *   trees      face_tree.* / edge_tree.* with morton, morton_sorted, sorted_to_orig, parent,
 *              children, object_idx, node_aabb
 *   contacts   pairs_vf, pairs_ee (last broad phase), contact_idx, contact_type, contact_n,
 *              contact_k (k1, k2, kappa * area), contact_w, contact_bary, contact_triplets /
 *              contact_triplet_blocks (the contact Hessian's off-diagonal blocks k2 w_i w_j n n^T
 *              of the current contact list, assembled on the GPU, sorted by (row, column) and summed
 *              per key: (row, column) uint32 pairs and 9 floats per block, row-major; the
 *              reference's device_sort_contact_triplet / device_assemble_contact_triplet,
 *              narrow_phase.cpp:1434-1758, 1883-2323), ccd_rest_vf /
 *              ccd_rest_ee (the last line search's candidate pairs whose ACCD ran past the first
 *              pass's iteration budget)
 *   energy     the total energy of each scene at the current x over the current contact list
 *              (double per scene; the energy line search's objective)
 * lcsx_solver_write accepts x, v, x_step, x_iter, x_tilde, dx and cgB. */
lcsx_status lcsx_solver_read(lcsx_solver* s, const char* name, void* out, size_t bytes, size_t* count_out);
lcsx_status lcsx_solver_write(lcsx_solver* s, const char* name, const void* in, size_t bytes);
/* Average device time (ms) of each kernel group over the calls since the last reset
 * (hipEvent timing on the solver's stream); entries are written as "name=ms,calls;..." into buf.
 * With timing on, three entries carry counts instead of times (average per Newton iteration):
 * "pairs_ccd" (swept-box candidates the line search's CCD processed), "pairs_dcd" (candidates the
 * DCD processed) and "contacts" (active contacts after the DCD). */
lcsx_status lcsx_solver_kernel_times(lcsx_solver* s, char* buf, size_t buf_len, int reset);
/* Timing level: 0 off, 1 stage groups (default), 2 also the device time of every 8th PCG SpMV
 * launch of a solve (events attached to the launch; reported as "spmv", only launches before
 * convergence are counted) and the contact slots those launches processed ("spmv_slots", slots
 * per launch); 3 as 2 for every SpMV launch. Each timed launch adds a few microseconds of gap
 * around it, which is why level 2 samples. */
lcsx_status lcsx_solver_set_timing(lcsx_solver* s, int level);
/* PCG launch mode (no counterpart in the reference, whose backend records its own command
 * lists). A solver on which neither this nor lcsx_solver_set_spmv_shape was called runs a solve as a
 * single launch where the system fits (lcsx_solver_set_one_launch), otherwise as three launches per
 * iteration. This call selects the launches: 1 captures each convergence-test interval of PCG iterations
 * as a hipGraph and replays it; 0 launches every kernel directly. Every form adds up the same terms in the
 * same order. On MI355X the replay does not shorten the device time of a solve (the gaps between
 * dependent kernels remain) and each new chunk shape costs a capture. Timing level 2 always launches
 * directly (its events are attached to the SpMV launches). */
lcsx_status lcsx_solver_set_graphs(lcsx_solver* s, int on);
/* The PCG in one launch (no counterpart in the reference). on 1, the default: a solve runs as a single
 * launch where the system fits (a scene of up to 131,072 rows of at most 12 blocks or 65,536 of at most 32,
 * a batch in up to two such launches, and contacts that are few beside the rows; rows of more than 16
 * blocks with contacts only in small scenes), whatever
 * lcsx_solver_set_graphs and lcsx_solver_set_spmv_shape say of the solves that do not; this takes back
 * their choice of the launches. 0: launches only. */
lcsx_status lcsx_solver_set_one_launch(lcsx_solver* s, int on);
/* LBVH traversal shape of the solver's broad-phase queries (no counterpart in the reference; the
 * same pairs in every shape). Binary steps (one 64 B record, two children tested per step, the
 * reference's 32-entry stack): 0 keeps the whole stack in LDS and stages 256 pairs per wavefront
 * before reserving output space; 1 keeps 16 stack entries in LDS (the rest in a global spill
 * area) and stages 512; 2: 16 and 1024; 3: 8 and 1024. 4-wide steps (one 128 B record of
 * the four grandchildren, about half the dependent steps; a 64-entry stack): 4: 16 in LDS and
 * 512; 5: 8 and 1024; 6: 32 and 512. 7 and 8: four lanes per query on the 128 B records (lane j
 * tests grandchild j, so a step's record is one contiguous load shared by the four lanes), 16 or
 * 32 stack entries in LDS, 512 pairs staged; 7 is the default. 9: two lanes per query on the 128 B
 * records (lane j tests grandchildren 2j and 2j + 1), 16 stack entries in LDS, 512 pairs staged
 * (faster where the queries fill the GPU, as in large batches). That is how a standalone tree is
 * queried; in a solver 7, 8 and 9 all walk its own hierarchies, 16 neighbouring queries per
 * wavefront, whose walks have no stack to overflow, or as shape 4 where those would be slow: scenes of
 * thousands of separate pieces, and batches of tiny scenes (lcsx_solver_read "cluster_use": faces, edges). */
lcsx_status lcsx_solver_set_query_shape(lcsx_solver* s, int shape);
/* Mapping of the PCG block SpMV (no counterpart in the reference; every shape gives the same
 * bits, the blocks of a row being added in the same order). 0: three blocks per lane and pass with
 * every load issued unconditionally (lanes past a row's width reread the pass's first block and
 * drop its product by a select); 1: three blocks per pass with loads predicated on the row's
 * width; 2: two blocks per pass, unconditional. 3-5: the same with the contact-slot chunks launched
 * before the row blocks (their dependent loads then overlap the row blocks' streaming); 3 is the
 * default. Selects the launched form of the PCG, as lcsx_solver_set_graphs does. */
lcsx_status lcsx_solver_set_spmv_shape(lcsx_solver* s, int shape);
/* Autotuner (no counterpart in the reference): times the runtime mappings on the current state
 * and keeps the fastest of each: the CCD first-pass iteration budget (8..128), the PCG launch
 * mode (direct or captured graphs), for a single scene the contact t_c kernel form (one thread
 * per contact or per 256-slot chunk), the PCG SpMV mapping (lcsx_solver_set_spmv_shape) and the
 * broad-phase traversal shape (lcsx_solver_set_query_shape; 7 to 9 are one in a solver); a setting
 * changes only for a candidate more than 3% faster than the current one. The PCG's settings are timed and
 * kept for the solves that run as launches; those that fit one launch still do. No choice changes a result.
 * The state (positions, velocities, statistics, timings) is restored. report (may be NULL) receives
 * "name[setting]=ms;...;chosen:..." (truncated to report_len). Best called after a few frames,
 * on a state with contacts. */
lcsx_status lcsx_solver_autotune(lcsx_solver* s, char* report, size_t report_len);

/* ----------------------------------------------- standalone LBVH (device pointers)
 * LBVH over faces (arity 3) or edges (arity 2), lbvh.h:166-304. All pointers are device
 * pointers on the solver-independent stream `stream` (a hipStream_t, NULL = default). The calls return
 * before the GPU is done: a tree's construction, refit and queries belong on one stream, or behind an
 * event or synchronisation of the caller's. A refit before the first construction and a query before the
 * first refit return LCSX_ERR_STATE. */
typedef struct lcsx_lbvh lcsx_lbvh;
lcsx_status lcsx_lbvh_create(int arity, const uint32_t* device_prims, int n_leaves, lcsx_lbvh** out);
lcsx_status lcsx_lbvh_destroy(lcsx_lbvh* t);
/* reduce_*_tree_aabb + construct_tree: n_verts_for_reduce reproduces the reference's
 * second-pass sizing (ceil(n/256) blocks of leaves enter the global box). */
lcsx_status lcsx_lbvh_construct(lcsx_lbvh* t, const float* device_x, int n_verts_for_reduce, void* stream);
/* update_*_leave_aabb + refit: leaf box of the element over x0 and x1, padded by pad[first vertex]. */
lcsx_status lcsx_lbvh_refit(lcsx_lbvh* t, const float* device_x0, const float* device_x1, const float* device_pad,
                            void* stream);
/* broad_phase_query_*: boxes are 6 floats (lo, hi) per query; edge_filter keeps query < leaf.
 * Pairs (query, leaf) are appended to device_pairs (2 uint32 each) up to capacity; the total
 * found is written to *device_count (uint32, device memory, must be zeroed by the caller). */
lcsx_status lcsx_lbvh_query(lcsx_lbvh* t, const float* device_boxes, int n_queries, int edge_filter,
                            uint32_t* device_pairs, uint32_t capacity, uint32_t* device_count, void* stream);
/* Traversal shape of lcsx_lbvh_query, as lcsx_solver_set_query_shape (no counterpart in the
 * reference; every shape finds the same pairs). */
lcsx_status lcsx_lbvh_set_query_shape(lcsx_lbvh* t, int shape);
/* Reads back tree arrays: "morton_sorted" (uint64), "sorted_to_orig", "parent", "children",
 * "object_idx" (uint32), "node_aabb" (6 floats per node), "global_aabb" (6 floats). */
lcsx_status lcsx_lbvh_read(lcsx_lbvh* t, const char* name, void* out, size_t bytes);

/* ----------------------------------------------- standalone block PCG (device pointers)
 * ConjugateGradientSolver::device_solve (Solver/LinearSolver/precond_cg.h:38-47,
 * precond_cg.cpp:626-771) on a caller's block system instead of the solver's own: the same
 * block-Jacobi PCG (x0 = 0, the reference's safe divisions and stopping test) with the SpMV
 * fixed to a block-CSR matrix, for a caller that assembles its own system (the reference passes
 * its SpMV as a function over its triplet arrays). All arrays are device arrays: row i's
 * off-diagonal blocks are [row_ptr[i], row_ptr[i + 1]) of col / blocks; blocks and diag hold 9
 * floats per 3x3 block, row-major; b and x hold 3 floats per row. The diagonal blocks are also the
 * preconditioner. A column outside [0, n_rows) or a row range outside [0, nnz) is rejected
 * (LCSX_ERR_ARG) without being read. */
typedef struct lcsx_bsr
{
    int            n_rows;
    int            nnz;      /* off-diagonal blocks */
    const int32_t* row_ptr;  /* n_rows + 1 */
    const int32_t* col;      /* nnz */
    const float*   blocks;   /* 9 * nnz */
    const float*   diag;     /* 9 * n_rows */
} lcsx_bsr;
typedef struct lcsx_pcg_options
{
    int   max_iters;   /* reference: pcg_iter_count (100)                                      */
    int   check_every; /* convergence test interval (reference: 25)                            */
    float rel_tol;     /* also stop when r.z <= rel_tol^2 r0.z0 (0: off, the reference)        */
    float abs_tol;     /* stop when r.z < abs_tol (reference: 1e-10)                           */
} lcsx_pcg_options;
typedef struct lcsx_pcg_result
{
    int   iters;      /* iterations run (the stopping one when the test stopped the solve)      */
    int   converged;  /* 1 when the test stopped the solve, 0 at the iteration cap              */
    float rz0, rz;    /* r.z at the start and at the last evaluated iteration                  */
} lcsx_pcg_result;
void lcsx_pcg_options_default(lcsx_pcg_options* o);
/* Solves A x = b on `stream` (a hipStream_t, NULL = default); allocates its scratch (about 128 B
 * per row) for the call and frees it before returning. */
lcsx_status lcsx_pcg_solve_bsr(const lcsx_bsr* A, const float* device_b, float* device_x,
                               const lcsx_pcg_options* options, void* stream, lcsx_pcg_result* result);
/* No counterpart in the reference: lcsx_pcg_solve_bsr for callers that cannot allocate device
 * memory (code under HIP graph capture, tight serving loops, harnesses that forbid hipMalloc). The
 * same solve with its scratch in a static device array of the library (one per GPU, about 17 MB,
 * held until the process ends) instead of an allocation; calls no hipMalloc or hipFree. At most
 * 131072 rows (LCSX_ERR_ARG above). Every call on one GPU shares that GPU's scratch: calls that
 * overlap on one GPU (other host threads, or other streams still running an earlier call) race. */
lcsx_status lcsx_pcg_solve_bsr_noalloc(const lcsx_bsr* A, const float* device_b, float* device_x,
                                       const lcsx_pcg_options* options, void* stream, lcsx_pcg_result* result);

/* device_SpMV (Solver/SimulationSolver/newton_solver.cpp:3397-3427: y = D x + sum of the
 * off-diagonal blocks times x) on a caller's block-CSR matrix: y = A x, with x and y 3 floats per
 * row on `stream`. Bad indices as in lcsx_pcg_solve_bsr. */
lcsx_status lcsx_spmv_bsr(const lcsx_bsr* A, const float* device_x, float* device_y, void* stream);

/* No counterpart in the reference: how many solves of this process on a device took which form
 * (lcsx_pcg_solve_bsr, its no-alloc form and the solvers'; all give the same bits). counts[0]: one launch,
 * to its end. counts[1]: began as one launch, but a row has more blocks, or 256 (512) rows name more others,
 * than it holds. counts[2]: began as one launch, but its workgroups did not all run at once (another process
 * on the GPU, a stream restricted to some CUs), found after about 0.14 s; the next 1024 solves on the device,
 * then 2048 and so on, take the launches at once. counts[3]: would have fitted, but another solve was
 * running in that form or it was such a next one. Solves of 1 to 3 ran as three launches per iteration, as
 * did the uncounted ones, which the form does not take by their size. */
lcsx_status lcsx_pcg_form_counts(int device, uint64_t counts[4]);

/* ConjugateGradientSolver::device_solve(stream, func_spmv, func_compute_energy) (precond_cg.h:41-43,
 * precond_cg.cpp:626-771) in its operator form: the caller supplies the product q = A p as a
 * function, the library runs the same block-Jacobi PCG around it (x0 = 0, the safe divisions, the
 * stopping test of lcsx_pcg_options). `spmv` is called once per iteration, on the calling thread,
 * with device arrays p and q (3 floats per row; p must not be written) and `stream`; it enqueues
 * its work on that stream (or completes it before returning). diag holds the 3x3 diagonal blocks
 * (9 floats per row, row-major), which are also the preconditioner. The reference's energy
 * function is used only by diagnostics that are commented out (precond_cg.cpp:518-521) and has no
 * counterpart. Scratch (about 84 B per row) is allocated for the call and freed before it returns. */
typedef void (*lcsx_spmv_fn)(void* user, const float* device_p, float* device_q, void* stream);
lcsx_status lcsx_pcg_solve_op(int n_rows, const float* device_diag, lcsx_spmv_fn spmv, void* user,
                              const float* device_b, float* device_x, const lcsx_pcg_options* options, void* stream,
                              lcsx_pcg_result* result);

/* ----------------------------------------------- standalone narrow phase (device pointers)
 * NarrowPhasesDetector's CCD and DCD queries (narrow_phase.h:54-201) on a caller's candidate list
 * and positions, for one scene without affine bodies. kind 0: vertex-face pairs (vertex, face) with
 * prims = 3 vertex ids per face; kind 1: edge-edge pairs (edge, edge) with prims = 2 per edge.
 * Positions are 3 floats per vertex, offset / dhat / areas one float per vertex (area_a, area_b:
 * vertex and face areas for kind 0, edge areas for kind 1). precision: 0 FP32, 1 or 2 the mixed
 * forms' FP64 (ACCD in double with its bound rounded down; DCD distances and barrier in double).
 * Both calls run on `stream` and return when it is done. */
/* vf_ccd_query / ee_ccd_query (narrow_phase.cpp:293-593): the CCD step bound, the smallest
 * ACCD time of impact / 1.25 over the pairs moving from x0 to x1 (1 when none collides), written
 * to device_toi[0]; pairs sharing a vertex are skipped. Scratch of 4 B per pair for the call. */
lcsx_status lcsx_ccd_pairs(int kind, const uint32_t* device_pairs, uint32_t n_pairs, const uint32_t* device_prims,
                           const float* device_x0, const float* device_x1, const float* device_offset, int precision,
                           float* device_toi, void* stream);
/* vf_dcd_query_repulsion / ee_dcd_query_repulsion (narrow_phase.cpp:771-1098): the pairs closer than
 * offset_a + offset_b + (dhat_a + dhat_b) / 2 at x become contacts, appended to the four arrays
 * (per contact: idx 4 uint32 with the pair type in bit 31 of entry 2 (VF) or 3 (EE); nk 4 floats:
 * normal and k2; w 4 floats: the weights; aux 4 floats: k1, kappa * mean area, two barycentrics)
 * up to capacity; *device_count (device memory, to be zeroed by the caller before a list starts)
 * receives the total found, so a count above capacity means the arrays were too small.
 * contact_energy_type: 1 IPC log barrier, 0 quadratic (lcsx_params). */
lcsx_status lcsx_dcd_pairs(int kind, const uint32_t* device_pairs, uint32_t n_pairs, const uint32_t* device_prims,
                           const float* device_x, const float* device_area_a, const float* device_area_b,
                           const float* device_offset, const float* device_dhat, float kappa, int contact_energy_type,
                           int precision, uint32_t* device_contact_idx, float* device_contact_nk,
                           float* device_contact_w, float* device_contact_aux, uint32_t capacity,
                           uint32_t* device_count, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* LCSX_H */
