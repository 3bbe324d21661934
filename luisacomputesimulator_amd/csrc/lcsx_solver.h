// The Newton solver context behind the C ABI (host side).
#pragma once
#include <map>
#include <string>
#include <tuple>
#include <vector>
#include "../../include/lcsx.h"
#include "lcsx_common.h"
#include "lcsx_internal.h"
#include "lcsx_kernels.h"
#include "lcsx_setup.h"

namespace lcsx
{

struct Solver
{
    lcsx_params           prm{};
    int                   device = 0;
    hipStream_t           stream = nullptr;
    hipStream_t           side   = nullptr;  // second stream (default priority) for overlapped passes
    hipEvent_t            ev_fork = nullptr, ev_join = nullptr;
    std::vector<MeshDesc> meshes;
    Setup                 S;
    bool                  inited = false;
    bool                  setup_ready = false;  // host setup built (readable without a GPU)
    int                   frame  = 0;
    lcsx_stats            stats{};

    // state (3 floats per vertex)
    DBuf<float> x, v, x_step, x_iter, x_tilde, dx, cgB, r, z, p[2], q, spmv_tmp;
    DBuf<float> diag, diag_mat, minv, sell_val;  // 9 planes (diag: with contact blocks; diag_mat: material only)
    DBuf<float> part_rz, part_pq;  // PCG per-block partial sums
    // mixed precision: FP16 off-diagonal blocks with a per-block exponent, and the compensated
    // (sum, error) partials of the replaced residual's r.z
    DBuf<uint32_t> sell_p;  // packed 16-bit blocks of the mixed-precision SpMV (5 planes)
    DBuf<float>  part_res;
    double       rz_true = 0.0;  // r.z of the last replaced residual (compensated, summed in double)
    // constants
    DBuf<float>    rest_x, offset, dhat, vert_mass, vert_area, face_area, edge_area, targets;
    DBuf<uint8_t>  is_fixed;
    DBuf<uint32_t> faces, edges, sf, bh, v_sf_ptr, v_sf, v_bh_ptr, v_bh, sl_off, sell_col, blk_ptr, blk_contrib, fixed_ids;
    DBuf<uint32_t> sp, v_sp_ptr, v_sp;
    DBuf<float4>   sf_Dm, sf_c, bh_c;
    DBuf<float2>   sp_c;
    DBuf<float>    face_stage, hinge_stage, spring_stage;
    Lbvh           tree_face, tree_edge;
    bool           sorted_ee = false;  // edge-edge candidates by the sorted self-query
    ClusterTree    cluster_face, cluster_edge;
    DBuf<uint32_t> cluster_vert;  // points in the order of their queries
    uint32_t       n_cluster_vert = 0;
    ClusterQuery   cluster_query(const float* x0) const;
    // collision buffers
    DBuf<uint32_t> pairs_vf, pairs_ee;
    uint32_t       cap_vf = 0, cap_ee = 0, cap_c = 0;
    DBuf<uint4>    c_idx;
    DBuf<float4>   c_nk, c_w, c_aux;
    DBuf<uint32_t> vc_cnt, vc_ptr, vc_list, vc_row;  // per-row contact slots (rebuilt with each contact assembly)
    DBuf<uint4>    c_gr;                              // generalized DOFs of the contacts (2 per contact)
    DBuf<float4>   c_gw;
    // affine bodies
    DBuf<BodyDev>  bodies_d;
    DBuf<uint8_t>  row_kind_d;
    DBuf<uint32_t> vert_body_d;
    DBuf<float>    body_X_d;
    uint32_t       slots_per_contact = 4;  // 8 with affine bodies (a rigid side has four rows)
    DBuf<float4>   vc_coef;                          // per slot
    DBuf<float>    vc_tc;                    // per contact
    DBuf<float4>   vc_runsum;                // per slot: sums of the SpMV's slot runs
    DBuf<uint32_t> ccd_rest_vf, ccd_rest_ee, ccd_rest_count;  // CCD pairs left for the full-budget pass
    bool           vc_ready = false;
    bool           ccd_pairs_fresh = false;  // pairs_* hold the last line search's swept candidates
    bool           dcd_reused      = false;  // the last DCD ran on them
    DBuf<Status>   status;
    DBuf<GapStatus> gap;  // per scene: post-step distance check
    DBuf<PcgState> pcg_state;  // per scene
    Status         host_status{};
    // batch of scenes: segmentation tables (lcsx_kernels.h SegView), the Newton loops' active
    // mask, per-scene line-search results and statistics
    DBuf<uint32_t>           sc_v0_d, sc_rb0_d, rb_scene_d, rb_row0_d, vert_scene_d, sc_cb0_d, sc_cb0_zero,
                             cb_scene_d, cb_slot0_d;
    DBuf<uint8_t>            active_d;
    std::vector<uint8_t>     active_h;
    DBuf<SceneStatus>        sst;
    std::vector<SceneStatus> host_sst;
    std::vector<PcgState>    host_pcg;
    std::vector<lcsx_stats>  scene_stats;
    std::vector<uint32_t>    verts_per_scene;
    int            last_bp = 0;  // 0 none, 1 DCD, 2 CCD
    int            pcg_parity = 0;
    std::vector<float> explicit_targets;  // per fixed vertex (3), when set
    std::vector<uint8_t> has_explicit;     // per mesh

    // timing
    bool                         timing = true;
    std::map<std::string, std::pair<double, int>> times;
    hipEvent_t                   ev[2] = {nullptr, nullptr};

    ~Solver();
    void init();
    void upload_state_constants();
    void alloc_collision(uint32_t vf, uint32_t ee, uint32_t nc);

    // stages
    void frame_begin();
    void predict();
    void iter_begin();
    void material();
    void broad_phase(bool ccd);
    void query_faces(bool ccd);  // vertex-triangle candidates (refit of the face tree + query)
    void query_edges(bool ccd);  // edge-edge candidates
    void dcd(bool from_ccd_pairs = false);
    void update_contacts(bool reuse_ccd_pairs = false);
    void contact_assemble();
    void pcg();
    void ccd();
    void ccd_ground();
    void ccd_pass(int kind, bool rest, hipStream_t s);
    void swept_ccd();  // the line search's broad phase + CCD with the VF rest pass on `side`
    void line_search();
    std::vector<double> energy();  // per scene
    void                energy_line_search();
    DBuf<double>        energy_d;
    bool newton_iteration();  // returns false if it must be redone (buffer growth)
    void frame_end();
    void post_dist_check();  // smallest FP64 gap over the final candidate pairs (stats min_gap)
    // newton_iteration until it completes; a redo follows a buffer growth, which cannot repeat
    // more than a few times from one state
    void newton_iteration_until_done();
    void step();
    void spmv_dx(bool lp = false);  // lp: the mixed form's 16-bit blocks
    void rigid_positions();  // x of the rigid vertices from their bodies' rows
    void read_status();
    bool grow_if_needed(bool ccd_only);

    ContactView contact_view() const;
    ContactTripletBufs ctb;  // contact-triplet assembly on demand (not used by the Newton loop)
    // The current contact list's off-diagonal Hessian blocks, sorted and summed per (row, column)
    // into ctb.out_rc / ctb.out_blk; returns their count.
    uint32_t    contact_triplets();
    SegView     seg_view(bool with_chunks) const;  // with_chunks: the contact-slot chunk tables
    unsigned    max_chunks(uint32_t nslots) const { return nslots / 256u + S.nscenes; }
    void        fold_stats();                       // per-scene statistics into stats
    SellView    sell_view() const;
    SellView    sell_view_lp() const;  // FP16 blocks (mixed precision)
    // PCG iterations on a.b from x = 0, at most max_iters; with replace_every > 0 the recursive
    // residual is replaced by the true one (FP32 blocks) after every replace_every iterations.
    // Returns the iterations run.
    int         pcg_run(PcgArgs& a, const SellView& A, const ContactView& cv, const VertContacts& vc, int max_iters,
                        int replace_every, bool one_launch = true);
    void        account_spmv(uint32_t iters, uint32_t nslots);
    VertContacts vert_contacts();
    unsigned    pair_grid(uint32_t cap) const;

    // timing helpers
    void tic();
    void toc(const char* name);
    void toc_part(const char* name);  // adds to the name's current call (closed by a toc)
    void       flush_events();
    hipEvent_t ev_get();
    void       ev_put(hipEvent_t e);
    // measurement mode: a hipEvent pair attached to every spmv_sample-th PCG SpMV launch of a solve
    // (0: none, 1: every launch); each pair adds a few microseconds between the launches it brackets
    int spmv_sample = 0;
    static constexpr int kSpmvSample = 8;  // timing level 2: every 8th launch
    struct SpmvEvent
    {
        uint32_t   k;  // PCG iteration of the launch
        hipEvent_t e0, e1;
    };
    std::vector<SpmvEvent> spmv_events;

    // PCG chunks captured as hipGraphs and replayed (one graph launch per convergence-test interval
    // instead of three kernel launches per iteration), when enabled. A graph bakes in its kernels'
    // arguments: the key holds what varies between chunks, and graph_epoch changes with every
    // (re)allocation of a buffer the captured launches name. Not used while SpMV launches are timed.
    struct GraphKey
    {
        uint64_t epoch;
        int      k0, len, par;
        unsigned grid;
        int      contacts, lp, per_contact, spmv;
        bool     operator<(const GraphKey& o) const
        {
            return std::tie(epoch, k0, len, par, grid, contacts, lp, per_contact, spmv) <
                   std::tie(o.epoch, o.k0, o.len, o.par, o.grid, o.contacts, o.lp, o.per_contact, o.spmv);
        }
    };
    std::map<GraphKey, hipGraphExec_t> pcg_graphs;
    uint64_t graph_epoch = 0;
    bool     use_graphs  = false;
    // PCG in one launch (lcsx_pcg_grid.h), the default where it fits; off while the caller chooses
    // the form of the launches (set_graphs, set_spmv_shape, set_one_launch) or times them
    bool                     pcg_grid = true;
    bool                     grid_withhold = false;  // exercises a wait that runs out: a workgroup is not launched
    GridPlan                 grid_shape;      // U 0: the rows or scenes do not fit
    uint32_t                 grid_most = 0;   // row blocks of the largest scene
    std::vector<uint32_t>    grid_round;      // workgroups of round r: [grid_round[r], grid_round[r + 1])
    DBuf<uint2>              grid_tab;        // per workgroup: scene, place in it (several scenes)
    DBuf<unsigned long long> grid_slots, grid_zx;
    uint32_t                 grid_epoch = 0;
    void                     plan_grid();
    // runtime mappings chosen by autotune() (defaults: the measured best on the 88K-vertex tube)
    // ACCD iterations per pair in the first CCD pass; pairs that need more run again in a second
    // pass over a compact list, so long iterations do not hold whole wavefronts
    int         ccd_budget            = 32;
    bool        contact_t_per_contact = true;  // one scene: t_c by one thread per contact
    int         query_variant         = kQueryDefault;  // LBVH traversal shape (lbvh_query)
    int         spmv_shape            = kSpmvShapeDefault;  // PCG SpMV mapping (launch_pcg_spmv)
    std::string autotune();
    void     clear_graphs();
    void     enqueue_pcg_chunk(const PcgArgs& a, const SellView& A, const ContactView& cv, const VertContacts& vc,
                               unsigned mc, int k0, int len, int par);
};

}  // namespace lcsx
