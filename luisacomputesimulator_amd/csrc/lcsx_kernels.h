// Kernel argument structs and launchers of lcsx_kernels.hip.
#pragma once
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "lcsx_internal.h"

namespace lcsx
{

// Per-iteration status counters, zeroed by launch_reset_status.
struct Status
{
    uint32_t n_vf, n_ee, n_contacts, overflow;  // broad-phase counts, contacts, stack overflow flag
    uint32_t nan;
    uint32_t n_vf_ccd, n_ee_ccd, pad0;
};
// Line-search results of one scene of the batch.
struct SceneStatus
{
    uint32_t toi_bits;    // ordered key (f2ord) of the step bound
    uint32_t maxdx_bits;  // float bits of max |dx|
    uint32_t pin_bits;    // float bits of max pinned |x - x_tilde|
    uint32_t pad;
};

// Scenes of a batch. Vertices of scene s are [sc_v0[s], sc_v0[s+1]); row blocks of 256 rows
// never straddle two scenes (block b: scene rb_scene[b], first row rb_row0[b]; scene s owns
// blocks [sc_rb0[s], sc_rb0[s+1])), and neither do the 256-slot chunks of the contact slots
// (chunk c: scene cb_scene[c], first slot cb_slot0[c]; scene s owns [sc_cb0[s], sc_cb0[s+1])),
// so every per-block partial sum belongs to one scene. One scene: the trivial tables.
struct SegView
{
    uint32_t        nscenes, n_rb;
    const uint32_t* sc_v0;
    const uint32_t* sc_rb0;
    const uint32_t* rb_scene;
    const uint32_t* rb_row0;
    const uint32_t* vert_scene;
    const uint8_t*  active;  // per scene: 1 while its Newton loop runs
    const uint32_t* sc_cb0;
    const uint32_t* cb_scene;
    const uint32_t* cb_slot0;
};

// PCG scalars shared between launches. r.z of iteration k is stored in rz[k & 1] by the SpMV of
// iteration k; converged / iters / nan are set when an iteration's convergence test stops.
struct PcgState
{
    float    rz[2], rz0;
    uint32_t converged, iters, nan;
    uint32_t bad_index;  // block-CSR solves: a column or row range lies outside the matrix
    uint32_t fail;       // the one-launch form gave up (kGridUnfit, kGridWaited); the solve starts over
};

// SELL-16 block matrix: rows in slices of 16; slice s stores sl_off[s + 1] - sl_off[s] block
// columns, block k of row l at (sl_off[s] + k) * 16 + l. Entries in 9 planes (plane c = entry c of
// the row-major 3x3 block) so a wavefront's load of one entry over 64 blocks is contiguous.
constexpr uint32_t kSellH = 16;
struct SellView
{
    const uint32_t* sl_off;
    const uint32_t* col;
    const float*    val;   // 9 planes of nblocks
    const float*    diag;  // 9 planes of n
    uint32_t        nblocks;
    // mixed precision: 5 planes of nblocks 32-bit words per block: words 0..3 hold the 16-bit
    // entries (2c, 2c + 1) of the block scaled by 2^-e, word 4 entry 8 in its low half and the
    // signed exponent e in bits 16..23 (kKeepFp32: the block is read from val)
    const uint32_t* val_p;
    int             bf16;  // the 16-bit entries are BF16 bit patterns instead of FP16
};

// Exponent of a block that stays FP32 in the mixed-precision SpMV (packed exponents lie in [-100, 100]).
constexpr int8_t kKeepFp32 = -128;

struct ContactView
{
    const uint4*    idx;
    const float4*   nk;
    const float4*   w;
    const float4*   aux;
    const uint32_t* count;
    uint32_t        capacity;
    // generalized DOFs, two entries per contact: up to 8 rows (~0u: unused) and their weights (a
    // soft vertex with its weight, a rigid side as its body's 4 rows with weights sum w (1, X));
    // null without bodies: the contact's own vertices and weights
    const uint4*    gr;
    const float4*   gw;
};
// Per-row contact lists: entries list[ptr[i] .. ptr[i+1]) are (contact << 3 | entry), entry one of
// the contact's generalized DOFs; ptr null means no contacts.
struct VertContacts
{
    const uint32_t* ptr;
    const uint32_t* list;
    const uint32_t* row;     // per slot: its row
    const float4*   coef;    // per slot: (k2 w_j n, contact id bits)
    float*          tc;      // per contact: sum_j w_j n.p_j of the vector being multiplied
    uint32_t        nslots;  // an upper bound of the slots (sizes grids)
    const uint32_t* total;   // the number of slots (ptr[rows])
    // per slot, written at the last slot of each run (a row's slots within one wavefront of 64):
    // the run's sum, folded into its row in slot order by fold_runs
    float4*         runsum = nullptr;
};
struct ContactBuf
{
    uint4*    idx;
    float4*   nk;
    float4*   w;
    float4*   aux;
    uint32_t* count;
    uint32_t  capacity;
};

struct VertArgs
{
    uint32_t        nv;
    const uint8_t*  row_kind;  // 0 soft vertex, 1 rigid vertex (identity row), 2+ body row
    const float*    x;
    const float*    x_tilde;
    const float*    mass;
    const uint8_t*  fixed;
    const float*    area;
    const float*    offset;
    const float*    dhat;
    float           h2inv, kD, kappa, floor_y;
    int             use_floor;
    int             quadratic;  // contact energy form: 1 quadratic penalty, 0 log barrier
    const uint32_t* v_sf_ptr;
    const uint32_t* v_sf;
    const uint32_t* v_bh_ptr;
    const uint32_t* v_bh;
    const uint32_t* v_sp_ptr;
    const uint32_t* v_sp;
    const float*    spring_stage;
    const float*    face_stage;
    const float*    hinge_stage;
    float*          cgB;
    float*          diag;
    float*          diag_mat;  // optional copy of the material diagonal (the SpMV's; contacts go to diag only)
};

struct DcdArgs
{
    const uint32_t* pairs;
    const uint32_t* pair_count;
    uint32_t        pair_capacity;
    const float*    x;
    const uint32_t* faces;
    const uint32_t* edges;
    const float*    area_a;  // VF: vertex areas, EE: edge areas
    const float*    area_b;  // VF: face areas,   EE: edge areas
    const float*    offset;
    const float*    dhat;
    float           kappa;
    int             fp64;  // mixed-precision mode: distances and barrier in double
    int             quadratic;  // contact energy form: 1 quadratic penalty, 0 log barrier
    ContactBuf      out;
    const uint32_t* vert_body;  // per row: body id or ~0u; pairs within one body are skipped (null: no bodies)
};

struct CcdArgs
{
    int             kind;  // 0 VF, 1 EE
    const uint32_t* pairs;
    const uint32_t* pair_count;
    uint32_t        pair_capacity;
    const float*    x0;
    const float*    x1;
    const uint32_t* faces;
    const uint32_t* edges;
    const float*    offset;
    uint32_t*       toi_bits;
    // two passes: the first runs every pair with an iteration budget and lists the pairs that
    // need more; the second (rest = 1) runs the listed pairs with the full budget
    int             budget;
    int             rest;
    int             fp64;  // mixed-precision mode: ACCD in double, step bound rounded down to FP32
    uint32_t*       rest_list;   // capacity pair_capacity
    uint32_t*       rest_count;
    SceneStatus*    sst;         // step bound per scene (scene of the pair's first vertex)
    const uint32_t* vert_scene;  // null: one scene
    const uint32_t* vert_body;   // per row: body id or ~0u; pairs within one body are skipped (null: no bodies)
};

// Post-step distance check (NewtonSolver::device_post_dist_check, newton_solver.cpp:3364-3375,
// which runs the DCD and reports a pair closer than its offsets): per scene, the smallest gap
// d - (offset_a + offset_b) over the candidate pairs with the distance in FP64 (the DCD's
// unclassified barycentrics), the ground gap y - floor - offset of the free vertices, and the
// number of pairs / vertices at or below 0.
struct GapStatus
{
    unsigned long long min_key;    // order-preserving key (d2ord) of the smallest gap
    uint32_t           n_pen;      // pairs or vertices with gap <= 0
    uint32_t           n_checked;  // pairs and vertices tested
};
struct GapArgs
{
    int             kind;  // 0 VF pairs, 1 EE pairs, 2 ground (vertex rows)
    const uint32_t* pairs;
    const uint32_t* pair_count;
    uint32_t        pair_capacity;
    uint32_t        nv;  // kind 2: rows
    const float*    x;
    const uint32_t* faces;
    const uint32_t* edges;
    const float*    offset;
    const uint32_t* vert_scene;
    const uint32_t* vert_body;  // pairs within one body are skipped, as in the DCD
    const uint8_t*  fixed;
    const uint8_t*  row_kind;
    float           floor_y;
    GapStatus*      out;  // per scene
};

struct BodyDev;
// Energy line search: the total energy per scene (sums in double).
struct EnergyArgs
{
    uint32_t        nv;  // rows
    const float*    x;
    const float*    x_tilde;
    const float*    mass;
    const uint8_t*  fixed;
    const uint8_t*  row_kind;
    const uint32_t* vert_scene;
    const float*    offset;
    const float*    dhat;
    const float*    vert_area;
    float           h2inv, kD, kappa, floor_y, scaling;
    int             use_floor, fp64;
    int             quadratic;  // contact energy form: 1 quadratic penalty, 0 log barrier
    uint32_t        nsf, nbh, nb, nsp;
    const uint32_t* sp;
    const float2*   sp_c;   // rest length, stiffness
    const uint32_t* sf;
    const float4*   sf_Dm;
    const float4*   sf_c;   // area, mu, lambda
    const uint32_t* bh;
    const float4*   bh_c;   // rest angle, h_bar, stiffness
    const BodyDev*  bodies;
    ContactView     c;
    double*         out;    // per scene, accumulated
};

struct LsArgs
{
    uint32_t       nv;
    const float*   x_iter;
    const float*   x;
    const float*   dx;
    const uint8_t* fixed;
    const float*   offset;
    float          floor_y;
    int            use_floor;
    Status*        st;
    SceneStatus*   sst;
    SegView        seg;  // launched over the scene-aligned row blocks
    const uint8_t* row_kind;  // body rows (kind >= 2) have no ground test
};

// Affine bodies (one per rigid mesh): rows row0 .. row0 + 3 hold q = (p, a0, a1, a2), vertices
// [v0, v1) follow x = p + A X (X: body_X). Same layout as the host setup's body record.
struct BodyDev
{
    uint32_t row0, v0, v1, fixed;
    float    stiff;    // kappa * volume
    float    M[16];    // mass matrix (times I3)
    uint32_t blk[12];  // SELL blocks (ii, jj != ii), row-major
};
struct AbdArgs
{
    uint32_t       nb, n_rows, nblocks;
    const BodyDev* bodies;
    const float*   x;
    const float*   x_tilde;
    const float*   body_X;
    const uint8_t* fixed;
    const float*   offset;
    const float*   dhat;
    const float*   area;
    float          h2inv, kD, kappa, floor_y;
    int            use_floor;
    int            quadratic;  // contact energy form: 1 quadratic penalty, 0 log barrier
    float*         cgB;
    float*         diag;
    float*         diag_mat;
    float*         sell_val;
};

struct PcgArgs
{
    uint32_t     n;
    const float* b;
    const float* diag;
    float*       minv;
    float*       x;
    float*       r;
    float*       z;
    float*       p_old;    // 4 floats per row
    float*       p_new;    // 4 floats per row
    float*       q;
    // contact part of q: per-run sums of the slots (VertContacts::runsum) and the slot offsets,
    // null without contacts
    const float4*   runsum;
    const uint32_t* vc_ptr;
    float*       part_rz;  // per row block: r.z partial of init / update
    float*       part_pq;  // p.q partials of the SpMV: row blocks, then contact-slot chunks
    SegView      seg;
    PcgState*    s;        // per scene
    float        rel2, abs_tol;
    uint32_t     check_every;
    uint32_t     k;  // iteration index of the launch
};

void launch_fill_u32(uint32_t* a, uint32_t n, uint32_t v, hipStream_t s);
void launch_pin_velocity(uint32_t nfix, const uint32_t* ids, const float* targets, const float* x, float* v, float dt,
                         hipStream_t s);
void launch_predict(uint32_t nv, const float* x_step, const float* v, const uint8_t* fixed, const uint8_t* row_kind,
                    float h, const float g[3], float* x_iter, float* x_tilde, float* x, hipStream_t s);
// Affine-body inertia, orthogonality and lifted ground terms into cgB, diag and the body rows'
// SELL blocks (after launch_offdiag).
void launch_abd_material(const AbdArgs& a, hipStream_t s);
// x of every rigid vertex from its body's q.
void launch_rigid_positions(uint32_t n_rows, const uint8_t* row_kind, const uint32_t* vert_body, const BodyDev* bodies,
                            const float* body_X, float* x, hipStream_t s);
// Generalized DOF lists of the contacts (after the DCD).
void launch_contact_lift(const ContactView& c, unsigned grid, const uint32_t* vert_body, const BodyDev* bodies,
                         const float* body_X, uint4* gr, float4* gw, hipStream_t s);
void launch_frame_end(uint32_t nv, float* x_step, const float* x, float* v, float h, float damp, hipStream_t s);
void launch_face_stage(uint32_t nsf, const uint32_t* sf, const float4* Dm, const float4* c, const float* x, float* stage,
                       hipStream_t s);
void launch_hinge_stage(uint32_t nbh, const uint32_t* bh, const float4* c, float scaling, const float* x, float* stage,
                        hipStream_t s);
void launch_vert_assemble(const VertArgs& a, hipStream_t s);
void launch_spring_stage(uint32_t nsp, const uint32_t* sp, const float2* c, const float* x, float* stage, hipStream_t s);
void launch_offdiag(uint32_t nblocks, const uint32_t* ptr, const uint32_t* con, const float* ss, const float* fs, const float* hs, float* val,
                    hipStream_t s);
void launch_dcd(const DcdArgs& a, int kind, unsigned grid, hipStream_t s);
// Per-vertex contact lists (cnt: nv + 1 scratch counters, ptr: nv + 1, list: 4 per contact), and
// the scene-aligned 256-slot chunks of the slot list (sc_cb0: nscenes + 1, cb_scene / cb_slot0:
// up to slots / 256 + nscenes entries).
// tmp: one word per slot (scratch of the slot ordering)
void launch_contact_adjacency(const ContactView& c, uint32_t nv, unsigned grid, uint32_t* cnt, uint32_t* ptr,
                              uint32_t* list, uint32_t* row, float4* coef, uint32_t* tmp, const SegView& g,
                              uint32_t* sc_cb0, uint32_t* cb_scene, uint32_t* cb_slot0, bool repeats,
                              hipStream_t s);
// Scratch of the contact-triplet assembly (grown on demand; not used by the Newton loop).
struct ContactTripletBufs
{
    DBuf<uint32_t> cnt_b, ptr_b, scan_b, scan2_b, row_b[2], col_b[2], idx_b[2], head_b, pos_b, hist_b, sort_b, out_rc;
    DBuf<float>    blk_b, out_blk;
    uint32_t *     cnt = nullptr, *ptr = nullptr, *scan_tmp = nullptr, *scan_tmp2 = nullptr, *row[2] = {}, *col[2] = {},
             *idx[2] = {}, *head = nullptr, *pos = nullptr, *hist = nullptr, *sort_tmp = nullptr;
    float*         blk = nullptr;
    // per-contact arrays for n contacts
    void contacts(uint32_t n)
    {
        cnt_b.alloc(n + 1);
        ptr_b.alloc(n + 1);
        scan_b.alloc(scan_tmp_words(n + 1));
        cnt = cnt_b.p;
        ptr = ptr_b.p;
        scan_tmp = scan_b.p;
    }
    // per-triplet arrays for t triplets
    void reserve(uint32_t t, hipStream_t)
    {
        for (int k = 0; k < 2; k++)
        {
            row_b[k].alloc(t);
            col_b[k].alloc(t);
            idx_b[k].alloc(t);
            row[k] = row_b[k].p;
            col[k] = col_b[k].p;
            idx[k] = idx_b[k].p;
        }
        head_b.alloc(t);
        pos_b.alloc(t + 1);
        scan2_b.alloc(scan_tmp_words(t));
        hist_b.alloc(sort_hist_words(t));
        sort_b.alloc(scan_tmp_words(sort_hist_words(t)));
        blk_b.alloc(9 * (size_t)t);
        head = head_b.p;
        pos = pos_b.p;
        scan_tmp2 = scan2_b.p;
        hist = hist_b.p;
        sort_tmp = sort_b.p;
        blk = blk_b.p;
    }
};
// The contact Hessian's off-diagonal blocks, sorted by (row, column) and summed per key, into
// b.out_rc (row, column pairs) and b.out_blk (9 floats each, row-major); returns their count.
// Reads the contact count back (two host synchronisations).
uint32_t launch_contact_triplets(const ContactView& c, uint32_t n_contacts, unsigned grid, ContactTripletBufs& b,
                                 hipStream_t s);
void launch_contact_assemble(const ContactView& c, const VertContacts& vc, float* cgB, float* diag, uint32_t nv,
                             hipStream_t s);
void launch_pcg_init(const PcgArgs& a, hipStream_t s);
// One PCG iteration = three launches: the direction (r.z, convergence test, beta, p = z + beta p
// stored once, t_c per contact), the SpMV (q = A p from the stored p: material blocks and contact
// slots, p.q), then the update (alpha, x, r, z, r.z). With start/stop events the SpMV is launched
// with hipExtLaunchKernelGGL, which timestamps the kernel's own execution. The p buffers hold 4
// floats per row. max_chunks: an upper bound of the contact-slot chunks (slots / 256 + scenes);
// blocks past the actual count return at once.
void launch_pcg_dir(const PcgArgs& a, const ContactView& c, const VertContacts& vc, unsigned max_chunks,
                    bool per_contact, hipStream_t s);
// shape: the SpMV mapping (0 .. kSpmvShapes - 1): shape % 3 selects three blocks per pass with
// unconditional loads (0), three with loads predicated on the row's width (1) or two with
// unconditional loads (2); shapes 3-5 launch the contact chunks before the row blocks, 0-2 after
// them. Every shape gives the same bits.
constexpr int kSpmvShapes       = 6;
constexpr int kSpmvShapeDefault = 3;
void launch_pcg_spmv(const PcgArgs& a, const SellView& A, const VertContacts& vc, unsigned max_chunks, int shape,
                     hipStream_t s, hipEvent_t start = nullptr, hipEvent_t stop = nullptr);
void launch_pcg_update(const PcgArgs& a, hipStream_t s);

// The PCG in one launch (lcsx_pcg_grid.h): limits, shape and workspace.
constexpr uint32_t kGridRows    = 4096;  // rows whose p a workgroup holds: its own and those its columns name
constexpr uint32_t kGridOwn     = 512;   // own rows of a workgroup
constexpr uint32_t kGridWgs     = 256;   // most workgroups of a launch: one per CU of the GPU (grid_wgs)
constexpr uint32_t kGridThreads = 512;
// Why a launch gave up: a row has more blocks, or a workgroup names more rows, than the shape holds; or a
// wait ran out.
constexpr uint32_t kGridUnfit = 1, kGridWaited = 2;
struct GridSync
{
    unsigned long long* rz;    // words, zero before the first launch: one per row block,
    unsigned long long* pq;    // four per row block and one per contact-slot chunk,
    unsigned long long* zx;    // and three per row: z as it is exchanged
    const uint2*        tab;   // per workgroup: its scene and its place in it (null: one scene)
    uint32_t            epoch; // of the launch's first iteration (from 2); later launches use later ones
};
struct GridPlan
{
    int U = 0, K = 0;  // row groups per thread and blocks per thread and row (0: the launches are used)
    uint32_t row_blocks() const { return (uint32_t)U * kGridThreads / 1024u; }  // of a workgroup
};
// Workgroups that a launch may have on a device: its CUs, at most kGridWgs (0: none, as with no device).
uint32_t grid_wgs(int device);
// The shape for scenes of up to n_rb_most row blocks, n_rb in all, of at most `width` blocks a row, in
// launches of up to `wgs` workgroups.
GridPlan grid_plan(uint32_t n_rb_most, uint32_t n_rb, uint32_t width, uint32_t wgs);
// Iterations [a.k, a.k + len) of a solve begun by launch_pcg_init, on `wgs` workgroups.
void launch_pcg_grid(const GridPlan& p, unsigned wgs, const PcgArgs& a, const SellView& A, const ContactView& c,
                     const VertContacts& vc, const GridSync& g, uint32_t len, hipStream_t s);
void launch_grid_clear(unsigned long long* words, size_t n, hipStream_t s);
// One such launch runs at a time per GPU in a process (its workgroups wait for each other, so all
// must be resident); without the lease a solve uses the launches, which give the same bits. Where a wait has
// run out (another process holds CUs of the GPU, or the stream may use some of them only) the next solves on
// that GPU get no lease: 1024 of them, and twice as many after every further wait, since a wait that runs out
// costs about 0.14 s, as much as a hundred solves.
struct GridLease
{
    int  dev = -1;
    bool take(int device);
    void outcome(uint32_t fail, bool remember = true);  // of the solve (0: it ran to its end)
    ~GridLease();
};
// Solves of a device since the process began: in one launch, given up as unfit, given up on a wait, and
// refused a lease.
struct GridCounts
{
    uint64_t one, unfit, waited, refused;
};
GridCounts grid_counts(int device);
// Mixed precision: FP16 copy of the off-diagonal blocks with a power-of-two scale per block.
void launch_energy(const EnergyArgs& a, unsigned contact_grid, uint32_t nscenes, hipStream_t s);
void launch_pack_fp16(uint32_t nslices, uint32_t n, const uint32_t* sl_off, uint32_t nblocks, const float* val,
                      const uint8_t* row_kind, uint32_t* val_p, int bf16, hipStream_t s);
// Residual replacement: r = b - y, z = Minv r, per-block r.z with TwoSum compensation into
// part_rz[block] (sum + error) and part_res[2 block] (sum, error).
void launch_residual(const SegView& g, const float* b, const float* y, const float* minv, float* r, float* z,
                     float* part_rz, float* part_res, hipStream_t s);
// y = A p (diagonal + material blocks + contacts), for the spmv stage
void launch_spmv(const SellView& A, const ContactView& c, const VertContacts& vc, unsigned contact_grid, const float* p,
                 float* y, uint32_t n, hipStream_t s);
// x = x_iter + alpha dx with alpha the step bound of the vertex's scene (sst) or alpha_const
// (sst null); vertices of scenes whose Newton loop has stopped keep x = x_iter.
void launch_apply_dx(uint32_t nv, const float* x_iter, const float* dx, float* x, const SceneStatus* sst,
                     float alpha_const, const SegView& g, hipStream_t s);
void launch_ground_ccd_maxdx(const LsArgs& a, hipStream_t s);
void launch_ccd(const CcdArgs& a, unsigned grid, hipStream_t s);
void launch_pin_delta(uint32_t nfix, const uint32_t* ids, const float* x, const float* x_tilde, SceneStatus* sst,
                      const uint32_t* vert_scene, hipStream_t s);
void launch_reset_status(Status* st, SceneStatus* sst, uint32_t nscenes, hipStream_t s);
void launch_reset_gap(GapStatus* g, uint32_t nscenes, hipStream_t s);
void launch_gap_check(const GapArgs& a, unsigned grid, hipStream_t s);
void launch_reset_line_search(Status* st, SceneStatus* sst, uint32_t nscenes, hipStream_t s);


// The narrow phase on a caller's pair list (one scene, no affine bodies), on device pointers.
// narrow_ccd: CCD step bound (ACCD time of impact / 1.25, 1 when no pair collides) of the VF
// (kind 0: pairs (vertex, face), prims = faces) or EE (kind 1: (edge, edge), prims = edges) pairs
// into toi[0]; work: 2 + n_pairs words after a 16-byte SceneStatus (4 words). narrow_dcd: the
// DCD's contacts appended to `out`; work: 1 word.
void narrow_ccd(int kind, const uint32_t* pairs, uint32_t n_pairs, const uint32_t* prims, const float* x0,
                const float* x1, const float* offset, int fp64, int budget, float* toi, uint32_t* work, hipStream_t s);
void narrow_dcd(int kind, const uint32_t* pairs, uint32_t n_pairs, const uint32_t* prims, const float* x,
                const float* area_a, const float* area_b, const float* offset, const float* dhat, float kappa,
                int quadratic, int fp64, const ContactBuf& out, uint32_t* work, hipStream_t s);

}  // namespace lcsx
