// Newton driver (host) for the MI355X path. Mirrors NewtonSolver::physics_step_GPU
// (reference Solver/SimulationSolver/newton_solver.cpp:4051-4345) with the host round trips
// reduced to one status read per Newton iteration plus one per PCG chunk.
#include "lcsx_solver.h"
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <optional>

namespace lcsx
{

namespace
{
constexpr unsigned kPairGridMax = 4096;
constexpr int      kPcgChunk    = 10;
constexpr float    kFltEpsilon  = 1.19209290e-7f;  // Epsilon of the energy test (constant_value.h:12)
constexpr int      kMixedSweep  = 25;  // PCG iterations between residual replacements (mixed precision)
// Largest candidate-pair list (per kind) and contact list the library allocates: 2^30 pairs are
// 8 GiB of indices per list (plus the CCD's rest list), 2^27 contacts 8 GiB of records and slots.
constexpr uint64_t kMaxPairs    = 1ull << 30;
constexpr uint64_t kMaxContacts = 1ull << 27;

struct EventPool
{
    struct Rec
    {
        std::string name;
        hipEvent_t  a, b;
        bool        count = true;  // false: adds its time to the name's current call
    };
    std::vector<hipEvent_t> free_;
    std::vector<Rec>        pending;
    hipEvent_t              get()
    {
        if (!free_.empty())
        {
            hipEvent_t e = free_.back();
            free_.pop_back();
            return e;
        }
        hipEvent_t e;
        LCSX_HIP(hipEventCreate(&e));
        return e;
    }
    ~EventPool()
    {
        for (auto e : free_) (void)hipEventDestroy(e);
        for (auto& r : pending)
        {
            (void)hipEventDestroy(r.a);
            (void)hipEventDestroy(r.b);
        }
    }
};
// per thread, as solvers may run in several at once
thread_local EventPool* g_pool = nullptr;
thread_local hipEvent_t g_open = nullptr;
}  // namespace

Solver::~Solver()
{
    clear_graphs();
    if (side) (void)hipStreamDestroy(side);
    if (ev_fork) (void)hipEventDestroy(ev_fork);
    if (ev_join) (void)hipEventDestroy(ev_join);
    if (stream) (void)hipStreamDestroy(stream);
}

void Solver::clear_graphs()
{
    for (auto& kv : pcg_graphs) (void)hipGraphExecDestroy(kv.second);
    pcg_graphs.clear();
    graph_epoch++;
}

unsigned Solver::pair_grid(uint32_t cap) const { return std::max(1u, std::min(kPairGridMax, grid_for(cap, 256))); }

void Solver::tic()
{
    if (!timing) return;
    if (!g_pool) g_pool = new EventPool();
    g_open = g_pool->get();
    LCSX_HIP(hipEventRecord(g_open, stream));
}
void Solver::toc(const char* name)
{
    if (!timing || !g_open) return;
    hipEvent_t b = g_pool->get();
    LCSX_HIP(hipEventRecord(b, stream));
    g_pool->pending.push_back({name, g_open, b, true});
    g_open = nullptr;
}
void Solver::toc_part(const char* name)
{
    if (!timing || !g_open) return;
    hipEvent_t b = g_pool->get();
    LCSX_HIP(hipEventRecord(b, stream));
    g_pool->pending.push_back({name, g_open, b, false});
    g_open = nullptr;
}

hipEvent_t Solver::ev_get()
{
    if (!g_pool) g_pool = new EventPool();
    return g_pool->get();
}
void Solver::ev_put(hipEvent_t e) { g_pool->free_.push_back(e); }

void Solver::read_status()
{
    host_sst.resize(S.nscenes);
    LCSX_HIP(hipMemcpyAsync(&host_status, status.p, sizeof(Status), hipMemcpyDeviceToHost, stream));
    LCSX_HIP(hipMemcpyAsync(host_sst.data(), sst.p, S.nscenes * sizeof(SceneStatus), hipMemcpyDeviceToHost, stream));
    LCSX_HIP(hipStreamSynchronize(stream));
    flush_events();
}

// Converts completed event pairs into per-name time sums (call after a stream synchronize).
void Solver::flush_events()
{
    if (g_pool)
    {
        for (auto& r : g_pool->pending)
        {
            float ms = 0.0f;
            if (hipEventElapsedTime(&ms, r.a, r.b) == hipSuccess)
            {
                auto& t = times[r.name];
                t.first += ms;
                if (r.count) t.second += 1;
            }
            g_pool->free_.push_back(r.a);
            g_pool->free_.push_back(r.b);
        }
        g_pool->pending.clear();
    }
}

void Solver::alloc_collision(uint32_t vf, uint32_t ee, uint32_t nc)
{
    clear_graphs();
    cap_vf = std::max(vf, 1024u);
    cap_ee = std::max(ee, 1024u);
    cap_c  = std::max(nc, 1024u);
    pairs_vf.alloc(2 * (size_t)cap_vf);
    pairs_ee.alloc(2 * (size_t)cap_ee);
    c_idx.alloc(cap_c);
    c_nk.alloc(cap_c);
    c_w.alloc(cap_c);
    c_aux.alloc(cap_c);
    ccd_rest_vf.alloc(cap_vf);
    ccd_pairs_fresh = false;
    ccd_rest_ee.alloc(cap_ee);
    vc_list.alloc(slots_per_contact * (size_t)cap_c);
    if (!S.bodies.empty())
    {
        c_gr.alloc(2 * (size_t)cap_c);
        c_gw.alloc(2 * (size_t)cap_c);
    }
    // per-block partial sums of the SpMV: row blocks + scene-aligned slot chunks (4 slots per contact)
    const size_t chunks = max_chunks(slots_per_contact * cap_c) + 1;
    part_pq.alloc(4 * (size_t)S.n_rb + chunks);  // four per row block (the SpMV's 64-row blocks), one per chunk
    cb_scene_d.alloc(chunks);
    cb_slot0_d.alloc(chunks);
    vc_row.alloc(slots_per_contact * (size_t)cap_c);
    vc_coef.alloc(slots_per_contact * (size_t)cap_c);
    vc_runsum.alloc(slots_per_contact * (size_t)cap_c);
    vc_tc.alloc(cap_c);
    vc_ready = false;
}

void Solver::init()
{
    clear_graphs();
    S.build(meshes);
    setup_ready = true;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
    {
        set_error("no HIP device available");
        throw NoDevice();
    }
    LCSX_HIP(hipSetDevice(device));
    if (!stream) LCSX_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    if (!side) LCSX_HIP(hipStreamCreateWithFlags(&side, hipStreamNonBlocking));  // default priority, as stream
    if (!ev_fork) LCSX_HIP(hipEventCreateWithFlags(&ev_fork, hipEventDisableTiming));
    if (!ev_join) LCSX_HIP(hipEventCreateWithFlags(&ev_join, hipEventDisableTiming));
    const uint32_t nv = S.nv;
    for (auto* b : {&x, &v, &x_step, &x_iter, &x_tilde, &dx, &cgB, &r, &z, &q, &spmv_tmp}) b->alloc(3 * (size_t)nv);
    for (auto* b : {&p[0], &p[1]}) b->alloc(4 * (size_t)nv);  // 16-byte rows for the SpMV's gathers
    diag.alloc(9 * (size_t)nv);
    diag_mat.alloc(9 * (size_t)nv);
    minv.alloc(9 * (size_t)nv);
    sell_val.alloc(9 * (size_t)std::max(S.nblocks, 1u));
    part_rz.alloc(S.n_rb + 1);
    plan_grid();
    // scene tables
    const uint32_t ns = S.nscenes;
    sc_v0_d.upload(S.sc_v0, stream);
    sc_rb0_d.upload(S.sc_rb0, stream);
    rb_scene_d.upload(S.rb_scene, stream);
    rb_row0_d.upload(S.rb_row0, stream);
    vert_scene_d.upload(S.vert_scene, stream);
    sc_cb0_d.alloc(ns + 1);
    sc_cb0_zero.alloc(ns + 1);
    LCSX_HIP(hipMemsetAsync(sc_cb0_d.p, 0, (ns + 1) * sizeof(uint32_t), stream));
    LCSX_HIP(hipMemsetAsync(sc_cb0_zero.p, 0, (ns + 1) * sizeof(uint32_t), stream));
    active_h.assign(ns, 1);
    active_d.upload(active_h, stream);
    sst.alloc(ns);
    energy_d.alloc(ns);
    host_sst.assign(ns, SceneStatus{});
    host_pcg.assign(ns, PcgState{});
    scene_stats.assign(ns, lcsx_stats{});
    for (auto& st : scene_stats) st.toi_min = 1.0f;
    stats.toi_min = 1.0f;
    verts_per_scene.assign(ns, 0);
    for (uint32_t sc = 0; sc < ns; sc++) verts_per_scene[sc] = S.sc_verts[sc];
    if (prm.precision >= 1)
    {
        sell_p.alloc(5 * (size_t)std::max(S.nblocks, 1u));
        part_res.alloc(2 * (size_t)S.n_rb);
    }
    slots_per_contact = S.bodies.empty() ? 4u : 8u;
    upload_state_constants();
    tree_face.init(3, faces.p, S.nf, S.sc_f0.data(), ns);
    tree_edge.init(2, edges.p, S.ne, S.sc_e0.data(), ns);
    // one offset and one d_hat for every vertex: the edge-edge pair test is symmetric, and the
    // edge tree is queried by itself in sorted leaf order (each pair found once, from its first leaf)
    sorted_ee = true;
    for (uint32_t i = 0; i < S.nv; i++)
        if (S.row_kind[i] < 2 && (S.offset[i] != S.offset[0] || S.dhat[i] != S.dhat[0])) sorted_ee = false;
    tree_edge.sorted_keys = sorted_ee ? 1 : 0;
    alloc_collision(24 * nv, 24 * S.ne, 12 * nv);
    vc_cnt.alloc(nv + 1);
    ccd_rest_count.alloc(2);
    vc_ptr.alloc(nv + 1);
    status.alloc(1);
    gap.alloc(ns);
    pcg_state.alloc(ns);
    LCSX_HIP(hipMemsetAsync(pcg_state.p, 0, ns * sizeof(PcgState), stream));
    LCSX_HIP(hipMemsetAsync(status.p, 0, sizeof(Status), stream));
    LCSX_HIP(hipMemsetAsync(sst.p, 0, ns * sizeof(SceneStatus), stream));
    host_status = Status{};
    LCSX_HIP(hipMemsetAsync(sell_val.p, 0, sell_val.n * sizeof(float), stream));
    explicit_targets.assign(3 * S.fixed_verts.size(), 0.0f);
    has_explicit.assign(meshes.size(), 0);
    LCSX_HIP(hipStreamSynchronize(stream));
    inited = true;
    frame  = 0;
}

// The one-launch PCG's shape, and the scenes dealt to launches ("rounds") of at most grid_wgs
// workgroups, the largest scenes first into the first round that still holds them. Up to two rounds: a
// solve takes 1.12 ms in one round of 121,000 rows (1.88 with three launches per iteration), 3.4 ms in two
// of 236,000 rows (4.0) and as long as the launches, 4.3 ms, in three of 306,000.
void Solver::plan_grid()
{
    grid_slots.free();
    grid_zx.free();
    uint32_t width = 0, most = 0;
    for (size_t k = 0; k + 1 < S.sl_off.size(); k++) width = std::max(width, S.sl_off[k + 1] - S.sl_off[k]);
    for (uint32_t sc = 0; sc < S.nscenes; sc++) most = std::max(most, S.sc_rb0[sc + 1] - S.sc_rb0[sc]);
    grid_most = most;
    const uint32_t limit = grid_wgs(device);
    grid_shape = grid_plan(most, S.n_rb, width, limit);
    grid_round.clear();
    if (!grid_shape.U) return;
    constexpr size_t kRounds = 2;
    const uint32_t per = grid_shape.row_blocks();
    auto           wgs = [&](uint32_t sc) { return (S.sc_rb0[sc + 1] - S.sc_rb0[sc] + per - 1) / per; };
    std::vector<uint32_t> order(S.nscenes);
    for (uint32_t sc = 0; sc < S.nscenes; sc++) order[sc] = sc;
    std::stable_sort(order.begin(), order.end(), [&](uint32_t x, uint32_t y) { return wgs(x) > wgs(y); });
    std::vector<uint32_t> used, round(S.nscenes);
    for (uint32_t sc : order)
    {
        size_t r = 0;
        while (r < used.size() && used[r] + wgs(sc) > limit) r++;
        if (r == used.size()) used.push_back(0u);
        used[r] += wgs(sc);
        round[sc] = (uint32_t)r;
    }
    if (used.size() > kRounds)
    {
        grid_shape = GridPlan{};
        return;
    }
    grid_round.push_back(0u);
    std::vector<uint2> tab;
    for (size_t r = 0; r < used.size(); r++)
    {
        for (uint32_t sc : order)
            if (round[sc] == r)
                for (uint32_t k = 0; k < wgs(sc); k++) tab.push_back(make_uint2(sc, k));
        grid_round.push_back((uint32_t)tab.size());
    }
    if (S.nscenes > 1) grid_tab.upload(tab, stream);
    LCSX_HIP(hipStreamSynchronize(stream));
}

void Solver::upload_state_constants()
{
    hipStream_t s = stream;
    x.upload(S.rest_x, s);
    rest_x.upload(S.rest_x, s);
    std::vector<float> zero(3 * (size_t)S.nv, 0.0f);
    v.upload(zero, s);
    x_step.upload(S.rest_x, s);
    offset.upload(S.offset, s);
    dhat.upload(S.dhat, s);
    vert_mass.upload(S.vert_mass, s);
    vert_area.upload(S.vert_area, s);
    face_area.upload(S.face_area, s);
    edge_area.upload(S.edge_area, s);
    is_fixed.upload(S.is_fixed, s);
    faces.upload(S.faces, s);
    edges.upload(S.edges, s);
    sf.upload(S.sf, s);
    bh.upload(S.bh, s);
    v_sf_ptr.upload(S.v_sf_ptr, s);
    v_sf.upload(S.v_sf, s);
    v_bh_ptr.upload(S.v_bh_ptr, s);
    v_bh.upload(S.v_bh, s);
    sp.upload(S.sp, s);
    v_sp_ptr.upload(S.v_sp_ptr, s);
    v_sp.upload(S.v_sp, s);
    sl_off.upload(S.sl_off, s);
    sell_col.upload(S.sell_col, s);
    blk_ptr.upload(S.blk_ptr, s);
    blk_contrib.upload(S.blk_contrib, s);
    fixed_ids.upload(S.fixed_verts, s);
    row_kind_d.upload(S.row_kind, s);
    cluster_vert.upload(S.cluster_v, s);
    n_cluster_vert = (uint32_t)S.cluster_v.size();
    if (S.cluster_f_use) cluster_face.init(3, faces.p, S.cluster_f, S.cluster_f_block, s);
    if (S.cluster_e_use) cluster_edge.init(2, edges.p, S.cluster_e, S.cluster_e_block, s);
    vert_body_d.upload(S.vert_body, s);
    body_X_d.upload(S.body_X, s);
    static_assert(sizeof(BodyDev) == sizeof(Setup::Body), "body record layout");
    if (!S.bodies.empty())
    {
        bodies_d.alloc(S.bodies.size());
        LCSX_HIP(hipMemcpyAsync(bodies_d.p, S.bodies.data(), S.bodies.size() * sizeof(BodyDev), hipMemcpyHostToDevice, s));
    }
    targets.alloc(3 * std::max<size_t>(S.fixed_verts.size(), 1));
    const size_t       nsf = S.sf.size() / 3, nbh = S.bh.size() / 4;
    std::vector<float4> dm(nsf), cc(nsf), hc(nbh);
    for (size_t f = 0; f < nsf; f++)
    {
        dm[f] = make_float4(S.sf_Dm[4 * f], S.sf_Dm[4 * f + 1], S.sf_Dm[4 * f + 2], S.sf_Dm[4 * f + 3]);
        cc[f] = make_float4(S.sf_area[f], S.sf_mu[f], S.sf_lambda[f], 0.0f);
    }
    for (size_t e = 0; e < nbh; e++) hc[e] = make_float4(S.bh_angle[e], S.bh_hbar[e], S.bh_k[e], 0.0f);
    sf_Dm.upload(dm, s);
    sf_c.upload(cc, s);
    bh_c.upload(hc, s);
    const size_t        nsp = S.sp.size() / 2;
    std::vector<float2> spc(nsp);
    for (size_t e = 0; e < nsp; e++) spc[e] = make_float2(S.sp_rest[e], S.sp_k[e]);
    sp_c.upload(spc, s);
    spring_stage.alloc(16 * std::max<size_t>(nsp, 1));
    face_stage.alloc(64 * std::max<size_t>(nsf, 1));
    hinge_stage.alloc(16 * std::max<size_t>(nbh, 1));
    LCSX_HIP(hipStreamSynchronize(s));
}

ContactView Solver::contact_view() const
{
    return ContactView{c_idx.p, c_nk.p, c_w.p, c_aux.p, &status.p->n_contacts, cap_c, c_gr.p, c_gw.p};
}
uint32_t Solver::contact_triplets()
{
    read_status();
    const uint32_t nc = (uint32_t)std::min<uint64_t>(host_status.n_contacts, cap_c);
    if (nc == 0) return 0;
    ctb.contacts(nc);
    const uint32_t m = launch_contact_triplets(contact_view(), nc, pair_grid(nc), ctb, stream);
    LCSX_HIP(hipStreamSynchronize(stream));
    return m;
}
VertContacts Solver::vert_contacts()
{
    // no lists before the first contact assembly, or without self collision; the slot count
    // sizes the SpMV's grid, so it is read back once (one small synchronisation)
    if (!(prm.use_self_collision && vc_ready)) return VertContacts{nullptr, nullptr, nullptr, nullptr, nullptr, 0u, nullptr};
    uint32_t nc = 0;
    LCSX_HIP(hipMemcpyAsync(&nc, &status.p->n_contacts, sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
    LCSX_HIP(hipStreamSynchronize(stream));
    nc = std::min(nc, cap_c);
    if (nc == 0) return VertContacts{nullptr, nullptr, nullptr, nullptr, nullptr, 0u, nullptr};
    return VertContacts{vc_ptr.p, vc_list.p, vc_row.p, vc_coef.p, vc_tc.p, slots_per_contact * nc, vc_ptr.p + S.nv,
                        vc_runsum.p};
}
// The SpMV's diagonal is the material one: contact diagonal blocks enter through the contact slots.
SegView Solver::seg_view(bool with_chunks) const
{
    SegView g{};
    g.nscenes    = S.nscenes;
    g.n_rb       = S.n_rb;
    g.sc_v0      = sc_v0_d.p;
    g.sc_rb0     = sc_rb0_d.p;
    g.rb_scene   = rb_scene_d.p;
    g.rb_row0    = rb_row0_d.p;
    g.vert_scene = vert_scene_d.p;
    g.active     = active_d.p;
    g.sc_cb0     = with_chunks ? sc_cb0_d.p : sc_cb0_zero.p;
    g.cb_scene   = cb_scene_d.p;
    g.cb_slot0   = cb_slot0_d.p;
    return g;
}

SellView Solver::sell_view() const
{
    return SellView{sl_off.p, sell_col.p, sell_val.p, diag_mat.p, S.nblocks, nullptr, 0};
}
SellView Solver::sell_view_lp() const
{
    return SellView{sl_off.p, sell_col.p, sell_val.p, diag_mat.p, S.nblocks, sell_p.p, prm.precision == 2};
}

// ------------------------------------------------------------------ stages
void Solver::frame_begin()
{
    ccd_pairs_fresh = false;  // the last line search may have covered only some scenes of a batch
    const float t   = (float)frame * prm.implicit_dt;
    const size_t nf = S.fixed_verts.size();
    if (nf)
    {
        std::vector<float> tg(3 * nf);
        for (size_t k = 0; k < nf; k++)
        {
            if (has_explicit[S.fixed_mesh[k]])
            {
                for (int d = 0; d < 3; d++) tg[3 * k + d] = explicit_targets[3 * k + d];
                continue;
            }
            animate_target(S.fixed_anim[k], t, &S.rest_x[3 * (size_t)S.fixed_verts[k]], &tg[3 * k]);
        }
        targets.upload(tg, stream);
        launch_pin_velocity((uint32_t)nf, fixed_ids.p, targets.p, x.p, v.p, prm.implicit_dt, stream);
    }
    LCSX_HIP(hipMemcpyAsync(x_step.p, x.p, x.n * sizeof(float), hipMemcpyDeviceToDevice, stream));
    tic();
    tree_face.construct(x_step.p, verts_per_scene.data(), stream);
    tree_edge.construct(x_step.p, verts_per_scene.data(), stream);
    toc("lbvh_build");
}

void Solver::predict()
{
    launch_predict(S.nv, x_step.p, v.p, is_fixed.p, row_kind_d.p, prm.implicit_dt, prm.gravity, x_iter.p, x_tilde.p, x.p,
                   stream);
}

void Solver::iter_begin()
{
    LCSX_HIP(hipMemcpyAsync(x_iter.p, x.p, x.n * sizeof(float), hipMemcpyDeviceToDevice, stream));
    launch_reset_status(status.p, sst.p, S.nscenes, stream);
}

void Solver::material()
{
    tic();
    const uint32_t nsf = (uint32_t)(S.sf.size() / 3), nbh = (uint32_t)(S.bh.size() / 4), nsp = (uint32_t)(S.sp.size() / 2);
    launch_spring_stage(nsp, sp.p, sp_c.p, x.p, spring_stage.p, stream);
    launch_face_stage(nsf, sf.p, sf_Dm.p, sf_c.p, x.p, face_stage.p, stream);
    launch_hinge_stage(nbh, bh.p, bh_c.p, prm.bending_scaling, x.p, hinge_stage.p, stream);
    VertArgs a{};
    a.nv       = S.nv;
    a.row_kind = row_kind_d.p;
    a.x        = x.p;
    a.x_tilde  = x_tilde.p;
    a.mass     = vert_mass.p;
    a.fixed    = is_fixed.p;
    a.area     = vert_area.p;
    a.offset   = offset.p;
    a.dhat     = dhat.p;
    float h    = prm.implicit_dt;
    a.h2inv    = 1.0f / (h * h);
    a.kD       = prm.stiffness_dirichlet;
    a.kappa    = prm.stiffness_collision;
    a.floor_y  = prm.floor_y;
    a.use_floor = prm.use_floor;
    a.quadratic = prm.contact_energy_type == 0;
    a.v_sf_ptr = v_sf_ptr.p;
    a.v_sf     = v_sf.p;
    a.v_bh_ptr = v_bh_ptr.p;
    a.v_bh     = v_bh.p;
    a.v_sp_ptr = v_sp_ptr.p;
    a.v_sp     = v_sp.p;
    a.spring_stage = spring_stage.p;
    a.face_stage  = face_stage.p;
    a.hinge_stage = hinge_stage.p;
    a.cgB      = cgB.p;
    a.diag     = diag.p;
    a.diag_mat = diag_mat.p;
    launch_vert_assemble(a, stream);
    launch_offdiag(S.nblocks, blk_ptr.p, blk_contrib.p, spring_stage.p, face_stage.p, hinge_stage.p, sell_val.p, stream);
    if (!S.bodies.empty())
    {
        AbdArgs b{};
        b.nb        = (uint32_t)S.bodies.size();
        b.n_rows    = S.nv;
        b.nblocks   = S.nblocks;
        b.bodies    = bodies_d.p;
        b.x         = x.p;
        b.x_tilde   = x_tilde.p;
        b.body_X    = body_X_d.p;
        b.fixed     = is_fixed.p;
        b.offset    = offset.p;
        b.dhat      = dhat.p;
        b.area      = vert_area.p;
        b.h2inv     = a.h2inv;
        b.kD        = a.kD;
        b.kappa     = a.kappa;
        b.floor_y   = a.floor_y;
        b.use_floor = a.use_floor;
        b.quadratic = a.quadratic;
        b.cgB       = cgB.p;
        b.diag      = diag.p;
        b.diag_mat  = diag_mat.p;
        b.sell_val  = sell_val.p;
        launch_abd_material(b, stream);
    }
    if (prm.precision >= 1)
        launch_pack_fp16(S.nslices, S.nv, sl_off.p, S.nblocks, sell_val.p, S.bodies.empty() ? nullptr : row_kind_d.p,
                         sell_p.p, prm.precision == 2, stream);
    toc("material");
}

ClusterQuery Solver::cluster_query(const float* x0) const
{
    ClusterQuery c{};
    c.vert_scene = vert_scene_d.p;
    c.active     = active_d.p;
    c.x0         = x0;
    c.x1         = x.p;
    c.offset     = offset.p;
    c.dhat       = dhat.p;
    return c;
}

void Solver::query_faces(bool ccd)
{
    if (S.nf == 0) return;
    const float* x0 = ccd ? x_iter.p : x.p;
    Status*      st = status.p;
    const bool clusters = S.cluster_f_use && query_by_clusters(query_variant);
    tree_face.refit(x0, x.p, offset.p, stream, !clusters);
    if (clusters)
    {
        ClusterQuery c = cluster_query(x0);
        c.order        = cluster_vert.p;
        c.n            = n_cluster_vert;
        c.pairs        = pairs_vf.p;
        c.capacity     = cap_vf;
        c.count        = ccd ? &st->n_vf_ccd : &st->n_vf;
        cluster_face.refit(x0, x.p, offset.p, nullptr, stream);
        cluster_face.query(c, nullptr, stream);
        return;
    }
    QueryArgs q{};
    q.vert_scene = vert_scene_d.p;
    q.active     = active_d.p;
    q.row_kind   = row_kind_d.p;
    q.mode       = QueryVerts;
    q.n_queries  = S.nv;
    q.x0         = x0;
    q.x1         = x.p;
    q.offset     = offset.p;
    q.dhat       = dhat.p;
    q.pairs      = pairs_vf.p;
    q.capacity   = cap_vf;
    q.count      = ccd ? &st->n_vf_ccd : &st->n_vf;
    q.overflow   = &st->overflow;
    q.variant    = query_variant;
    lbvh_query(tree_face, q, stream);
}

void Solver::query_edges(bool ccd)
{
    if (S.ne == 0) return;
    const float* x0 = ccd ? x_iter.p : x.p;
    Status*      st = status.p;
    const bool clusters = S.cluster_e_use && query_by_clusters(query_variant);
    tree_edge.refit(x0, x.p, offset.p, stream, !clusters);
    if (clusters)
    {
        ClusterQuery    c       = cluster_query(x0);
        const uint32_t* leaf_of = sorted_ee ? tree_edge.leaf_of.p : nullptr;
        c.order                 = cluster_edge.elem.p;
        c.n                     = cluster_edge.blocks * kClusterLeaves;
        c.edges                 = edges.p;
        c.pairs                 = pairs_ee.p;
        c.capacity              = cap_ee;
        c.count                 = ccd ? &st->n_ee_ccd : &st->n_ee;
        cluster_edge.refit(x0, x.p, offset.p, leaf_of, stream);
        cluster_edge.query(c, leaf_of, stream);
        return;
    }
    QueryArgs q{};
    q.vert_scene = vert_scene_d.p;
    q.active     = active_d.p;
    q.row_kind   = row_kind_d.p;
    q.mode       = QueryEdges;
    q.n_queries  = S.ne;
    q.x0         = x0;
    q.x1         = x.p;
    q.edges      = edges.p;
    q.offset     = offset.p;
    q.dhat       = dhat.p;
    q.pairs      = pairs_ee.p;
    q.capacity   = cap_ee;
    q.count      = ccd ? &st->n_ee_ccd : &st->n_ee;
    q.overflow   = &st->overflow;
    q.variant    = query_variant;
    q.sorted_self = sorted_ee ? 1 : 0;
    q.order       = tree_edge.sorted_to_orig;
    lbvh_query(tree_edge, q, stream);
}

void Solver::broad_phase(bool ccd)
{
    tic();
    query_faces(ccd);
    query_edges(ccd);
    last_bp = ccd ? 2 : 1;
    toc(ccd ? "broadphase_ccd" : "broadphase_dcd");
}

void Solver::dcd(bool from_ccd_pairs)
{
    vc_ready = false;  // new contact set: the per-vertex lists are rebuilt by contact_assemble
    tic();
    ContactBuf out{c_idx.p, c_nk.p, c_w.p, c_aux.p, &status.p->n_contacts, cap_c};
    DcdArgs    a{};
    a.x      = x.p;
    a.faces  = faces.p;
    a.edges  = edges.p;
    a.offset = offset.p;
    a.dhat   = dhat.p;
    a.kappa  = prm.stiffness_collision;
    a.fp64   = prm.precision >= 1;
    a.quadratic = prm.contact_energy_type == 0;
    a.out    = out;
    a.vert_body = S.bodies.empty() ? nullptr : vert_body_d.p;
    a.pairs = pairs_vf.p;
    a.pair_count = from_ccd_pairs ? &status.p->n_vf_ccd : &status.p->n_vf;
    a.pair_capacity = cap_vf;
    a.area_a = vert_area.p;
    a.area_b = face_area.p;
    launch_dcd(a, 0, pair_grid(cap_vf), stream);
    a.pairs = pairs_ee.p;
    a.pair_count = from_ccd_pairs ? &status.p->n_ee_ccd : &status.p->n_ee;
    a.pair_capacity = cap_ee;
    a.area_a = edge_area.p;
    a.area_b = edge_area.p;
    launch_dcd(a, 1, pair_grid(cap_ee), stream);
    if (!S.bodies.empty())
        launch_contact_lift(contact_view(), pair_grid(cap_c), vert_body_d.p, bodies_d.p, body_X_d.p, c_gr.p, c_gw.p, stream);
    toc("dcd");
}

// The DCD candidates of a Newton iteration after the first of a frame: the swept boxes of the
// previous line search (x_iter to x_iter + dx, padded as the DCD boxes) contain the boxes at
// x_iter + alpha dx for any alpha in [0, 1], so its candidate pairs include every pair the DCD
// broad phase would find; the narrow phase keeps exactly the same contacts (its distance test
// decides). Skips one of the two broad phases per iteration.
void Solver::update_contacts(bool reuse_ccd_pairs)
{
    if (!prm.use_self_collision) return;
    dcd_reused = reuse_ccd_pairs && ccd_pairs_fresh;
    if (!dcd_reused) broad_phase(false);
    dcd(dcd_reused);
}

void Solver::contact_assemble()
{
    if (!prm.use_self_collision) return;
    tic();
    // the run sums are free until the PCG: their words hold the ordered slot list meanwhile
    launch_contact_adjacency(contact_view(), S.nv, pair_grid(cap_c), vc_cnt.p, vc_ptr.p, vc_list.p, vc_row.p, vc_coef.p,
                             reinterpret_cast<uint32_t*>(vc_runsum.p), seg_view(true), sc_cb0_d.p, cb_scene_d.p,
                             cb_slot0_d.p, S.repeats, stream);
    vc_ready = true;
    VertContacts vc{vc_ptr.p, vc_list.p, vc_row.p, vc_coef.p, vc_tc.p, 0u, vc_ptr.p + S.nv};  // assembly walks the per-row lists
    launch_contact_assemble(contact_view(), vc, cgB.p, diag.p, S.nv, stream);
    toc("contact_assemble");
}

int Solver::pcg_run(PcgArgs& a, const SellView& A, const ContactView& cv, const VertContacts& vc, int max_iters,
                    int replace_every, bool one_launch)
{
    const uint32_t ns = S.nscenes;
    const unsigned mc = vc.ptr ? max_chunks(vc.nslots) : 0u;
    launch_pcg_init(a, stream);
    host_pcg.assign(ns, PcgState{});
    // one launch (per round of scenes) for all iterations up to the next residual replacement, or three
    // per iteration. The launches' time hardly depends on the contacts, the one launch's does. One row
    // block per workgroup: up to two slot chunks per 256 threads (a 200 x 200 cloth on a sphere, 300
    // iterations: 1.35 ms against 2.02 at 4,276 contacts; a 100 x 100 tube 1.30 against 1.56 at 13,000). Two
    // row blocks per workgroup spill with contacts (94,000 rows, 100 iterations: 1.09 against 1.94 ms
    // without contacts, 1.95 against 2.05 with 215, 2.19 against 2.09 with 1,172, 2.87 against 2.22 with
    // 18,000): a chunk per scene and one for 16 workgroups, or 8 in a batch, whose scenes wait for their own
    // chunks only (202,000 rows with a chunk for 11 workgroups: 2.48 against 2.99). Rows of 17 to 32 blocks
    // (irregular triangulations) spill most with contacts, and what is spilled is read back every iteration:
    // only up to 20 row blocks in the largest scene, or 64 of 16-bit blocks (one launch against the launches,
    // us a solve of about 100 iterations in first contact: FP32 4,867 rows 239 and 224 to 267 from run to run,
    // 10,051 292 and 283, 63,142 595 and 385; FP16 13,186 rows 319 and 336, 40,642 384 and 356; FP32 8 scenes
    // of 4,867 322 and 349).
    GridPlan  gp;
    GridLease lease;
    const uint32_t gw = grid_round.empty() ? 0u : grid_round.back();
    const uint32_t grid_chunks = 2u * gw * (kGridThreads / 256u);  // that the words are for
    const uint32_t most_chunks = grid_shape.U == 2 ? grid_chunks : std::min(grid_chunks, ns + gw / (ns == 1u ? 16u : 8u));
    const bool     wide = grid_shape.K == 8 && mc && grid_most > (A.val_p ? 64u : 20u);
    if (one_launch && pcg_grid && grid_shape.U && spmv_sample == 0 && mc <= most_chunks && !wide &&
        lease.take(device))
        gp = grid_shape;
    const size_t grid_words = 5 * (size_t)S.n_rb + grid_chunks;
    // (a solve's epochs stay below kPoison, whatever its cap)
    if (gp.U && (!grid_slots.p || (uint64_t)grid_epoch + (uint64_t)std::max(max_iters, 0) > 0xfffffff0u))
    {
        if (!grid_slots.p) grid_slots.alloc(grid_words);
        if (!grid_zx.p) grid_zx.alloc(3 * (size_t)S.nv);
        launch_grid_clear(grid_slots.p, grid_slots.n, stream);
        launch_grid_clear(grid_zx.p, grid_zx.n, stream);
        grid_epoch = 2;
    }
    int  issued = 0;
    int  par    = 0;
    bool nan    = false;
    while (issued < max_iters)
    {
        // one host check per convergence-test interval (at least kPcgChunk launches), chunks
        // ending at the residual replacements
        int chunk = std::min(gp.U ? max_iters : std::max(kPcgChunk, a.check_every > 1 ? (int)a.check_every : 0),
                             max_iters - issued);
        if (replace_every > 0) chunk = std::min(chunk, replace_every - issued % replace_every);
        if (gp.U)
        {
            PcgArgs b = a;
            b.p_old   = p[par].p;
            b.p_new   = p[1 - par].p;
            b.k       = (uint32_t)issued;
            for (size_t r = 0; r + 1 < grid_round.size(); r++)
            {
                const uint32_t w0 = grid_round[r];
                const GridSync g{grid_slots.p, grid_slots.p + S.n_rb, grid_zx.p, ns > 1 ? grid_tab.p + w0 : nullptr, grid_epoch};
                const uint32_t wgs = grid_round[r + 1] - w0;
                launch_pcg_grid(gp, grid_withhold && wgs > 1 ? wgs - 1 : wgs, b, A, cv, vc, g, (uint32_t)chunk, stream);
            }
            grid_epoch += (uint32_t)chunk;
            par = (par + chunk) & 1;
            if (timing) times["pcg_grid"].second += 1;  // launches of this form (no time of its own)
        }
        else if (spmv_sample > 0 || !use_graphs)
        {
            for (int k = 0; k < chunk; k++)
            {
                PcgArgs b = a;
                b.p_old   = p[par].p;
                b.p_new   = p[1 - par].p;
                b.k       = (uint32_t)(issued + k);
                hipEvent_t e0 = nullptr, e1 = nullptr;
                if (spmv_sample > 0 && b.k % (uint32_t)spmv_sample == 0u)
                {
                    e0 = ev_get();
                    e1 = ev_get();
                    spmv_events.push_back({b.k, e0, e1});
                }
                launch_pcg_dir(b, cv, vc, mc, contact_t_per_contact, stream);
                launch_pcg_spmv(b, A, vc, mc, spmv_shape, stream, e0, e1);
                LCSX_HIP(hipGetLastError());
                launch_pcg_update(b, stream);
                par = 1 - par;
            }
        }
        else
        {
            // the slot-chunk grid rounded up to a power of two (blocks past the scene tables' chunk
            // count exit at once), so one graph serves Newton iterations with similar contact counts
            unsigned g = 0;
            if (vc.ptr)
            {
                g = 1;
                while (g < mc) g <<= 1;
                g = std::min(g, max_chunks(slots_per_contact * cap_c));
            }
            const GraphKey key{graph_epoch, issued, chunk, par, g, vc.ptr != nullptr, A.val_p != nullptr,
                               contact_t_per_contact, spmv_shape};
            auto           it = pcg_graphs.find(key);
            if (it == pcg_graphs.end())
            {
                const auto t0 = std::chrono::steady_clock::now();
                if (pcg_graphs.size() >= 64) clear_graphs();
                hipGraph_t     graph = nullptr;
                hipGraphExec_t exec  = nullptr;
                // the captured kernels size their slot work from the device tables, not nslots
                VertContacts vg = vc;
                vg.nslots       = 0u;
                LCSX_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
                enqueue_pcg_chunk(a, A, cv, vg, g, issued, chunk, par);
                LCSX_HIP(hipStreamEndCapture(stream, &graph));
                const hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
                (void)hipGraphDestroy(graph);
                LCSX_HIP(e);
                it = pcg_graphs.emplace(key, exec).first;
                if (timing)
                {
                    // host time of capture + instantiation ("graph_capture_host", not device time)
                    auto& t = times["graph_capture_host"];
                    t.first += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
                    t.second += 1;
                }
            }
            LCSX_HIP(hipGraphLaunch(it->second, stream));
            par = (par + chunk) & 1;
        }
        issued += chunk;
        const bool replace = replace_every > 0 && issued % replace_every == 0 && issued < max_iters;
        if (replace)
        {
            // r = b - A x with the FP32 blocks; the next iteration's r.z (and its stopping test)
            // is this residual's. After convergence x no longer changes and this is harmless.
            launch_spmv(sell_view(), cv, vc, pair_grid(cap_c), a.x, spmv_tmp.p, S.nv, stream);
            launch_residual(a.seg, a.b, spmv_tmp.p, a.minv, a.r, a.z, a.part_rz, part_res.p, stream);
        }
        LCSX_HIP(hipMemcpyAsync(host_pcg.data(), pcg_state.p, ns * sizeof(PcgState), hipMemcpyDeviceToHost, stream));
        std::vector<float> res;
        if (replace)
        {
            res.resize(part_res.n);
            LCSX_HIP(hipMemcpyAsync(res.data(), part_res.p, res.size() * sizeof(float), hipMemcpyDeviceToHost, stream));
        }
        LCSX_HIP(hipStreamSynchronize(stream));
        flush_events();
        uint32_t gave_up = 0u;
        for (const PcgState& h : host_pcg) gave_up |= gp.U ? h.fail : 0u;
        if (gave_up)
        {
            // the launches from the start; from now on, if the rows do not fit (the pattern stays what it is)
            lease.outcome(gave_up, !grid_withhold);
            grid_withhold = false;
            if (gave_up & kGridUnfit) grid_shape = GridPlan{};
            grid_slots.free();
            if (timing) times["pcg_grid_gave_up"].second += 1;
            return pcg_run(a, A, cv, vc, max_iters, replace_every, false);
        }
        bool done = true;
        for (const PcgState& h : host_pcg)
        {
            done = done && h.converged;
            nan  = nan || h.nan;
        }
        if (!done && !res.empty())
        {
            double t = 0.0;
            for (size_t k = 0; k < res.size(); k += 2) t += (double)res[k] + (double)res[k + 1];
            rz_true = t;
        }
        if (done || nan) break;
    }
    if (gp.U && issued > 0) lease.outcome(0u);
    if (nan)
    {
        set_error("NaN/Inf in the PCG iteration");
        throw HipFailure();
    }
    // per scene: iterations run (the stopping one when the test stopped it, else the cap) and
    // r.z of its last evaluated iteration
    int most = 0;
    for (uint32_t sc = 0; sc < ns; sc++)
    {
        const PcgState& h  = host_pcg[sc];
        const bool      on = active_h.empty() || active_h[sc];
        const int       it = !on ? 0 : (h.converged ? (int)h.iters : issued);
        const float     rl = h.rz[(h.converged ? h.iters : (uint32_t)std::max(issued - 1, 0)) & 1u];
        if (on)
        {
            lcsx_stats& st = scene_stats[sc];
            st.pcg_iters   = it;
            st.pcg_iters_total += it;
            st.pcg_rel     = h.rz0 > 0.0f ? std::sqrt(rl / h.rz0) : 0.0f;
        }
        most = std::max(most, it);
    }
    account_spmv((uint32_t)most, vc.nslots);
    return most;
}

// The launches of PCG iterations [k0, k0 + len) (the direct form of a captured chunk).
void Solver::enqueue_pcg_chunk(const PcgArgs& a, const SellView& A, const ContactView& cv, const VertContacts& vc,
                               unsigned mc, int k0, int len, int par)
{
    for (int k = 0; k < len; k++)
    {
        PcgArgs b = a;
        b.p_old   = p[par].p;
        b.p_new   = p[1 - par].p;
        b.k       = (uint32_t)(k0 + k);
        launch_pcg_dir(b, cv, vc, mc, contact_t_per_contact, stream);
        launch_pcg_spmv(b, A, vc, mc, spmv_shape, stream, nullptr, nullptr);
        launch_pcg_update(b, stream);
        par = 1 - par;
    }
}

// Timed SpMV launches: only launches of the first `iters` iterations did work (later ones exit on
// the converged flag).
void Solver::account_spmv(uint32_t iters, uint32_t nslots)
{
    uint32_t counted = 0;
    for (const SpmvEvent& e : spmv_events)
    {
        float ms = 0.0f;
        if (e.k < iters && hipEventElapsedTime(&ms, e.e0, e.e1) == hipSuccess)
        {
            auto& t = times["spmv"];
            t.first += ms;
            t.second += 1;
            counted++;
        }
        ev_put(e.e0);
        ev_put(e.e1);
    }
    spmv_events.clear();
    if (counted)
    {
        // contact slots the timed launches processed ("spmv_slots": slots per launch)
        auto& t = times["spmv_slots"];
        t.first += (double)nslots * counted;
        t.second += (int)counted;
    }
}

// ConjugateGradientSolver (pcg_solver.cpp:15-197), with the stopping test of the reference on
// r.z, per scene of the batch. FP32: every block in FP32. Mixed precision: the SpMV inside the
// iteration reads FP16 blocks (half the bytes); x, r, z, p stay FP32, and after every
// kMixedSweep iterations the recursive residual is replaced by the true residual b - A x computed
// with the FP32 blocks and a compensated r.z (residual replacement: the iteration keeps its search
// direction, so the Krylov progress made so far is not thrown away as a restarted refinement
// would).
void Solver::pcg()
{
    tic();
    ContactView  cv = contact_view();
    VertContacts vc = vert_contacts();
    PcgArgs a{};
    a.n        = S.nv;
    a.b        = cgB.p;
    a.diag     = diag.p;
    a.minv     = minv.p;
    a.x        = dx.p;
    a.r        = r.p;
    a.z        = z.p;
    a.p_old    = p[0].p;  // zeroed by the init (the first iteration reads it)
    a.p_new    = p[1].p;
    a.q        = q.p;
    a.part_rz  = part_rz.p;
    a.part_pq  = part_pq.p;
    a.s        = pcg_state.p;
    a.rel2     = prm.pcg_rel_tol * prm.pcg_rel_tol;
    a.abs_tol  = prm.pcg_abs_tol;
    a.check_every = (uint32_t)std::max(1, prm.pcg_check_every);
    a.runsum   = vc.ptr ? vc_runsum.p : nullptr;
    a.vc_ptr   = vc.ptr;
    a.seg      = seg_view(vc.ptr != nullptr);
    const bool mixed = prm.precision >= 1;
    // replacements at multiples of the test interval, so the test after one sees the true residual
    const int every = (int)a.check_every;
    const int repl  = mixed ? every * ((kMixedSweep + every - 1) / every) : 0;
    rz_true         = -1.0;
    pcg_run(a, mixed ? sell_view_lp() : sell_view(), cv, vc, prm.pcg_iter_count, repl);
    toc("pcg");
    fold_stats();
}

void Solver::ccd_ground()
{
    LsArgs l{};
    l.nv        = S.nv;
    l.x_iter    = x_iter.p;
    l.x         = x.p;
    l.dx        = dx.p;
    l.fixed     = is_fixed.p;
    l.offset    = offset.p;
    l.floor_y   = prm.floor_y;
    l.use_floor = prm.use_floor && prm.use_ccd_linesearch;
    l.st        = status.p;
    l.sst       = sst.p;
    l.seg       = seg_view(false);
    l.row_kind  = row_kind_d.p;
    launch_ground_ccd_maxdx(l, stream);
}

// One ACCD pass over the swept candidates of one kind (0 VF, 1 EE): the first pass runs every
// pair with the iteration budget and lists those that need more; the rest pass runs the listed
// pairs with the full budget (a small grid: grid-stride over the list).
void Solver::ccd_pass(int kind, bool rest, hipStream_t s)
{
    CcdArgs c{};
    c.x0            = x_iter.p;
    c.x1            = x.p;
    c.faces         = faces.p;
    c.edges         = edges.p;
    c.offset        = offset.p;
    c.sst           = sst.p;
    c.vert_scene    = S.nscenes > 1 ? vert_scene_d.p : nullptr;
    c.vert_body     = S.bodies.empty() ? nullptr : vert_body_d.p;
    c.fp64          = prm.precision >= 1;
    c.budget        = ccd_budget;
    c.rest          = rest ? 1 : 0;
    c.kind          = kind;
    c.pairs         = kind == 0 ? pairs_vf.p : pairs_ee.p;
    c.pair_count    = kind == 0 ? &status.p->n_vf_ccd : &status.p->n_ee_ccd;
    c.pair_capacity = kind == 0 ? cap_vf : cap_ee;
    c.rest_list     = kind == 0 ? ccd_rest_vf.p : ccd_rest_ee.p;
    c.rest_count    = ccd_rest_count.p + kind;
    // first pass: up to 8192 workgroups (pairs run from 1 to 32 ACCD iterations, and smaller
    // workgroup shares of the list balance better: 0.655 ms per tube Newton iteration against
    // 0.67 ms with 4096 and 0.71 ms with one resident round of 1792; 16384 gives the same)
    launch_ccd(c, rest ? std::min(1024u, pair_grid(c.pair_capacity)) : std::max(1u, std::min(8192u, grid_for(c.pair_capacity, 256))), s);
}

// CCD over the last swept broad phase (the "ccd" stage): ground bound, then each kind's passes.
void Solver::ccd()
{
    tic();
    ccd_ground();
    if (prm.use_ccd_linesearch && prm.use_self_collision)
    {
        launch_fill_u32(ccd_rest_count.p, 2, 0u, stream);
        for (int kind = 0; kind < 2; kind++) ccd_pass(kind, false, stream);
        for (int kind = 0; kind < 2; kind++) ccd_pass(kind, true, stream);
    }
    toc("ccd");
}

// The line search's swept broad phase and CCD, interleaved: the vertex-face query and first pass,
// then the vertex-face rest pass on the side stream while the edge tree is refit and queried and
// the edge-edge passes run; the stream waits for the side stream before the step is applied.
// The rest pass is a handful of long ACCD loops (one lane each), which otherwise leave the GPU
// idle; the step bound is a minimum over pairs, so the order of the passes does not change it.
void Solver::swept_ccd()
{
    tic();
    ccd_ground();
    launch_fill_u32(ccd_rest_count.p, 2, 0u, stream);
    toc_part("ccd");
    tic();
    query_faces(true);
    toc_part("broadphase_ccd");
    tic();
    ccd_pass(0, false, stream);
    LCSX_HIP(hipEventRecord(ev_fork, stream));
    LCSX_HIP(hipStreamWaitEvent(side, ev_fork, 0));
    ccd_pass(0, true, side);
    LCSX_HIP(hipEventRecord(ev_join, side));
    toc_part("ccd");
    tic();
    query_edges(true);
    toc("broadphase_ccd");
    tic();
    ccd_pass(1, false, stream);
    ccd_pass(1, true, stream);
    LCSX_HIP(hipStreamWaitEvent(stream, ev_join, 0));
    toc("ccd");
    last_bp = 2;
}

// Grows the pair and contact lists to 1.5x the counts of the last iteration when a count
// exceeded its capacity. Sizes are computed in 64 bits and capped (kMaxPairs, kMaxContacts); a
// count at the device counters' saturation point (kCountCeil) or above a cap is an error, so a
// truncated iteration is never redone with the same capacity.
bool Solver::grow_if_needed(bool ccd_only)
{
    const uint64_t vf = ccd_only ? host_status.n_vf_ccd : std::max(host_status.n_vf, host_status.n_vf_ccd);
    const uint64_t ee = ccd_only ? host_status.n_ee_ccd : std::max(host_status.n_ee, host_status.n_ee_ccd);
    const uint64_t nc = ccd_only ? 0 : host_status.n_contacts;
    if (vf <= cap_vf && ee <= cap_ee && nc <= cap_c) return false;
    const uint64_t nvf = grown_capacity(cap_vf, vf, kMaxPairs), nee = grown_capacity(cap_ee, ee, kMaxPairs),
                   ncc = grown_capacity(cap_c, nc, kMaxContacts);
    if (nvf == 0 || nee == 0 || ncc == 0)
    {
        set_error("candidate pairs (" + std::to_string(vf) + " vertex-face, " + std::to_string(ee) +
                  " edge-edge) or contacts (" + std::to_string(nc) + ") exceed the library's limit of " +
                  std::to_string(kMaxPairs) + " pairs per kind and " + std::to_string(kMaxContacts) + " contacts");
        throw CapacityFailure();
    }
    alloc_collision((uint32_t)nvf, (uint32_t)nee, (uint32_t)ncc);
    return true;
}

// NewtonSolver::line_search, newton_solver.cpp:3685-3884 (CCD step bound, no energy backtracking)
void Solver::line_search()
{
    const SegView g = seg_view(false);
    launch_reset_line_search(status.p, sst.p, S.nscenes, stream);
    launch_apply_dx(S.nv, x_iter.p, dx.p, x.p, nullptr, 1.0f, g, stream);
    rigid_positions();
    ccd_pairs_fresh = prm.use_ccd_linesearch && prm.use_self_collision;
    if (ccd_pairs_fresh) swept_ccd();
    else ccd();
    launch_apply_dx(S.nv, x_iter.p, dx.p, x.p, sst.p, 1.0f, g, stream);
    rigid_positions();
    if (prm.use_energy_linesearch) energy_line_search();
    launch_pin_delta((uint32_t)S.fixed_verts.size(), fixed_ids.p, x.p, x_tilde.p, sst.p, vert_scene_d.p, stream);
}

// Total energy of every scene at the current x (element energies in FP32, barrier terms in FP64
// in the mixed form, sums in double).
std::vector<double> Solver::energy()
{
    EnergyArgs a{};
    a.nv         = S.nv;
    a.x          = x.p;
    a.x_tilde    = x_tilde.p;
    a.mass       = vert_mass.p;
    a.fixed      = is_fixed.p;
    a.row_kind   = row_kind_d.p;
    a.vert_scene = vert_scene_d.p;
    a.offset     = offset.p;
    a.dhat       = dhat.p;
    a.vert_area  = vert_area.p;
    const float h = prm.implicit_dt;
    a.h2inv      = 1.0f / (h * h);
    a.kD         = prm.stiffness_dirichlet;
    a.kappa      = prm.stiffness_collision;
    a.floor_y    = prm.floor_y;
    a.scaling    = prm.bending_scaling;
    a.use_floor  = prm.use_floor;
    a.fp64       = prm.precision >= 1;
    a.quadratic  = prm.contact_energy_type == 0;
    a.nsf        = (uint32_t)(S.sf.size() / 3);
    a.sf         = sf.p;
    a.sf_Dm      = sf_Dm.p;
    a.sf_c       = sf_c.p;
    a.nbh        = (uint32_t)(S.bh.size() / 4);
    a.nsp        = (uint32_t)(S.sp.size() / 2);
    a.sp         = sp.p;
    a.sp_c       = sp_c.p;
    a.bh         = bh.p;
    a.bh_c       = bh_c.p;
    a.nb         = (uint32_t)S.bodies.size();
    a.bodies     = bodies_d.p;
    if (prm.use_self_collision) a.c = contact_view();
    a.out = energy_d.p;
    launch_energy(a, prm.use_self_collision ? pair_grid(cap_c) : 0u, S.nscenes, stream);
    std::vector<double> e(S.nscenes);
    LCSX_HIP(hipMemcpyAsync(e.data(), energy_d.p, e.size() * sizeof(double), hipMemcpyDeviceToHost, stream));
    LCSX_HIP(hipStreamSynchronize(stream));
    return e;
}

// newton_solver.cpp:3803-3856, per scene: scenes still iterating whose |dx| is not below the
// convergence tolerance start from the CCD bound and halve their step while E(alpha) >= E(0) +
// Epsilon, at most 20 times; a step below 1e-4 is a failure (the reference stops with an error).
void Solver::energy_line_search()
{
    tic();
    read_status();
    // a truncated pair or contact list bounded the step with only part of its pairs (the contact
    // energy of an incomplete list may even be infinite): leave the search to the redo of the
    // iteration that newton_iteration starts after growing the lists
    if (host_status.n_vf_ccd > cap_vf || host_status.n_ee_ccd > cap_ee || host_status.n_contacts > cap_c ||
        host_status.n_vf > cap_vf || host_status.n_ee > cap_ee)
    {
        toc("energy_line_search");
        return;
    }
    const uint32_t       ns  = S.nscenes;
    const float          tol = prm.newton_tol * prm.implicit_dt;
    std::vector<float>   alpha(ns);
    std::vector<uint8_t> search(ns, 0);
    bool                 any = false;
    for (uint32_t s = 0; s < ns; s++)
    {
        alpha[s]  = ord2f(host_sst[s].toi_bits);
        search[s] = (active_h.empty() || active_h[s]) &&
                    !(__builtin_bit_cast(float, host_sst[s].maxdx_bits) < tol);
        any       = any || search[s];
    }
    if (!any)
    {
        toc("energy_line_search");
        return;
    }
    const SegView g   = seg_view(false);
    auto          put = [&](const std::vector<float>& al) {
        for (uint32_t s = 0; s < ns; s++) host_sst[s].toi_bits = f2ord(al[s]);
        sst.upload(host_sst, stream);
        launch_apply_dx(S.nv, x_iter.p, dx.p, x.p, sst.p, 1.0f, g, stream);
        rigid_positions();
    };
    std::vector<float> zero = alpha;
    for (uint32_t s = 0; s < ns; s++)
        if (search[s]) zero[s] = 0.0f;
    put(zero);
    const std::vector<double> e0 = energy();
    put(alpha);
    std::vector<double> e = energy();
    for (uint32_t s = 0; s < ns; s++)
        if (search[s] && !std::isfinite(e[s]))
        {
            set_error("energy is not finite in scene " + std::to_string(s));
            throw HipFailure();
        }
    for (int c = 0; c < 20; c++)
    {
        bool more = false;
        for (uint32_t s = 0; s < ns; s++)
        {
            if (!search[s]) continue;
            if (e[s] < e0[s] + (double)kFltEpsilon) { search[s] = 0; continue; }
            alpha[s] *= 0.5f;
            more = true;
        }
        if (!more) break;
        put(alpha);
        e = energy();
        for (uint32_t s = 0; s < ns; s++)
            if (search[s] && alpha[s] < 1e-4f)
            {
                set_error("energy line search failed in scene " + std::to_string(s));
                throw HipFailure();
            }
    }
    toc("energy_line_search");
}

bool Solver::newton_iteration()
{
    iter_begin();
    material();
    update_contacts(true);
    contact_assemble();
    pcg();
    line_search();
    read_status();
    if (host_status.nan)
    {
        set_error("NaN/Inf in the Newton direction");
        throw HipFailure();
    }
    if (grow_if_needed(false))
    {
        // contact lists were truncated: restore the iterate and redo the iteration
        LCSX_HIP(hipMemcpyAsync(x.p, x_iter.p, x.n * sizeof(float), hipMemcpyDeviceToDevice, stream));
        return false;
    }
    std::vector<uint32_t> pin_scene(S.nscenes, 0u);
    for (uint32_t v : S.fixed_verts) pin_scene[S.vert_scene[v]] = 1u;
    for (uint32_t sc = 0; sc < S.nscenes; sc++)
    {
        if (!active_h[sc]) continue;
        lcsx_stats& st = scene_stats[sc];
        st.toi         = ord2f(host_sst[sc].toi_bits);
        st.max_dx      = __builtin_bit_cast(float, host_sst[sc].maxdx_bits);
        st.pin_delta   = pin_scene[sc] ? __builtin_bit_cast(float, host_sst[sc].pin_bits) : -1e9f;
        if (!(st.toi > 0.0f && st.toi <= 1.0f))
        {
            set_error("invalid CCD step bound " + std::to_string(st.toi) + " in scene " + std::to_string(sc));
            throw HipFailure();
        }
    }
    stats.num_pairs_vf = (int)(dcd_reused ? host_status.n_vf_ccd : host_status.n_vf);
    stats.num_pairs_ee = (int)(dcd_reused ? host_status.n_ee_ccd : host_status.n_ee);
    stats.num_contacts = (int)host_status.n_contacts;
    stats.num_ccd_pairs = (int)std::min<uint64_t>((uint64_t)host_status.n_vf_ccd + host_status.n_ee_ccd, INT32_MAX);
    for (uint32_t sc = 0; sc < S.nscenes; sc++)
        if (active_h[sc]) scene_stats[sc].toi_min = std::min(scene_stats[sc].toi_min, scene_stats[sc].toi);
    if (timing)
    {
        // counts per Newton iteration beside the kernel groups' times (pairs/s of the narrow phases)
        auto add = [&](const char* k, double v) {
            auto& t = times[k];
            t.first += v;
            t.second += 1;
        };
        add("pairs_ccd", (double)host_status.n_vf_ccd + (double)host_status.n_ee_ccd);
        add("pairs_dcd", (double)stats.num_pairs_vf + (double)stats.num_pairs_ee);
        add("contacts", (double)host_status.n_contacts);
    }
    stats.broadphase_overflow |= host_status.overflow ? 1 : 0;
    fold_stats();
    return true;
}

void Solver::newton_iteration_until_done()
{
    for (int redo = 0; !newton_iteration(); redo++)
        if (redo >= 8)
        {
            // every redo follows a growth of at least 1.5x from the same start state
            set_error("the Newton iteration kept overflowing its pair lists after 8 growths");
            throw CapacityFailure();
        }
}

// NewtonSolver::device_post_dist_check (newton_solver.cpp:3364-3375): the reference runs the DCD at
// the step's positions and stops on a pair closer than its offsets. Here the DCD broad phase at
// the final positions gives the candidate pairs (every pair with d < offsets + d_hat is one), and
// k_gap_check takes the smallest FP64 gap d - (offset_a + offset_b) over them and over the ground,
// per scene, with the count of pairs at or below zero, into the scene's statistics.
void Solver::post_dist_check()
{
    tic();
    launch_reset_gap(gap.p, S.nscenes, stream);
    GapArgs g{};
    g.x          = x.p;
    g.faces      = faces.p;
    g.edges      = edges.p;
    g.offset     = offset.p;
    g.vert_scene = vert_scene_d.p;
    g.vert_body  = vert_body_d.p;
    g.fixed      = is_fixed.p;
    g.row_kind   = row_kind_d.p;
    g.floor_y    = prm.floor_y;
    g.out        = gap.p;
    if (prm.use_self_collision)
    {
        for (int tries = 0;; tries++)
        {
            launch_reset_status(status.p, sst.p, S.nscenes, stream);
            broad_phase(false);
            read_status();
            if (!grow_if_needed(false)) break;
            if (tries >= 8)
            {
                set_error("the post-step broad phase kept overflowing its pair lists");
                throw CapacityFailure();
            }
        }
        g.kind          = 0;
        g.pairs         = pairs_vf.p;
        g.pair_count    = &status.p->n_vf;
        g.pair_capacity = cap_vf;
        launch_gap_check(g, pair_grid(cap_vf), stream);
        g.kind          = 1;
        g.pairs         = pairs_ee.p;
        g.pair_count    = &status.p->n_ee;
        g.pair_capacity = cap_ee;
        launch_gap_check(g, pair_grid(cap_ee), stream);
    }
    if (prm.use_floor)
    {
        g.kind = 2;
        g.nv   = S.nv;
        launch_gap_check(g, pair_grid(S.nv), stream);
    }
    std::vector<GapStatus> h(S.nscenes);
    LCSX_HIP(hipMemcpyAsync(h.data(), gap.p, h.size() * sizeof(GapStatus), hipMemcpyDeviceToHost, stream));
    LCSX_HIP(hipStreamSynchronize(stream));
    toc("post_dist_check");
    double   mg  = INFINITY;
    int64_t  pen = 0, chk = 0;
    for (uint32_t sc = 0; sc < S.nscenes; sc++)
    {
        lcsx_stats& st     = scene_stats[sc];
        st.min_gap         = h[sc].n_checked ? ord2d(h[sc].min_key) : INFINITY;
        st.num_penetrating = (int)h[sc].n_pen;
        st.gap_pairs       = (int)h[sc].n_checked;
        mg                 = std::min(mg, st.min_gap);
        pen += h[sc].n_pen;
        chk += h[sc].n_checked;
    }
    stats.min_gap         = mg;
    stats.num_penetrating = (int)std::min<int64_t>(pen, INT32_MAX);
    stats.gap_pairs       = (int)std::min<int64_t>(chk, INT32_MAX);
}

// Batch totals into stats: sums of the per-scene iteration counts, the smallest step bound and the
// largest |dx| and pin distance of the scenes still iterating (one scene: that scene's values).
void Solver::fold_stats()
{
    int   pcg_last = 0, pcg_total = 0, newton = 0, conv = 1;
    float toi = 1.0f, mdx = 0.0f, pin = -1e9f, rel = 0.0f, toi_min = 1.0f;
    for (uint32_t sc = 0; sc < S.nscenes; sc++)
    {
        const lcsx_stats& st = scene_stats[sc];
        pcg_total += st.pcg_iters_total;
        newton += st.newton_iters;
        conv = conv && st.converged;
        toi_min = std::min(toi_min, st.toi_min);
        if (!active_h.empty() && !active_h[sc]) continue;
        pcg_last = std::max(pcg_last, st.pcg_iters);
        toi      = std::min(toi, st.toi);
        mdx      = std::max(mdx, st.max_dx);
        pin      = std::max(pin, st.pin_delta);
        rel      = std::max(rel, st.pcg_rel);
    }
    stats.pcg_iters       = pcg_last;
    stats.pcg_iters_total = pcg_total;
    stats.pcg_rel         = rel;
    stats.toi             = toi;
    stats.toi_min         = toi_min;
    stats.max_dx          = mdx;
    stats.pin_delta       = pin;
    stats.newton_iters    = newton;
    stats.converged       = conv;
    stats.pcg_rz_true     = rz_true;
}

void Solver::frame_end()
{
    float h = prm.implicit_dt;
    launch_frame_end(S.nv, x_step.p, x.p, v.p, h, std::exp(-prm.damping_cloth * h), stream);
    frame += 1;
    stats.frame = frame;
}

// physics_step_GPU (newton_solver.cpp:4051-4345), each scene of the batch with its own Newton
// loop: a scene stops on `converged || (iter >= nonlinear_iter_count && dirichlet)` or at the
// iteration cap; stopped scenes keep their positions (their step is 0) while the others iterate.
void Solver::step()
{
    frame_begin();
    predict();
    const uint32_t       ns = S.nscenes;
    std::vector<uint8_t> conv(ns, 0), dir(ns, 0);
    active_h.assign(ns, 1);
    for (auto& st : scene_stats)
    {
        st.pcg_iters_total     = 0;
        st.broadphase_overflow = 0;
        st.newton_iters        = 0;
        st.converged           = 0;
        st.min_gap             = NAN;  // until post_dist_check runs
        st.num_penetrating     = -1;
        st.gap_pairs           = -1;
        st.toi_min             = 1.0f;
    }
    stats.broadphase_overflow = 0;
    stats.min_gap             = NAN;
    stats.num_penetrating     = -1;
    stats.gap_pairs           = -1;
    int it = 0;
    for (it = 0; it < prm.newton_max_iters; it++)
    {
        bool any = false;
        for (uint32_t sc = 0; sc < ns; sc++)
        {
            if (!active_h[sc]) continue;
            if (conv[sc] || (it >= prm.nonlinear_iter_count && dir[sc]))
            {
                active_h[sc]                 = 0;
                scene_stats[sc].newton_iters = it;
            }
            else
                any = true;
        }
        if (!any) break;
        active_d.upload(active_h, stream);
        newton_iteration_until_done();
        for (uint32_t sc = 0; sc < ns; sc++)
        {
            if (!active_h[sc]) continue;
            const lcsx_stats& st = scene_stats[sc];
            if (st.max_dx < prm.newton_tol * prm.implicit_dt)
                conv[sc] = dir[sc] = 1;
            else
            {
                conv[sc] = 0;
                dir[sc]  = st.pin_delta < 1e-3f;
            }
        }
    }
    for (uint32_t sc = 0; sc < ns; sc++)
    {
        if (active_h[sc]) scene_stats[sc].newton_iters = it;
        scene_stats[sc].converged = conv[sc];
    }
    active_h.assign(ns, 1);  // every scene's stats count in the totals
    active_d.upload(active_h, stream);
    fold_stats();
    if (prm.post_dist_check) post_dist_check();
    frame_end();
    for (auto& st : scene_stats) st.frame = frame;
    LCSX_HIP(hipStreamSynchronize(stream));
}

void Solver::rigid_positions()
{
    if (!S.bodies.empty())
        launch_rigid_positions(S.nv, row_kind_d.p, vert_body_d.p, bodies_d.p, body_X_d.p, x.p, stream);
}

void Solver::spmv_dx(bool lp)
{
    launch_spmv(lp && prm.precision >= 1 ? sell_view_lp() : sell_view(), contact_view(), vert_contacts(),
                pair_grid(cap_c), dx.p, spmv_tmp.p, S.nv, stream);
    LCSX_HIP(hipMemcpyAsync(dx.p, spmv_tmp.p, dx.n * sizeof(float), hipMemcpyDeviceToDevice, stream));
}

// Times the runtime mappings on the current state and keeps the fastest of each: the CCD
// first-pass budget (iterations per pair before a pair moves to the full-budget pass), the PCG
// launch mode (direct or captured graphs), with one scene the form of the contact t_c kernel (one
// thread per contact or per slot chunk), the SpMV mapping and the broad-phase traversal shape.
// None of them changes a result: the step bound is a minimum over the same pairs, and the PCG
// runs the same arithmetic. The PCG's settings are those of its launches and are timed as launches, also
// where the present system would run in one: they are for the solves that do not fit it, and choosing
// them leaves that rule as it is. The state
// (positions, velocities, statistics, timings) is restored afterwards.
std::string Solver::autotune()
{
    DBuf<float> sx, sv;
    sx.alloc(x.n);
    sv.alloc(v.n);
    LCSX_HIP(hipMemcpyAsync(sx.p, x.p, x.n * sizeof(float), hipMemcpyDeviceToDevice, stream));
    LCSX_HIP(hipMemcpyAsync(sv.p, v.p, v.n * sizeof(float), hipMemcpyDeviceToDevice, stream));
    const auto saved_times = times;
    const auto saved_stats = stats;
    const auto saved_scene = scene_stats;
    const bool saved_timing = timing;
    const int  saved_spmv   = spmv_sample;
    timing      = false;
    spmv_sample = 0;
    hipEvent_t e0, e1;
    LCSX_HIP(hipEventCreate(&e0));
    LCSX_HIP(hipEventCreate(&e1));
    auto time_ms = [&](auto&& fn, int reps) {
        std::vector<float> t;
        for (int r = 0; r < reps; r++)
        {
            LCSX_HIP(hipEventRecord(e0, stream));
            fn();
            LCSX_HIP(hipEventRecord(e1, stream));
            LCSX_HIP(hipEventSynchronize(e1));
            float ms = 0.0f;
            LCSX_HIP(hipEventElapsedTime(&ms, e0, e1));
            t.push_back(ms);
        }
        std::sort(t.begin(), t.end());
        return t[t.size() / 2];
    };
    std::string out;
    char        buf[160];
    // a Newton system at the current state
    active_h.assign(S.nscenes, 1);
    active_d.upload(active_h, stream);
    frame_begin();
    predict();
    iter_begin();
    material();
    launch_reset_status(status.p, sst.p, S.nscenes, stream);
    update_contacts(false);
    read_status();
    if (grow_if_needed(false))
    {
        launch_reset_status(status.p, sst.p, S.nscenes, stream);
        update_contacts(false);
    }
    contact_assemble();
    struct Launched  // launches only, while this lives
    {
        bool&      flag;
        const bool was;
        explicit Launched(bool& f) : flag(f), was(f) { f = false; }
        ~Launched() { flag = was; }
    };
    std::optional<Launched> launched(std::in_place, pcg_grid);
    // PCG: launch mode x contact t_c form. A candidate replaces the current setting only when it
    // is faster by more than kTuneMargin (timings repeat to within ~2%)
    constexpr float kTuneMargin = 0.97f;
    float best = 1e30f, cur = 1e30f;
    bool  bg = use_graphs, bc = contact_t_per_contact;
    const bool g0 = use_graphs, c0 = contact_t_per_contact;
    for (int graphs = 0; graphs < 2; graphs++)
        for (int per_contact = 1; per_contact >= (S.nscenes == 1 ? 0 : 1); per_contact--)
        {
            use_graphs            = graphs != 0;
            contact_t_per_contact = per_contact != 0;
            pcg();  // first run: captures graphs, warms caches
            const float ms = time_ms([&] { pcg(); }, 3);
            std::snprintf(buf, sizeof(buf), "pcg[graphs=%d,per_contact=%d]=%.4f;", graphs, per_contact, ms);
            out += buf;
            if (use_graphs == g0 && contact_t_per_contact == c0) cur = ms;
            if (ms < best)
            {
                best = ms;
                bg   = use_graphs;
                bc   = contact_t_per_contact;
            }
        }
    // captured graphs must win by more: the three timed replays do not see the captures that new
    // contact-slot grids cost later (0.35 ms each), nor the grid rounded up to a power of two
    constexpr float kGraphMargin = 0.95f;
    const bool pcg_change = best < (bg && !g0 ? kGraphMargin : kTuneMargin) * cur;
    use_graphs            = pcg_change ? bg : g0;
    contact_t_per_contact = pcg_change ? bc : c0;
    // the SpMV mapping, under the chosen launch mode (chunk order matters only with contacts)
    {
        best         = 1e30f;
        cur          = 1e30f;
        const int s0 = spmv_shape;
        int       sb = spmv_shape;
        for (int shape = 0; shape < kSpmvShapes; shape++)
        {
            spmv_shape = shape;
            pcg();
            const float ms = time_ms([&] { pcg(); }, 3);
            std::snprintf(buf, sizeof(buf), "pcg[spmv=%d]=%.4f;", shape, ms);
            out += buf;
            if (shape == s0) cur = ms;
            if (ms < best)
            {
                best = ms;
                sb   = shape;
            }
        }
        spmv_shape = best < kTuneMargin * cur ? sb : s0;
    }
    launched.reset();
    pcg();
    // line search: CCD first-pass budget
    if (prm.use_ccd_linesearch && prm.use_self_collision)
    {
        best         = 1e30f;
        cur          = 1e30f;
        const int b0 = ccd_budget;
        int       bb = ccd_budget;
        for (int budget : {8, 16, 32, 64, 128})
        {
            ccd_budget = budget;
            line_search();
            read_status();
            if (grow_if_needed(true)) line_search();
            const float ms = time_ms([&] { line_search(); }, 3);
            std::snprintf(buf, sizeof(buf), "line_search[ccd_budget=%d]=%.4f;", budget, ms);
            out += buf;
            if (budget == b0) cur = ms;
            if (ms < best)
            {
                best = ms;
                bb   = budget;
            }
        }
        ccd_budget = best < kTuneMargin * cur ? bb : b0;
        // the swept broad phase's traversal shape (LDS stack entries, pair staging). The shapes that walk the
        // solver's own hierarchies are one code path here: one of them is timed, so that noise picks none
        best         = 1e30f;
        cur          = 1e30f;
        const int v0 = query_variant;
        int       vb = query_variant;
        const int vc = query_by_clusters(v0) ? v0 : kQueryDefault;
        for (int v = 0; v < kQueryVariants; v++)
        {
            if (query_by_clusters(v) && v != vc) continue;
            query_variant = v;
            line_search();
            read_status();
            if (grow_if_needed(true)) line_search();
            const float ms = time_ms([&] { line_search(); }, 3);
            std::snprintf(buf, sizeof(buf), "line_search[query=%d]=%.4f;", v, ms);
            out += buf;
            if (v == v0) cur = ms;
            if (ms < best)
            {
                best = ms;
                vb   = v;
            }
        }
        query_variant = best < kTuneMargin * cur ? vb : v0;
    }
    std::snprintf(buf, sizeof(buf), "chosen:ccd_budget=%d,graphs=%d,per_contact=%d,spmv=%d,query=%d", ccd_budget,
                  use_graphs ? 1 : 0, contact_t_per_contact ? 1 : 0, spmv_shape, query_variant);
    out += buf;
    // restore the state
    LCSX_HIP(hipMemcpyAsync(x.p, sx.p, x.n * sizeof(float), hipMemcpyDeviceToDevice, stream));
    LCSX_HIP(hipMemcpyAsync(v.p, sv.p, v.n * sizeof(float), hipMemcpyDeviceToDevice, stream));
    LCSX_HIP(hipStreamSynchronize(stream));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    ccd_pairs_fresh = false;
    vc_ready        = false;
    timing          = saved_timing;
    spmv_sample     = saved_spmv;
    times           = saved_times;
    stats           = saved_stats;
    scene_stats     = saved_scene;
    return out;
}

}  // namespace lcsx
