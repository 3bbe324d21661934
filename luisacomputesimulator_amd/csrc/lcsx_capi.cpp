// extern "C" boundary of the lcsx library (declared in include/lcsx.h).
#include <algorithm>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <sstream>
#include <exception>
#include <string>
#include "lcsx_io.h"
#include "lcsx_solver.h"

namespace lcsx
{
static thread_local std::string g_err;
void set_error(const std::string& msg) { g_err = msg; }
}  // namespace lcsx

using namespace lcsx;

#define LCSX_GUARD(body)                                                                                    \
    try                                                                                                     \
    {                                                                                                       \
        body                                                                                                \
    }                                                                                                       \
    catch (const HipFailure&)                                                                               \
    {                                                                                                       \
        return g_err.find("NaN") != std::string::npos ? LCSX_ERR_NAN : LCSX_ERR_HIP;                        \
    }                                                                                                       \
    catch (const NoDevice&)                                                                                 \
    {                                                                                                       \
        return LCSX_ERR_NO_GPU;                                                                             \
    }                                                                                                       \
    catch (const CapacityFailure&)                                                                          \
    {                                                                                                       \
        return LCSX_ERR_CAPACITY;                                                                           \
    }                                                                                                       \
    catch (const std::exception& e)                                                                         \
    {                                                                                                       \
        set_error(e.what());                                                                                \
        return LCSX_ERR_ARG;                                                                                \
    }

struct lcsx_solver
{
    Solver   s;
    uint32_t cur_scene = 0;  // scene of the meshes added next
};
struct lcsx_lbvh
{
    Lbvh        t;
    hipStream_t last  = nullptr;
    int         shape = kQueryDefault;
    bool        constructed = false, refitted = false;  // (what comes before has nothing to read)
};

namespace
{
lcsx_status arg_error(const char* m)
{
    set_error(m);
    return LCSX_ERR_ARG;
}

// Host copy of a named solver buffer in the canonical layout.
struct Blob
{
    std::vector<uint8_t> bytes;
    size_t               count = 0;
    template <class T>
    void set(const std::vector<T>& v)
    {
        bytes.resize(v.size() * sizeof(T));
        if (!v.empty()) std::memcpy(bytes.data(), v.data(), bytes.size());
        count = v.size();
    }
};

template <class T>
std::vector<T> dl(const DBuf<T>& b, size_t n, hipStream_t s)
{
    std::vector<T> h(n);
    b.download(h.data(), n, s);
    LCSX_HIP(hipStreamSynchronize(s));
    return h;
}

std::vector<float> planes_to_rows(const std::vector<float>& P, size_t n)
{
    std::vector<float> o(9 * n);
    for (size_t i = 0; i < n; i++)
        for (int c = 0; c < 9; c++) o[9 * i + c] = P[c * n + i];
    return o;
}

bool read_tree(const Lbvh& t, const std::string& f, hipStream_t s, Blob& out)
{
    size_t n = t.n, nn = t.n_nodes();
    if (f == "morton_sorted") out.set(dl(t.morton_sorted, n, s));
    else if (f == "sorted_to_orig")
    {
        std::vector<uint32_t> h(n);
        if (n) LCSX_HIP(hipMemcpyAsync(h.data(), t.sorted_to_orig, n * 4, hipMemcpyDeviceToHost, s));
        LCSX_HIP(hipStreamSynchronize(s));
        out.set(h);
    }
    else if (f == "parent") out.set(dl(t.parent, nn, s));
    else if (f == "object_idx") out.set(dl(t.object_idx, nn, s));
    else if (f == "children")
    {
        auto                  c = dl(t.children, nn, s);
        std::vector<uint32_t> h(2 * nn);
        for (size_t i = 0; i < nn; i++)
        {
            h[2 * i]     = c[i].x;
            h[2 * i + 1] = c[i].y;
        }
        out.set(h);
    }
    else if (f == "node_aabb")
    {
        auto               b = dl(t.nodes, nn, s);
        std::vector<float> h(6 * nn);
        for (size_t i = 0; i < nn; i++)
        {
            float v[6] = {b[i].lo.x, b[i].lo.y, b[i].lo.z, b[i].hi.x, b[i].hi.y, b[i].hi.z};
            std::memcpy(&h[6 * i], v, sizeof(v));
        }
        out.set(h);
    }
    else if (f == "global_aabb")
    {
        auto               g = dl(t.gbox, 6 * (size_t)t.nseg, s);
        std::vector<float> h(g.size());
        for (size_t k = 0; k < g.size(); k++) h[k] = ord2f(g[k]);
        out.set(h);
    }
    else
        return false;
    return true;
}

// Buffers produced by the host setup alone (readable after init even without a GPU).
bool is_static_buffer(const std::string& n)
{
    static const char* k[] = {"rest_x", "faces", "edges", "hinges", "csr", "stretch_faces", "bending_hinges",
                              "fixed_verts", "is_fixed", "face_area", "edge_area", "vert_area", "vert_mass", "offset",
                              "dhat", "sf_Dm", "sf_area", "sf_mu", "sf_lambda", "bh_angle", "bh_hbar", "bh_k",
                              "stretch_springs", "sp_rest", "sp_k", "cluster_use"};
    for (const char* c : k)
        if (n == c) return true;
    return false;
}

bool read_named(Solver& S, const std::string& name, Blob& out)
{
    hipStream_t s  = S.stream;
    size_t      nv = S.S.nv;
    auto        v3 = [&](const DBuf<float>& b) { out.set(dl(b, 3 * nv, s)); return true; };
    if (name == "x") return v3(S.x);
    if (name == "v") return v3(S.v);
    if (name == "x_step") return v3(S.x_step);
    if (name == "x_iter") return v3(S.x_iter);
    if (name == "x_tilde") return v3(S.x_tilde);
    if (name == "dx") return v3(S.dx);
    if (name == "cgB") return v3(S.cgB);
    if (name == "rest_x") { out.set(S.S.rest_x); return true; }
    if (name == "diag") { out.set(planes_to_rows(dl(S.diag, 9 * nv, s), nv)); return true; }
    if (name == "offdiag")
    {
        auto               P = dl(S.sell_val, 9 * (size_t)S.S.nblocks, s);
        std::vector<float> o(9 * S.S.csr.size(), 0.0f);
        for (size_t k = 0; k < S.S.csr.size(); k++)
        {
            uint32_t b = S.S.csr_to_sell[k];
            if (b == 0xffffffffu) continue;
            for (int c = 0; c < 9; c++) o[9 * k + c] = P[(size_t)c * S.S.nblocks + b];
        }
        out.set(o);
        return true;
    }
    if (name == "faces") { out.set(S.S.faces); return true; }
    if (name == "edges") { out.set(S.S.edges); return true; }
    if (name == "cluster_use")
    {
        out.set(std::vector<uint32_t>{S.S.cluster_f_use, S.S.cluster_e_use});
        return true;
    }
    if (name == "hinges") { out.set(S.S.hinges); return true; }
    if (name == "csr") { out.set(S.S.csr); return true; }
    if (name == "stretch_faces") { out.set(S.S.sf); return true; }
    if (name == "bending_hinges") { out.set(S.S.bh); return true; }
    if (name == "stretch_springs") { out.set(S.S.sp); return true; }
    if (name == "sp_rest") { out.set(S.S.sp_rest); return true; }
    if (name == "sp_k") { out.set(S.S.sp_k); return true; }
    if (name == "fixed_verts") { out.set(S.S.fixed_verts); return true; }
    if (name == "is_fixed") { out.set(S.S.is_fixed); return true; }
    if (name == "face_area") { out.set(S.S.face_area); return true; }
    if (name == "edge_area") { out.set(S.S.edge_area); return true; }
    if (name == "vert_area") { out.set(S.S.vert_area); return true; }
    if (name == "vert_mass") { out.set(S.S.vert_mass); return true; }
    if (name == "offset") { out.set(S.S.offset); return true; }
    if (name == "dhat") { out.set(S.S.dhat); return true; }
    if (name == "sf_Dm") { out.set(S.S.sf_Dm); return true; }
    if (name == "sf_area") { out.set(S.S.sf_area); return true; }
    if (name == "sf_mu") { out.set(S.S.sf_mu); return true; }
    if (name == "sf_lambda") { out.set(S.S.sf_lambda); return true; }
    if (name == "bh_angle") { out.set(S.S.bh_angle); return true; }
    if (name == "bh_hbar") { out.set(S.S.bh_hbar); return true; }
    if (name == "bh_k") { out.set(S.S.bh_k); return true; }
    if (name == "face_stage") { out.set(dl(S.face_stage, S.face_stage.n, s)); return true; }
    if (name == "toi")
    {
        S.read_status();
        std::vector<float> t(S.S.nscenes);
        for (uint32_t k = 0; k < S.S.nscenes; k++) t[k] = ord2f(S.host_sst[k].toi_bits);
        out.set(t);
        return true;
    }
    if (name.rfind("face_tree.", 0) == 0) return read_tree(S.tree_face, name.substr(10), s, out);
    if (name.rfind("edge_tree.", 0) == 0) return read_tree(S.tree_edge, name.substr(10), s, out);
    if (name == "pairs_vf" || name == "pairs_ee")
    {
        S.read_status();
        bool     vf = name == "pairs_vf";
        uint32_t n  = S.last_bp == 2 ? (vf ? S.host_status.n_vf_ccd : S.host_status.n_ee_ccd)
                                     : (S.last_bp == 1 ? (vf ? S.host_status.n_vf : S.host_status.n_ee) : 0u);
        n = std::min(n, vf ? S.cap_vf : S.cap_ee);
        out.set(dl(vf ? S.pairs_vf : S.pairs_ee, 2 * (size_t)n, s));
        return true;
    }
    if (name == "energy")
    {
        // total energy of each scene at the current x, over the current contact list (doubles)
        out.set(S.energy());
        return true;
    }
    if (name == "ccd_rest_vf" || name == "ccd_rest_ee")
    {
        // the candidate pairs of the last line search whose ACCD ran past the first pass's budget
        const bool vf    = name == "ccd_rest_vf";
        auto       cnt   = dl(S.ccd_rest_count, 2, s);
        uint32_t   n     = std::min(cnt[vf ? 0 : 1], vf ? S.cap_vf : S.cap_ee);
        auto       ids   = dl(vf ? S.ccd_rest_vf : S.ccd_rest_ee, n, s);
        auto       pairs = dl(vf ? S.pairs_vf : S.pairs_ee, 2 * (size_t)(vf ? S.cap_vf : S.cap_ee), s);
        std::vector<uint32_t> o(2 * (size_t)n);
        for (uint32_t k = 0; k < n; k++)
        {
            o[2 * k]     = pairs[2 * (size_t)ids[k]];
            o[2 * k + 1] = pairs[2 * (size_t)ids[k] + 1];
        }
        out.set(o);
        return true;
    }
    if (name == "contact_triplets" || name == "contact_triplet_blocks")
    {
        const uint32_t m = S.contact_triplets();
        if (name == "contact_triplets") out.set(dl(S.ctb.out_rc, 2 * (size_t)m, s));
        else out.set(dl(S.ctb.out_blk, 9 * (size_t)m, s));
        return true;
    }
    if (name.rfind("contact_", 0) == 0)
    {
        S.read_status();
        size_t n   = std::min(S.host_status.n_contacts, S.cap_c);
        auto   idx = dl(S.c_idx, n, s);
        auto   nk  = dl(S.c_nk, n, s);
        auto   w   = dl(S.c_w, n, s);
        auto   ax  = dl(S.c_aux, n, s);
        if (name == "contact_idx")
        {
            std::vector<uint32_t> h(4 * n);
            for (size_t i = 0; i < n; i++)
            {
                h[4 * i] = idx[i].x & 0x7fffffffu;
                h[4 * i + 1] = idx[i].y & 0x7fffffffu;
                h[4 * i + 2] = idx[i].z & 0x7fffffffu;
                h[4 * i + 3] = idx[i].w & 0x7fffffffu;
            }
            out.set(h);
        }
        else if (name == "contact_type")
        {
            std::vector<uint32_t> h(n);
            for (size_t i = 0; i < n; i++) h[i] = (idx[i].z & 0x80000000u) ? 4u : 8u;
            out.set(h);
        }
        else if (name == "contact_n")
        {
            std::vector<float> h(3 * n);
            for (size_t i = 0; i < n; i++) { h[3 * i] = nk[i].x; h[3 * i + 1] = nk[i].y; h[3 * i + 2] = nk[i].z; }
            out.set(h);
        }
        else if (name == "contact_k")
        {
            std::vector<float> h(3 * n);
            for (size_t i = 0; i < n; i++) { h[3 * i] = ax[i].x; h[3 * i + 1] = nk[i].w; h[3 * i + 2] = ax[i].y; }
            out.set(h);
        }
        else if (name == "contact_w")
        {
            std::vector<float> h(4 * n);
            for (size_t i = 0; i < n; i++) { h[4 * i] = w[i].x; h[4 * i + 1] = w[i].y; h[4 * i + 2] = w[i].z; h[4 * i + 3] = w[i].w; }
            out.set(h);
        }
        else if (name == "contact_bary")
        {
            std::vector<float> h(2 * n);
            for (size_t i = 0; i < n; i++) { h[2 * i] = ax[i].z; h[2 * i + 1] = ax[i].w; }
            out.set(h);
        }
        else
            return false;
        return true;
    }
    return false;
}
}  // namespace

extern "C"
{
const char* lcsx_last_error(void) { return g_err.c_str(); }
const char* lcsx_version(void) { return "lcsx 0.1 (gfx950)"; }
int         lcsx_device_count(void)
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

void lcsx_params_default(lcsx_params* p)
{
    std::memset(p, 0, sizeof(*p));
    p->implicit_dt          = 1.0f / 60.0f;
    p->nonlinear_iter_count = 3;
    p->newton_max_iters     = 100;
    p->pcg_iter_count       = 100;
    p->pcg_check_every      = 25;
    p->pcg_rel_tol          = 0.0f;
    p->pcg_abs_tol          = 1e-10f;
    p->gravity[1]           = -9.8f;
    p->use_floor            = 1;
    p->use_self_collision   = 1;
    p->use_ccd_linesearch   = 1;
    p->floor_y              = 0.0f;
    p->stiffness_collision  = 1e7f;
    p->stiffness_dirichlet  = 1e9f;
    p->damping_cloth        = 2.0f;
    p->bending_scaling      = 1.0f;
    p->newton_tol           = 1e-2f;
    p->precision            = 0;
    p->use_energy_linesearch = 0;
    p->contact_energy_type   = 1;
    p->post_dist_check       = 1;
}
void lcsx_material_default(lcsx_material* m)
{
    m->thickness              = 2e-3f;
    m->youngs_modulus         = 1e5f;
    m->poisson_ratio          = 0.25f;
    m->area_bending_stiffness = 5e-3f;
    m->density                = 1e3f;
    m->mass                   = 0.0f;
    m->d_hat                  = 2e-3f;
    m->body                   = 0;
    m->rigid_stiffness        = 1e6f;
    m->stretch_spring         = 0;
}

lcsx_status lcsx_solver_create(const lcsx_params* params, int device, lcsx_solver** out)
{
    if (!out) return arg_error("out is NULL");
    if (params && (params->precision < 0 || params->precision > 2))
        return arg_error("precision must be 0 (FP32), 1 (mixed, FP16 blocks) or 2 (mixed, BF16 blocks)");
    if (params && (params->contact_energy_type < 0 || params->contact_energy_type > 1))
        return arg_error("contact_energy_type must be 0 (quadratic) or 1 (log barrier)");
    auto* h = new lcsx_solver();
    if (params) h->s.prm = *params;
    else lcsx_params_default(&h->s.prm);
    h->s.device = device;
    *out        = h;
    return LCSX_OK;
}
lcsx_status lcsx_solver_destroy(lcsx_solver* s)
{
    delete s;
    return LCSX_OK;
}

lcsx_status lcsx_solver_add_mesh(lcsx_solver* s, const float* verts, int n_verts, const int32_t* tris, int n_tris,
                                 const lcsx_material* material, int* mesh_id)
{
    if (!s || !verts || !tris || n_verts <= 0 || n_tris <= 0) return arg_error("invalid mesh arguments");
    if (s->s.inited) { set_error("add_mesh after init"); return LCSX_ERR_STATE; }
    for (int i = 0; i < 3 * n_tris; i++)
        if (tris[i] < 0 || tris[i] >= n_verts) return arg_error("triangle index out of range");
    MeshDesc m;
    m.x.assign(verts, verts + 3 * (size_t)n_verts);
    m.tris.assign(tris, tris + 3 * (size_t)n_tris);
    if (material) m.mat = *material;
    else lcsx_material_default(&m.mat);
    m.scene = s->cur_scene;
    s->s.meshes.push_back(std::move(m));
    if (mesh_id) *mesh_id = (int)s->s.meshes.size() - 1;
    return LCSX_OK;
}

lcsx_status lcsx_solver_add_fixed_points(lcsx_solver* s, int mesh_id, int method, float range, const lcsx_fixed_anim* anim,
                                         int* num_selected)
{
    if (!s || mesh_id < 0 || mesh_id >= (int)s->s.meshes.size()) return arg_error("invalid mesh id");
    if (s->s.inited) { set_error("add_fixed_points after init"); return LCSX_ERR_STATE; }
    if (method < 0 || method > 21 || method == 1 || method == 2) return arg_error("unsupported fixed-point method");
    lcsx_fixed_anim a{};
    a.scale[0] = a.scale[1] = a.scale[2] = 1.0f;
    a.rot_axis[0] = 1.0f;
    if (anim) a = *anim;
    MeshDesc& m  = s->s.meshes[mesh_id];
    size_t    n0 = m.pinned.size();
    pin_by_method(m, method, range, a);
    if (num_selected) *num_selected = (int)(m.pinned.size() - n0);
    return LCSX_OK;
}

lcsx_status lcsx_solver_load_scene_json(lcsx_solver* s, const char* json_path, const char* mesh_dir)
{
    if (!s || !json_path) return arg_error("invalid arguments");
    if (s->s.inited) { set_error("load_scene_json after init"); return LCSX_ERR_STATE; }
    std::string err;
    const size_t first = s->s.meshes.size();
    if (!load_scene_json(json_path, mesh_dir ? mesh_dir : "", s->s.prm, s->s.meshes, err))
    {
        set_error(err);
        return LCSX_ERR_IO;
    }
    for (size_t k = first; k < s->s.meshes.size(); k++) s->s.meshes[k].scene = s->cur_scene;
    return LCSX_OK;
}

lcsx_status lcsx_solver_begin_scene(lcsx_solver* s, int* scene_id)
{
    if (!s) return arg_error("solver is NULL");
    if (s->s.inited) { set_error("begin_scene after init"); return LCSX_ERR_STATE; }
    if (!s->s.meshes.empty() && s->s.meshes.back().scene == s->cur_scene) s->cur_scene++;
    if (scene_id) *scene_id = (int)s->cur_scene;
    return LCSX_OK;
}

int lcsx_solver_num_scenes(lcsx_solver* s) { return s && (s->s.inited || s->s.setup_ready) ? (int)s->s.S.nscenes : 0; }

lcsx_status lcsx_solver_scene_range(lcsx_solver* s, int scene, int* first_vertex, int* num_verts)
{
    if (!s || !(s->s.inited || s->s.setup_ready) || scene < 0 || scene >= (int)s->s.S.nscenes)
        return arg_error("invalid scene");
    if (first_vertex) *first_vertex = (int)s->s.S.sc_v0[scene];
    if (num_verts) *num_verts = (int)(s->s.S.sc_v0[scene + 1] - s->s.S.sc_v0[scene]);
    return LCSX_OK;
}

lcsx_status lcsx_solver_get_scene_stats(lcsx_solver* s, int scene, lcsx_stats* out)
{
    if (!s || !out || !s->s.inited || scene < 0 || scene >= (int)s->s.scene_stats.size())
        return arg_error("invalid scene");
    *out = s->s.scene_stats[scene];
    out->num_pairs_vf = s->s.stats.num_pairs_vf;
    out->num_pairs_ee = s->s.stats.num_pairs_ee;
    out->num_contacts = s->s.stats.num_contacts;
    out->pcg_rz_true  = s->s.stats.pcg_rz_true;
    return LCSX_OK;
}

lcsx_status lcsx_solver_init(lcsx_solver* s)
{
    if (!s) return arg_error("solver is NULL");
    if (s->s.meshes.empty()) { set_error("no meshes"); return LCSX_ERR_STATE; }
    LCSX_GUARD(s->s.init(); return LCSX_OK;)
}

lcsx_status lcsx_solver_step(lcsx_solver* s, int frames)
{
    if (!s || frames < 0) return arg_error("invalid arguments");
    if (!s->s.inited) { set_error("step before init"); return LCSX_ERR_STATE; }
    LCSX_GUARD(for (int f = 0; f < frames; f++) s->s.step(); return LCSX_OK;)
}

lcsx_status lcsx_solver_get_positions(lcsx_solver* s, float* out, size_t n)
{
    if (!s || !out || !s->s.inited || n < 3 * (size_t)s->s.S.nv) return arg_error("invalid arguments");
    LCSX_GUARD(s->s.x.download(out, 3 * (size_t)s->s.S.nv, s->s.stream); LCSX_HIP(hipStreamSynchronize(s->s.stream)); return LCSX_OK;)
}
lcsx_status lcsx_solver_get_velocities(lcsx_solver* s, float* out, size_t n)
{
    if (!s || !out || !s->s.inited || n < 3 * (size_t)s->s.S.nv) return arg_error("invalid arguments");
    LCSX_GUARD(s->s.v.download(out, 3 * (size_t)s->s.S.nv, s->s.stream); LCSX_HIP(hipStreamSynchronize(s->s.stream)); return LCSX_OK;)
}
lcsx_status lcsx_solver_set_state(lcsx_solver* s, const float* x, const float* v, size_t n)
{
    if (!s || !s->s.inited || n != 3 * (size_t)s->s.S.nv) return arg_error("invalid arguments");
    s->s.ccd_pairs_fresh = false;
    LCSX_GUARD(if (x) s->s.x.upload(x, n, s->s.stream); if (v) s->s.v.upload(v, n, s->s.stream);
               LCSX_HIP(hipStreamSynchronize(s->s.stream)); return LCSX_OK;)
}
namespace
{
// Vertex rows (kind < 2) in row order, and the body rows (4 per body) in body order.
void split_rows(const Solver& S, std::vector<uint32_t>& verts, std::vector<uint32_t>& body_rows)
{
    verts.clear();
    body_rows.clear();
    for (uint32_t i = 0; i < S.S.nv; i++)
        if (S.S.row_kind[i] < 2) verts.push_back(i);
    for (const auto& b : S.S.bodies)
        for (uint32_t k = 0; k < 4; k++) body_rows.push_back(b.row0 + k);
}
}  // namespace

// save_current_frame_state_to_host, solver_interface.cpp:206-276: sections "o position" and
// "o velocity" (one "v x y z" line per mesh vertex), "o q" and "o qv" (four lines per affine body),
// written with 9 significant digits so that a load restores the floats exactly.
static lcsx_status save_state_impl(Solver& S, const char* path)
{
    std::vector<float> x(3 * (size_t)S.S.nv), v(x.size());
    S.x.download(x.data(), x.size(), S.stream);
    S.v.download(v.data(), v.size(), S.stream);
    LCSX_HIP(hipStreamSynchronize(S.stream));
    std::vector<uint32_t> verts, brows;
    split_rows(S, verts, brows);
    std::ofstream f(path);
    if (!f) { set_error(std::string("cannot write ") + path); return LCSX_ERR_IO; }
    char line[96];
    auto put = [&](const char* head, const std::vector<float>& a, const std::vector<uint32_t>& rows) {
        f << head << '\n';
        for (uint32_t r : rows)
        {
            std::snprintf(line, sizeof(line), "v %.9g %.9g %.9g\n", a[3 * (size_t)r], a[3 * (size_t)r + 1], a[3 * (size_t)r + 2]);
            f << line;
        }
    };
    put("o position", x, verts);
    put("o velocity", v, verts);
    put("o q", x, brows);
    put("o qv", v, brows);
    if (!f) { set_error(std::string("write failed: ") + path); return LCSX_ERR_IO; }
    return LCSX_OK;
}

lcsx_status lcsx_solver_save_state(lcsx_solver* s, const char* path)
{
    if (!s || !path) return arg_error("invalid arguments");
    if (!s->s.inited) { set_error("save_state before init"); return LCSX_ERR_STATE; }
    Solver& S = s->s;
    LCSX_GUARD(return save_state_impl(S, path);)
}

// load_saved_state_from_host, solver_interface.cpp:277-410; "o qv" is matched before "o q"
// (the reference tests "o q" first, so its q section also swallows the qv lines). Files with
// fewer lines than the solver has rows leave the other rows as they are, as the reference does;
// a section with more lines is an error. frame >= 0 also sets the frame counter (pinned targets).
static lcsx_status load_state_impl(Solver& S, const char* path, int frame)
{
    std::ifstream f(path);
    if (!f) { set_error(std::string("cannot read ") + path); return LCSX_ERR_IO; }
    std::vector<float> x(3 * (size_t)S.S.nv), v(x.size());
    S.x.download(x.data(), x.size(), S.stream);
    S.v.download(v.data(), v.size(), S.stream);
    LCSX_HIP(hipStreamSynchronize(S.stream));
    std::vector<uint32_t> verts, brows;
    split_rows(S, verts, brows);
    int         sec = -1;
    size_t      idx = 0;
    std::string ln;
    while (std::getline(f, ln))
    {
        if (ln.empty()) continue;
        if (ln.rfind("o position", 0) == 0) { sec = 0; idx = 0; continue; }
        if (ln.rfind("o velocity", 0) == 0) { sec = 1; idx = 0; continue; }
        if (ln.rfind("o qv", 0) == 0) { sec = 3; idx = 0; continue; }
        if (ln.rfind("o q", 0) == 0) { sec = 2; idx = 0; continue; }
        if (ln[0] != 'v' || sec < 0) continue;
        std::istringstream iss(ln.substr(1));
        float a, b, c;
        if (!(iss >> a >> b >> c)) { set_error("malformed line in " + std::string(path) + ": " + ln); return LCSX_ERR_IO; }
        const std::vector<uint32_t>& rows = sec < 2 ? verts : brows;
        if (idx >= rows.size()) { set_error("more lines than rows in a section of " + std::string(path)); return LCSX_ERR_IO; }
        std::vector<float>& dst = (sec == 0 || sec == 2) ? x : v;
        const size_t        r   = rows[idx++];
        dst[3 * r] = a;
        dst[3 * r + 1] = b;
        dst[3 * r + 2] = c;
    }
    S.x.upload(x.data(), x.size(), S.stream);
    S.v.upload(v.data(), v.size(), S.stream);
    LCSX_HIP(hipStreamSynchronize(S.stream));
    S.ccd_pairs_fresh = false;
    if (frame >= 0) S.frame = frame;
    return LCSX_OK;
}

lcsx_status lcsx_solver_load_state(lcsx_solver* s, const char* path, int frame)
{
    if (!s || !path) return arg_error("invalid arguments");
    if (!s->s.inited) { set_error("load_state before init"); return LCSX_ERR_STATE; }
    Solver& S = s->s;
    LCSX_GUARD(return load_state_impl(S, path, frame);)
}

// saveToOBJ_combined, mesh_reader.cpp:681-750: one "o mesh_<i>" object per registered mesh with its
// current vertex positions and its triangles, indices offset across meshes (1-based).
static lcsx_status save_obj_impl(Solver& S, const char* path)
{
    std::vector<float> x(3 * (size_t)S.S.nv);
    S.x.download(x.data(), x.size(), S.stream);
    LCSX_HIP(hipStreamSynchronize(S.stream));
    std::vector<uint32_t> verts, brows;
    split_rows(S, verts, brows);
    std::ofstream f(path);
    if (!f) { set_error(std::string("cannot write ") + path); return LCSX_ERR_IO; }
    f << "# Simulated by LuisaComputeSolver\n";
    char   line[96];
    size_t at = 0, prefix = 1;
    for (size_t mi = 0; mi < S.meshes.size(); mi++)
    {
        const MeshDesc& m  = S.meshes[mi];
        const size_t    mv = m.x.size() / 3;
        f << "o mesh_" << mi << '\n';
        for (size_t k = 0; k < mv; k++)
        {
            const size_t r = verts[at + k];
            std::snprintf(line, sizeof(line), "v %.9g %.9g %.9g\n", x[3 * r], x[3 * r + 1], x[3 * r + 2]);
            f << line;
        }
        for (size_t t = 0; t + 2 < m.tris.size(); t += 3)
            f << "f " << prefix + m.tris[t] << ' ' << prefix + m.tris[t + 1] << ' ' << prefix + m.tris[t + 2] << '\n';
        at += mv;
        prefix += mv;
    }
    if (!f) { set_error(std::string("write failed: ") + path); return LCSX_ERR_IO; }
    return LCSX_OK;
}

lcsx_status lcsx_solver_save_obj(lcsx_solver* s, const char* path)
{
    if (!s || !path) return arg_error("invalid arguments");
    if (!s->s.inited) { set_error("save_obj before init"); return LCSX_ERR_STATE; }
    Solver& S = s->s;
    LCSX_GUARD(return save_obj_impl(S, path);)
}

lcsx_status lcsx_solver_set_pinned_targets(lcsx_solver* s, int mesh_id, const float* targets, int n_pinned)
{
    if (!s || !s->s.inited || mesh_id < 0 || mesh_id >= (int)s->s.meshes.size() || !targets)
        return arg_error("invalid arguments");
    Solver& S = s->s;
    int     k = 0;
    for (size_t i = 0; i < S.S.fixed_verts.size(); i++)
        if ((int)S.S.fixed_mesh[i] == mesh_id)
        {
            if (k >= n_pinned) return arg_error("n_pinned smaller than the mesh's pinned count");
            for (int d = 0; d < 3; d++) S.explicit_targets[3 * i + d] = targets[3 * k + d];
            k++;
        }
    if (k != n_pinned) return arg_error("n_pinned does not match the mesh's pinned count");
    S.has_explicit[mesh_id] = 1;
    return LCSX_OK;
}
lcsx_status lcsx_solver_get_stats(lcsx_solver* s, lcsx_stats* out)
{
    if (!s || !out) return arg_error("invalid arguments");
    *out = s->s.stats;
    return LCSX_OK;
}
int lcsx_solver_num_verts(lcsx_solver* s) { return s && (s->s.inited || s->s.setup_ready) ? (int)s->s.S.nv : 0; }

lcsx_status lcsx_solver_run_stage(lcsx_solver* s, const char* stage)
{
    if (!s || !stage) return arg_error("invalid arguments");
    if (!s->s.inited) { set_error("stage before init"); return LCSX_ERR_STATE; }
    std::string st = stage;
    Solver&     S  = s->s;
    LCSX_GUARD(
        if (st == "frame_begin") S.frame_begin();
        else if (st == "predict") S.predict();
        else if (st == "iter_begin") S.iter_begin();
        else if (st == "material") S.material();
        else if (st == "broad_phase_dcd") { launch_reset_status(S.status.p, S.sst.p, S.S.nscenes, S.stream); S.broad_phase(false); }
        else if (st == "broad_phase_ccd") { launch_reset_line_search(S.status.p, S.sst.p, S.S.nscenes, S.stream); S.broad_phase(true); }
        else if (st == "dcd") S.dcd();
        else if (st == "update_contacts") { launch_reset_status(S.status.p, S.sst.p, S.S.nscenes, S.stream); S.update_contacts(); }
        else if (st == "contact_assemble") S.contact_assemble();
        else if (st == "pcg") S.pcg();
        else if (st == "ccd") { S.ccd(); }
        else if (st == "line_search") { S.line_search(); }
        else if (st == "newton_iteration") S.newton_iteration_until_done();
        else if (st == "post_dist_check") S.post_dist_check();
        else if (st == "shrink_lists") S.alloc_collision(1024u, 1024u, 1024u);  // exercises the growth path
        else if (st == "withhold_workgroup") S.grid_withhold = true;  // exercises a wait that runs out
        else if (st == "frame_end") S.frame_end();
        else if (st == "step") S.step();
        else if (st == "spmv_dx") S.spmv_dx();
        else if (st == "spmv_dx_lp") S.spmv_dx(true);
        else { set_error("unknown stage " + st); return LCSX_ERR_ARG; }
        S.read_status();
        if (S.host_status.n_vf > S.cap_vf || S.host_status.n_ee > S.cap_ee || S.host_status.n_contacts > S.cap_c ||
            S.host_status.n_vf_ccd > S.cap_vf || S.host_status.n_ee_ccd > S.cap_ee)
        {
            S.grow_if_needed(false);
            set_error("contact buffers were too small and have been grown; re-run the stage");
            return LCSX_ERR_CAPACITY;
        }
        return LCSX_OK;)
}

lcsx_status lcsx_solver_read(lcsx_solver* s, const char* name, void* out, size_t bytes, size_t* count_out)
{
    if (!s || !name) return arg_error("invalid arguments");
    if (!s->s.inited && !(s->s.setup_ready && is_static_buffer(name)))
    {
        set_error("read before init");
        return LCSX_ERR_STATE;
    }
    LCSX_GUARD(
        Blob b;
        if (!read_named(s->s, name, b)) { set_error(std::string("unknown buffer ") + name); return LCSX_ERR_ARG; }
        if (count_out) *count_out = b.count;
        if (out)
        {
            if (bytes < b.bytes.size()) return arg_error("output buffer too small");
            if (!b.bytes.empty()) std::memcpy(out, b.bytes.data(), b.bytes.size());
        }
        return LCSX_OK;)
}

lcsx_status lcsx_solver_write(lcsx_solver* s, const char* name, const void* in, size_t bytes)
{
    if (!s || !name || !in) return arg_error("invalid arguments");
    if (!s->s.inited) { set_error("write before init"); return LCSX_ERR_STATE; }
    Solver&      S = s->s;
    std::string  n = name;
    DBuf<float>* b = nullptr;
    S.ccd_pairs_fresh = false;
    if (n == "x") b = &S.x;
    else if (n == "v") b = &S.v;
    else if (n == "x_step") b = &S.x_step;
    else if (n == "x_iter") b = &S.x_iter;
    else if (n == "x_tilde") b = &S.x_tilde;
    else if (n == "dx") b = &S.dx;
    else if (n == "cgB") b = &S.cgB;
    if (!b) { set_error("buffer " + n + " is not writable"); return LCSX_ERR_ARG; }
    if (bytes != 3 * (size_t)S.S.nv * sizeof(float)) return arg_error("size mismatch");
    LCSX_GUARD(b->upload((const float*)in, 3 * (size_t)S.S.nv, S.stream); LCSX_HIP(hipStreamSynchronize(S.stream)); return LCSX_OK;)
}

lcsx_status lcsx_solver_kernel_times(lcsx_solver* s, char* buf, size_t len, int reset)
{
    if (!s || !buf || len == 0) return arg_error("invalid arguments");
    std::string o;
    for (auto& kv : s->s.times)
        o += kv.first + "=" + std::to_string(kv.second.second ? kv.second.first / kv.second.second : 0.0) + "," +
             std::to_string(kv.second.second) + ";";
    std::strncpy(buf, o.c_str(), len - 1);
    buf[len - 1] = 0;
    if (reset) s->s.times.clear();
    return o.size() < len ? LCSX_OK : LCSX_ERR_ARG;
}

lcsx_status lcsx_solver_set_timing(lcsx_solver* s, int level)
{
    if (!s || level < 0 || level > 3) return arg_error("invalid arguments");
    s->s.timing      = level >= 1;
    s->s.spmv_sample = level >= 3 ? 1 : level == 2 ? Solver::kSpmvSample : 0;
    return LCSX_OK;
}

lcsx_status lcsx_solver_autotune(lcsx_solver* s, char* report, size_t report_len)
{
    if (!s) return arg_error("invalid arguments");
    if (!s->s.inited) { set_error("autotune before init"); return LCSX_ERR_STATE; }
    LCSX_GUARD(
        const std::string r = s->s.autotune();
        if (report && report_len)
        {
            std::strncpy(report, r.c_str(), report_len - 1);
            report[report_len - 1] = 0;
        }
        return LCSX_OK;)
}

lcsx_status lcsx_solver_set_graphs(lcsx_solver* s, int on)
{
    if (!s || (on != 0 && on != 1)) return arg_error("invalid arguments");
    s->s.use_graphs = on == 1;
    s->s.pcg_grid   = false;  // the caller chooses the form of the launches
    return LCSX_OK;
}

lcsx_status lcsx_solver_set_one_launch(lcsx_solver* s, int on)
{
    if (!s || (on != 0 && on != 1)) return arg_error("invalid arguments");
    s->s.pcg_grid = on == 1;
    return LCSX_OK;
}

lcsx_status lcsx_solver_set_query_shape(lcsx_solver* s, int shape)
{
    if (!s || shape < 0 || shape >= kQueryVariants) return arg_error("invalid arguments");
    s->s.query_variant = shape;
    return LCSX_OK;
}

lcsx_status lcsx_solver_set_spmv_shape(lcsx_solver* s, int shape)
{
    if (!s || shape < 0 || shape >= kSpmvShapes) return arg_error("invalid arguments");
    s->s.spmv_shape = shape;
    s->s.pcg_grid   = false;  // a mapping of the launched product
    return LCSX_OK;
}

// ------------------------------------------------------------ standalone narrow phase
namespace
{
// Device words of one call's scratch, allocated for the call and freed before it returns.
struct CallWork
{
    uint32_t* p = nullptr;
    explicit CallWork(size_t words) { LCSX_HIP(hipMalloc((void**)&p, std::max<size_t>(words, 1) * sizeof(uint32_t))); }
    ~CallWork()
    {
        if (p) (void)hipFree(p);
    }
};
}  // namespace

lcsx_status lcsx_ccd_pairs(int kind, const uint32_t* pairs, uint32_t n_pairs, const uint32_t* prims, const float* x0,
                           const float* x1, const float* offset, int precision, float* toi, void* stream)
{
    if ((kind != 0 && kind != 1) || (n_pairs && (!pairs || !prims || !x0 || !x1 || !offset)) || !toi ||
        precision < 0 || precision > 2)
        return arg_error("invalid arguments");
    LCSX_GUARD(
        const hipStream_t s = (hipStream_t)stream;
        CallWork          w(6 + (size_t)n_pairs);
        narrow_ccd(kind, pairs, n_pairs, prims, x0, x1, offset, precision >= 1 ? 1 : 0, 32, toi, w.p, s);
        LCSX_HIP(hipGetLastError());
        LCSX_HIP(hipStreamSynchronize(s));
        return LCSX_OK;)
}

lcsx_status lcsx_dcd_pairs(int kind, const uint32_t* pairs, uint32_t n_pairs, const uint32_t* prims, const float* x,
                           const float* area_a, const float* area_b, const float* offset, const float* dhat,
                           float kappa, int contact_energy_type, int precision, uint32_t* contact_idx,
                           float* contact_nk, float* contact_w, float* contact_aux, uint32_t capacity,
                           uint32_t* count, void* stream)
{
    if ((kind != 0 && kind != 1) || (n_pairs && (!pairs || !prims || !x || !area_a || !area_b || !offset || !dhat)) ||
        !count || (capacity && (!contact_idx || !contact_nk || !contact_w || !contact_aux)) ||
        (contact_energy_type != 0 && contact_energy_type != 1) || precision < 0 || precision > 2)
        return arg_error("invalid arguments");
    LCSX_GUARD(
        const hipStream_t s = (hipStream_t)stream;
        CallWork          w(1);
        ContactBuf        out;
        out.idx      = reinterpret_cast<uint4*>(contact_idx);
        out.nk       = reinterpret_cast<float4*>(contact_nk);
        out.w        = reinterpret_cast<float4*>(contact_w);
        out.aux      = reinterpret_cast<float4*>(contact_aux);
        out.count    = count;
        out.capacity = capacity;
        narrow_dcd(kind, pairs, n_pairs, prims, x, area_a, area_b, offset, dhat, kappa, contact_energy_type == 0 ? 1 : 0,
                   precision >= 1 ? 1 : 0, out, w.p, s);
        LCSX_HIP(hipGetLastError());
        LCSX_HIP(hipStreamSynchronize(s));
        return LCSX_OK;)
}

// ------------------------------------------------------------ standalone LBVH
lcsx_status lcsx_lbvh_create(int arity, const uint32_t* device_prims, int n_leaves, lcsx_lbvh** out)
{
    if (!out || (arity != 2 && arity != 3) || n_leaves <= 0 || !device_prims) return arg_error("invalid arguments");
    auto* t = new lcsx_lbvh();
    LCSX_GUARD(t->t.init(arity, device_prims, (uint32_t)n_leaves); *out = t; return LCSX_OK;)
}
lcsx_status lcsx_lbvh_destroy(lcsx_lbvh* t)
{
    delete t;
    return LCSX_OK;
}
lcsx_status lcsx_lbvh_construct(lcsx_lbvh* t, const float* x, int n_verts, void* stream)
{
    if (!t || !x || n_verts <= 0) return arg_error("invalid arguments");
    t->last = (hipStream_t)stream;
    const uint32_t nvs = (uint32_t)n_verts;
    LCSX_GUARD(t->t.construct(x, &nvs, (hipStream_t)stream); t->constructed = true; return LCSX_OK;)
}
lcsx_status lcsx_lbvh_refit(lcsx_lbvh* t, const float* x0, const float* x1, const float* pad, void* stream)
{
    if (!t || !x0 || !x1 || !pad) return arg_error("invalid arguments");
    if (!t->constructed) { set_error("refit before construct"); return LCSX_ERR_STATE; }
    t->last = (hipStream_t)stream;
    LCSX_GUARD(t->t.refit(x0, x1, pad, (hipStream_t)stream); t->refitted = true; return LCSX_OK;)
}
lcsx_status lcsx_lbvh_query(lcsx_lbvh* t, const float* boxes, int n_queries, int edge_filter, uint32_t* pairs,
                            uint32_t capacity, uint32_t* count, void* stream)
{
    if (!t || !boxes || n_queries < 0 || !pairs || !count) return arg_error("invalid arguments");
    if (!t->refitted) { set_error("query before refit"); return LCSX_ERR_STATE; }
    QueryArgs q{};
    q.mode        = QueryBoxes;
    q.n_queries   = (uint32_t)n_queries;
    q.boxes       = boxes;
    q.edge_filter = edge_filter;
    q.pairs       = pairs;
    q.capacity    = capacity;
    q.count       = count;
    q.variant     = t->shape;
    t->last       = (hipStream_t)stream;
    LCSX_GUARD(lbvh_query(t->t, q, (hipStream_t)stream); return LCSX_OK;)
}
lcsx_status lcsx_lbvh_set_query_shape(lcsx_lbvh* t, int shape)
{
    if (!t || shape < 0 || shape >= kQueryVariants) return arg_error("invalid arguments");
    t->shape = shape;
    return LCSX_OK;
}
lcsx_status lcsx_lbvh_read(lcsx_lbvh* t, const char* name, void* out, size_t bytes)
{
    if (!t || !name || !out) return arg_error("invalid arguments");
    LCSX_GUARD(
        Blob b;
        if (!read_tree(t->t, name, t->last, b)) { set_error(std::string("unknown tree buffer ") + name); return LCSX_ERR_ARG; }
        if (bytes < b.bytes.size()) return arg_error("output buffer too small");
        std::memcpy(out, b.bytes.data(), b.bytes.size());
        return LCSX_OK;)
}
}
