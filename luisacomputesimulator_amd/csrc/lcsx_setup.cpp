// Host-side scene setup. Reference counterparts:
//   edges / hinges           Solver/MeshOperation/mesh_reader.cpp:219-352
//   pins                     Solver/Initializer/init_mesh_data.cpp:59-95, 117-240
//   areas / mass / thickness Solver/Initializer/init_mesh_data.cpp:783-995
//   offset / d_hat           Solver/Initializer/init_collision_data.cpp:71-174
//   elements / CSR / offsets Solver/Initializer/init_sim_data.cpp:19-48, 189-480, 760-896
#include "lcsx_setup.h"
#include <algorithm>
#include <stdexcept>
#include <cmath>
#include <map>
#include <numeric>
#include "lcsx_physics.h"

namespace lcsx
{

namespace
{
struct EdgeKey
{
    uint32_t a, b, f;
};

// Unique sorted edges and hinges (e0 < e1, opposite vertex of the lower then higher face).
void topology(const std::vector<int32_t>& tris, std::vector<uint32_t>& E, std::vector<uint32_t>& H)
{
    size_t               nt = tris.size() / 3;
    std::vector<EdgeKey> k(3 * nt);
    for (size_t f = 0; f < nt; f++)
    {
        uint32_t v[3] = {(uint32_t)tris[3 * f], (uint32_t)tris[3 * f + 1], (uint32_t)tris[3 * f + 2]};
        std::sort(v, v + 3);
        k[3 * f]     = {v[0], v[1], (uint32_t)f};
        k[3 * f + 1] = {v[0], v[2], (uint32_t)f};
        k[3 * f + 2] = {v[1], v[2], (uint32_t)f};
    }
    std::sort(k.begin(), k.end(), [](const EdgeKey& l, const EdgeKey& r) {
        return l.a != r.a ? l.a < r.a : (l.b != r.b ? l.b < r.b : l.f < r.f);
    });
    auto same = [&](size_t i, size_t j) { return k[i].a == k[j].a && k[i].b == k[j].b; };
    E.clear();
    H.clear();
    std::vector<uint8_t> first_of_pair(k.size(), 0);
    for (size_t i = 0; i < k.size(); i++)
    {
        bool has_next = i + 1 < k.size() && same(i, i + 1);
        bool has_prev = i > 0 && same(i, i - 1);
        if (has_prev || !has_next)
        {
            E.push_back(k[i].a);
            E.push_back(k[i].b);
        }
        if (has_next && !has_prev) first_of_pair[i] = 1;
        if (has_next && has_prev) first_of_pair[i] = 0;  // middle of a non-manifold fan
    }
    for (size_t i = 0; i < k.size(); i++)
    {
        if (!first_of_pair[i]) continue;
        const int32_t* c = &tris[3 * k[i].f];
        const int32_t* d = &tris[3 * k[i + 1].f];
        uint32_t       s = k[i].a + k[i].b;
        H.push_back(k[i].a);
        H.push_back(k[i].b);
        H.push_back((uint32_t)(c[0] + c[1] + c[2]) - s);
        H.push_back((uint32_t)(d[0] + d[1] + d[2]) - s);
    }
}

f3 at(const std::vector<float>& x, uint32_t i) { return mk(x[3 * i], x[3 * i + 1], x[3 * i + 2]); }
}  // namespace

void pin_by_method(MeshDesc& m, int method, float r, const lcsx_fixed_anim& anim)
{
    size_t n = m.x.size() / 3;
    float  lo[3] = {3.4e38f, 3.4e38f, 3.4e38f}, hi[3] = {-3.4e38f, -3.4e38f, -3.4e38f};
    for (size_t i = 0; i < n; i++)
        for (int d = 0; d < 3; d++)
        {
            lo[d] = std::min(lo[d], m.x[3 * i + d]);
            hi[d] = std::max(hi[d], m.x[3 * i + d]);
        }
    float inv[3];
    for (int d = 0; d < 3; d++) inv[d] = 1.0f / std::max(hi[d] - lo[d], 0.0001f);
    for (size_t i = 0; i < n; i++)
    {
        float x = (m.x[3 * i] - lo[0]) * inv[0], y = (m.x[3 * i + 1] - lo[1]) * inv[1], z = (m.x[3 * i + 2] - lo[2]) * inv[2];
        bool  L = x < r, R = x > 1.0f - r, F = z < r, B = z > 1.0f - r, U = y > 1.0f - r, D = y < r;
        bool  sel = false;
        switch (method)
        {
            case 3: sel = L; break;
            case 4: sel = R; break;
            case 5: sel = F; break;
            case 6: sel = B; break;
            case 7: sel = U; break;
            case 8: sel = D; break;
            case 9: sel = L && U; break;
            case 10: sel = L && D; break;
            case 11: sel = L && B; break;  // LeftFront: x < r, z > 1 - r (init_mesh_data.cpp:180)
            case 12: sel = L && F; break;  // LeftBack:  x < r, z < r
            case 13: sel = R && U; break;
            case 14: sel = R && D; break;
            case 15: sel = R && B; break;  // RightFront
            case 16: sel = R && F; break;  // RightBack
            case 17: sel = F && U; break;
            case 18: sel = F && D; break;
            case 19: sel = B && U; break;
            case 20: sel = B && D; break;
            case 21: sel = true; break;
            default: sel = false;
        }
        if (sel)
        {
            m.pinned.push_back((uint32_t)i);
            m.anim.push_back(anim);
        }
    }
}

void animate_target(const lcsx_fixed_anim& a, float t, const float in[3], float out[3])
{
    f3 p = mk(in[0], in[1], in[2]);
    if (a.use_scale) p = mk(a.scale[0] * t * p.x, a.scale[1] * t * p.y, a.scale[2] * t * p.z);
    if (a.use_rotate)
    {
        float ang = t * a.rot_deg_per_s / 180.0f * 3.14159265358979323846f;
        f3    c   = mk(a.rot_center[0], a.rot_center[1], a.rot_center[2]);
        f3    rel = p - c;
        if (ang != 0.0f)
        {
            f3    ax = normalize(mk(a.rot_axis[0], a.rot_axis[1], a.rot_axis[2]));
            float co = std::cos(ang), si = std::sin(ang);
            f3    tt = (1.0f - co) * ax;
            f3    c0 = mk(co + tt.x * ax.x, tt.x * ax.y + si * ax.z, tt.x * ax.z - si * ax.y);
            f3    c1 = mk(tt.y * ax.x - si * ax.z, co + tt.y * ax.y, tt.y * ax.z + si * ax.x);
            f3    c2 = mk(tt.z * ax.x + si * ax.y, tt.z * ax.y - si * ax.x, co + tt.z * ax.z);
            rel      = (c0 * rel.x + c1 * rel.y) + c2 * rel.z;
        }
        p = c + rel;
    }
    if (a.use_translate) p = p + mk(a.translate[0] * t, a.translate[1] * t, a.translate[2] * t);
    out[0] = p.x;
    out[1] = p.y;
    out[2] = p.z;
}

// Sorts n ids by their 30-bit codes, equal ones by id (they come in ascending order): three stable
// counting passes, or std::sort for few.
static void sort_by_code(uint32_t* id, const std::vector<uint32_t>& code, size_t n, std::vector<uint32_t>& tmp)
{
    if (n < 1024)
    {
        std::stable_sort(id, id + n, [&](uint32_t x, uint32_t y) { return code[x] < code[y]; });
        return;
    }
    tmp.resize(std::max(tmp.size(), n));
    uint32_t *from = id, *to = tmp.data();
    for (int shift = 0; shift < 30; shift += 10)
    {
        uint32_t at[1024] = {}, sum = 0;
        for (size_t i = 0; i < n; i++) at[(code[from[i]] >> shift) & 1023u]++;
        for (uint32_t& c : at) std::swap(c, sum), sum += c;
        for (size_t i = 0; i < n; i++) to[at[(code[from[i]] >> shift) & 1023u]++] = from[i];
        std::swap(from, to);
    }
    std::copy(from, from + n, id);  // (three passes end in tmp)
}

void Setup::cluster()
{
    // per mesh: the rest pose's box (a cube of its largest side, so that distances along the axes count alike)
    uint32_t nm = 0;
    for (uint32_t i = 0; i < nv; i++) nm = std::max(nm, vert_mesh[i] + 1u);
    std::vector<float>    lo(3 * (size_t)nm, 3.0e38f), hi(3 * (size_t)nm, -3.0e38f), scale(nm);
    std::vector<uint32_t> mesh_scene(nm, 0);
    auto                  point = [&](uint32_t i) { return row_kind[i] < 2; };
    for (uint32_t i = 0; i < nv; i++)
    {
        const uint32_t m = vert_mesh[i];
        mesh_scene[m]    = vert_scene[i];
        for (uint32_t k = 0; point(i) && k < 3; k++)
        {
            lo[3 * m + k] = std::min(lo[3 * m + k], rest_x[3 * i + k]);
            hi[3 * m + k] = std::max(hi[3 * m + k], rest_x[3 * i + k]);
        }
    }
    for (uint32_t m = 0; m < nm; m++)
    {
        float side = 1e-12f;
        for (uint32_t k = 0; k < 3; k++) side = std::max(side, hi[3 * m + k] - lo[3 * m + k]);
        scale[m] = 1024.0f / side;
    }
    auto spread = [](uint32_t v) {  // ten bits, two zeros between any two
        v = (v | (v << 16)) & 0x030000ffu;
        v = (v | (v << 8)) & 0x0300f00fu;
        v = (v | (v << 4)) & 0x030c30c3u;
        return (v | (v << 2)) & 0x09249249u;
    };
    auto morton = [&](uint32_t m, const float c[3]) {
        uint32_t code = 0;
        for (uint32_t k = 0; k < 3; k++)
        {
            const float v = (c[k] - lo[3 * m + k]) * scale[m];
            code |= spread(v > 0.0f ? (uint32_t)std::min(v, 1023.0f) : 0u) << (2 - k);
        }
        return code;
    };
    // the elements of all meshes, each mesh's along its curve, every scene padded to whole units (the meshes
    // are numbered scene by scene); arity 0: points
    std::vector<uint32_t> code, id, first, tmp;
    auto ordered = [&](uint32_t n, uint32_t arity, const std::vector<uint32_t>& prims, uint32_t unit,
                       std::vector<uint32_t>& out, std::vector<uint32_t>* block) {
        auto mesh = [&](uint32_t i) { return vert_mesh[arity ? prims[arity * i] : i]; };
        code.resize(n);
        first.assign(nm + 1, 0);
        for (uint32_t i = 0; i < n; i++)
        {
            if (!arity && !point(i)) continue;
            float c[3] = {0.0f, 0.0f, 0.0f};
            for (uint32_t k = 0; k < 3; k++)
                if (!arity) c[k] = rest_x[3 * i + k];
                else
                    for (uint32_t a = 0; a < arity; a++) c[k] += rest_x[3 * prims[arity * i + a] + k] / (float)arity;
            code[i] = morton(mesh(i), c);
            first[mesh(i) + 1]++;
        }
        for (uint32_t m = 0; m < nm; m++) first[m + 1] += first[m];
        id.resize(first[nm]);
        std::vector<uint32_t> at(first.begin(), first.end() - 1);
        for (uint32_t i = 0; i < n; i++)
            if (arity || point(i)) id[at[mesh(i)]++] = i;
        uint32_t m = 0;
        for (uint32_t sc = 0; sc < nscenes; sc++)
        {
            if (block) block->push_back((uint32_t)(out.size() / unit));
            for (; m < nm && mesh_scene[m] <= sc; m++)
            {
                sort_by_code(id.data() + first[m], code, first[m + 1] - first[m], tmp);
                out.insert(out.end(), id.begin() + first[m], id.begin() + first[m + 1]);
            }
            while (out.size() % unit) out.push_back(kInvalid);
        }
        if (block) block->push_back((uint32_t)(out.size() / unit));
    };
    ordered(nv, 0, faces, 64, cluster_v, nullptr);
    ordered(nf, 3, faces, kClusterLeaves, cluster_f, &cluster_f_block);
    ordered(ne, 2, edges, kClusterLeaves, cluster_e, &cluster_e_block);
    // Pieces: what edges hold together (made when first asked for). A block of a piece's elements stays small in
    // space however the pieces move; one over many pieces may reach over the whole scene, and so may all such
    // blocks.
    std::vector<uint32_t> piece;
    auto root = [&](uint32_t i) {
        while (piece[i] != i) i = piece[i] = piece[piece[i]];
        return i;
    };
    auto join = [&]() {
        piece.resize(nv);
        for (uint32_t i = 0; i < nv; i++) piece[i] = i;
        for (uint32_t e = 0; e < ne; e++)
        {
            const uint32_t a = root(edges[2 * e]), b = root(edges[2 * e + 1]);
            piece[std::max(a, b)] = std::min(a, b);
        }
    };
    // The blocks are walked unless a scene has more than kMost of them over several pieces (every query meets
    // nearly all of those: the line is one step of the walk over the blocks), or there are more than kMost in all
    // and less than a quarter of their positions are taken (batches of tiny scenes; a block costs the same
    // however empty). The queries then walk the LBVH, a lane each. A swept broad phase,
    // blocks against LBVH: boxes of 18 edges, 2,000 of them (47 mixed blocks) 12.2 and 13.6 us, 3,000 (66) 16.6 and
    // 14.5, 6,000 30.8 and 16.4, 24,000 368 and 57; 2,000 scenes of 7 x 7 cloths (120 edges) 47 and 20 us,
    // 11 x 11 (320) 45 and 42, 13 x 13 (456) 45 and 57.
    auto use = [&](uint32_t n, uint32_t arity, const std::vector<uint32_t>& prims, const std::vector<uint32_t>& order,
                   const std::vector<uint32_t>& block) {
        constexpr uint32_t kMost = 64;
        uint32_t           most  = 0;
        for (uint32_t sc = 0; sc < nscenes; sc++)
        {
            if (block[sc + 1] - block[sc] <= kMost) continue;
            if (piece.empty()) join();
            uint32_t mixed = 0;
            for (uint32_t b = block[sc]; b < block[sc + 1]; b++)
            {
                const uint32_t* el = &order[(size_t)b * kClusterLeaves];
                const uint32_t  p  = root(prims[arity * el[0]]);
                bool            m  = false;
                for (uint32_t k = 1; k < kClusterLeaves && el[k] != kInvalid && !m; k++) m = root(prims[arity * el[k]]) != p;
                mixed += m ? 1u : 0u;
            }
            most = std::max(most, mixed);
        }
        const uint32_t blocks = block[nscenes];
        return most <= kMost && (blocks <= kMost || 4ull * n >= (uint64_t)blocks * kClusterLeaves);
    };
    cluster_f_use = use(nf, 3, faces, cluster_f, cluster_f_block);
    cluster_e_use = use(ne, 2, edges, cluster_e, cluster_e_block);
}

void Setup::build(const std::vector<MeshDesc>& meshes)
{
    *this = Setup();
    std::vector<uint32_t> mesh_v0(meshes.size(), 0);
    for (size_t mi = 0; mi < meshes.size(); mi++)
    {
        const MeshDesc&       m  = meshes[mi];
        uint32_t              bv = nv;
        mesh_v0[mi]              = bv;
        const bool            rigid = m.mat.body != 0;
        std::vector<uint32_t> E, H;
        topology(m.tris, E, H);
        // init_mesh_data.cpp:396-421: a rigid mesh (shell or solid) must be closed, i.e. every
        // edge is a hinge of two triangles
        if (rigid && H.size() / 4 != E.size() / 2)
            throw std::runtime_error("mesh " + std::to_string(mi) + ": a rigid body's mesh must be closed");
        uint32_t mv = (uint32_t)(m.x.size() / 3);
        rest_x.insert(rest_x.end(), m.x.begin(), m.x.end());
        vert_mesh.insert(vert_mesh.end(), mv, (uint32_t)mi);
        is_fixed.insert(is_fixed.end(), mv, 0);
        for (int32_t t : m.tris) faces.push_back(bv + (uint32_t)t);
        face_mesh.insert(face_mesh.end(), m.tris.size() / 3, (uint32_t)mi);
        for (uint32_t e : E) edges.push_back(bv + e);
        edge_mesh.insert(edge_mesh.end(), E.size() / 2, (uint32_t)mi);
        for (uint32_t h : H) hinges.push_back(bv + h);
        for (size_t k = 0; k < m.pinned.size(); k++)
        {
            is_fixed[bv + m.pinned[k]] = 1;
            if (rigid) continue;  // a pinned rigid vertex fixes its body (no target)
            fixed_verts.push_back(bv + m.pinned[k]);
            fixed_mesh.push_back((uint32_t)mi);
            fixed_local.push_back((uint32_t)k);
            fixed_anim.push_back(m.anim[k]);
        }
        row_kind.insert(row_kind.end(), mv, rigid ? 1 : 0);
        vert_body.insert(vert_body.end(), mv, rigid ? (uint32_t)bodies.size() : ~0u);
        for (uint32_t i = 0; i < mv; i++)
            for (int d = 0; d < 3; d++) body_X.push_back(rigid ? m.x[3 * i + d] : 0.0f);
        if (rigid)
        {
            Body b{};
            b.v0 = bv;
            b.v1 = bv + mv;
            b.fixed = m.pinned.empty() ? 0u : 1u;
            bodies.push_back(b);
        }
        nv += mv;
        // the scene's body rows follow its last mesh
        const bool scene_end = mi + 1 == meshes.size() || meshes[mi + 1].scene != m.scene;
        if (scene_end)
            for (size_t b = 0; b < bodies.size(); b++)
            {
                if (bodies[b].row0 != 0 || vert_mesh[bodies[b].v0] > mi) continue;
                if (meshes[vert_mesh[bodies[b].v0]].scene != m.scene) continue;
                bodies[b].row0 = nv;
                static const float q0[12] = {0, 0, 0, 1, 0, 0, 0, 1, 0, 0, 0, 1};
                rest_x.insert(rest_x.end(), q0, q0 + 12);
                vert_mesh.insert(vert_mesh.end(), 4, vert_mesh[bodies[b].v0]);
                is_fixed.insert(is_fixed.end(), 4, (uint8_t)bodies[b].fixed);
                for (int k = 0; k < 4; k++) row_kind.push_back((uint8_t)(2 + k));
                vert_body.insert(vert_body.end(), 4, (uint32_t)b);
                body_X.insert(body_X.end(), 12, 0.0f);
                nv += 4;
            }
    }
    nf = (uint32_t)(faces.size() / 3);
    ne = (uint32_t)(edges.size() / 2);
    nh = (uint32_t)(hinges.size() / 4);
    // (edges are sorted within a mesh; two listings of a face are the two sides of a hinge, unless a third
    // face makes its edge a repeated one; a face that names a vertex twice has the edge of that vertex)
    for (uint32_t e = 0; e < ne; e++)
        repeats = repeats || edges[2 * e] == edges[2 * e + 1] ||
                  (e && edges[2 * e] == edges[2 * e - 2] && edges[2 * e + 1] == edges[2 * e - 1]);
    for (uint32_t h = 0; h < nh; h++) repeats = repeats || hinges[4 * h + 2] == hinges[4 * h + 3];

    // scene ranges (meshes arrive in non-decreasing scene order) and scene-aligned row blocks
    nscenes = meshes.empty() ? 1u : meshes.back().scene + 1u;
    sc_v0.assign(nscenes + 1, 0);
    sc_f0.assign(nscenes + 1, 0);
    sc_e0.assign(nscenes + 1, 0);
    sc_verts.assign(nscenes, 0);
    for (size_t mi = 0; mi < meshes.size(); mi++)
    {
        uint32_t sc = meshes[mi].scene;
        sc_v0[sc + 1] += (uint32_t)(meshes[mi].x.size() / 3) + (meshes[mi].mat.body != 0 ? 4u : 0u);
        sc_verts[sc] += (uint32_t)(meshes[mi].x.size() / 3);
    }
    for (uint32_t f = 0; f < nf; f++) sc_f0[meshes[face_mesh[f]].scene + 1]++;
    for (uint32_t e = 0; e < ne; e++) sc_e0[meshes[edge_mesh[e]].scene + 1]++;
    for (uint32_t sc = 0; sc < nscenes; sc++)
    {
        sc_v0[sc + 1] += sc_v0[sc];
        sc_f0[sc + 1] += sc_f0[sc];
        sc_e0[sc + 1] += sc_e0[sc];
    }
    vert_scene.assign(nv, 0);
    sc_rb0.assign(nscenes + 1, 0);
    rb_scene.clear();
    rb_row0.clear();
    for (uint32_t sc = 0; sc < nscenes; sc++)
    {
        for (uint32_t i = sc_v0[sc]; i < sc_v0[sc + 1]; i++) vert_scene[i] = sc;
        for (uint32_t r = sc_v0[sc]; r < sc_v0[sc + 1]; r += 256u)
        {
            rb_scene.push_back(sc);
            rb_row0.push_back(r);
        }
        sc_rb0[sc + 1] = (uint32_t)rb_scene.size();
    }
    n_rb = (uint32_t)rb_scene.size();

    // areas: faces in float, vertices and edges accumulate face/3 in double
    face_area.resize(nf);
    std::vector<std::vector<uint32_t>> v_faces(nv);
    for (uint32_t f = 0; f < nf; f++)
    {
        const uint32_t* t = &faces[3 * f];
        face_area[f]       = length(cross(at(rest_x, t[1]) - at(rest_x, t[0]), at(rest_x, t[2]) - at(rest_x, t[0]))) * 0.5f;
        for (int j = 0; j < 3; j++) v_faces[t[j]].push_back(f);
    }
    {
        // edges are sorted (lexicographic within each mesh, meshes in order): binary search, the
        // last of equal keys (a non-manifold edge listed twice) as a key -> edge map would keep
        std::vector<uint64_t> ekey(ne);
        for (uint32_t e = 0; e < ne; e++) ekey[e] = ((uint64_t)edges[2 * e] << 32) | edges[2 * e + 1];
        std::vector<double> acc(ne, 0.0);
        for (uint32_t f = 0; f < nf; f++)
            for (int j = 0; j < 3; j++)
            {
                uint32_t a = faces[3 * f + j], b = faces[3 * f + (j + 1) % 3];
                uint64_t k  = ((uint64_t)std::min(a, b) << 32) | std::max(a, b);
                auto     it = std::upper_bound(ekey.begin(), ekey.end(), k);
                if (it != ekey.begin() && *(it - 1) == k) acc[(it - 1) - ekey.begin()] += face_area[f] / 3.0;
            }
        edge_area.resize(ne);
        for (uint32_t e = 0; e < ne; e++) edge_area[e] = (float)acc[e];
    }
    vert_area.resize(nv);
    std::vector<float> vvol(nv);
    for (uint32_t i = 0; i < nv; i++)
    {
        double a = 0.0;
        for (uint32_t f : v_faces[i]) a += face_area[f] / 3.0;
        vert_area[i] = (float)a;
        vvol[i]      = vert_area[i] * meshes[vert_mesh[i]].mat.thickness;
    }
    std::vector<float> body_vol(meshes.size(), 0.0f), body_mass(meshes.size(), 0.0f);
    for (uint32_t f = 0; f < nf; f++) body_vol[face_mesh[f]] += face_area[f] * meshes[face_mesh[f]].mat.thickness;
    for (size_t mi = 0; mi < meshes.size(); mi++)
        body_mass[mi] = meshes[mi].mat.mass != 0.0f ? meshes[mi].mat.mass : body_vol[mi] * meshes[mi].mat.density;
    vert_mass.resize(nv);
    for (uint32_t i = 0; i < nv; i++) vert_mass[i] = (vvol[i] / body_vol[vert_mesh[i]]) * body_mass[vert_mesh[i]];

    // contact offset and d_hat, clamped to 0.9 of the smallest rest edge length / altitude
    std::vector<float> min_dist(meshes.size(), 1e10f);
    for (uint32_t e = 0; e < ne; e++)
        min_dist[edge_mesh[e]] = std::min(min_dist[edge_mesh[e]], length(at(rest_x, edges[2 * e]) - at(rest_x, edges[2 * e + 1])));
    for (uint32_t f = 0; f < nf; f++)
    {
        float rd = 10000.0f;
        for (int i = 0; i < 3; i++)
        {
            f3    v0 = at(rest_x, faces[3 * f + i]), v1 = at(rest_x, faces[3 * f + (i + 1) % 3]), v2 = at(rest_x, faces[3 * f + (i + 2) % 3]);
            float c0, c1;
            pe_coeff(v0, v1, v2, c0, c1);
            rd = std::min(rd, length((c0 * v1 + c1 * v2) - v0));
        }
        min_dist[face_mesh[f]] = std::min(min_dist[face_mesh[f]], rd);
    }
    offset.resize(nv);
    dhat.resize(nv);
    for (uint32_t i = 0; i < nv; i++)
    {
        const lcsx_material& mt = meshes[vert_mesh[i]].mat;
        // a rigid solid has no contact thickness (init_mesh_data.cpp:405-414)
        float so = mt.body == 2 ? 0.0f : 0.5f * mt.thickness, sd = mt.d_hat, safe = 0.9f * min_dist[vert_mesh[i]];
        if (!(so + mt.d_hat < safe))
        {
            if (so > 0.5f * safe) so = 0.5f * safe;
            if (sd > safe - so) sd = safe - so;
        }
        offset[i] = so;
        dhat[i]   = sd;
    }

    // culled stretch faces and bending hinges (all-pinned elements dropped)
    for (uint32_t f = 0; f < nf; f++)
    {
        const uint32_t* t = &faces[3 * f];
        if (vert_body[t[0]] != ~0u) continue;  // rigid meshes have no stretch terms
        if (meshes[face_mesh[f]].mat.stretch_spring) continue;  // springs instead
        if (is_fixed[t[0]] && is_fixed[t[1]] && is_fixed[t[2]]) continue;
        sf.insert(sf.end(), t, t + 3);
        float d[4];
        dm_inv(at(rest_x, t[0]), at(rest_x, t[1]), at(rest_x, t[2]), d);
        sf_Dm.insert(sf_Dm.end(), d, d + 4);
        sf_area.push_back(face_area[f]);
        const lcsx_material& mt = meshes[face_mesh[f]].mat;
        double mu = mt.youngs_modulus / (2.0 * (1.0 + mt.poisson_ratio));
        double la = mt.youngs_modulus * mt.poisson_ratio / ((1.0 + mt.poisson_ratio) * (1.0 - 2.0 * mt.poisson_ratio));
        sf_mu.push_back((float)(mt.thickness * mu));
        sf_lambda.push_back((float)(mt.thickness * la));
    }
    for (uint32_t h = 0; h < nh; h++)
    {
        const uint32_t* q = &hinges[4 * h];
        if (vert_body[q[0]] != ~0u) continue;
        if (is_fixed[q[0]] && is_fixed[q[1]] && is_fixed[q[2]] && is_fixed[q[3]]) continue;
        bh.insert(bh.end(), q, q + 4);
        f3 p0 = at(rest_x, q[0]), p1 = at(rest_x, q[1]), p2 = at(rest_x, q[2]), p3 = at(rest_x, q[3]);
        bh_angle.push_back(dihedral_angle(p0, p1, p2, p3));
        float A1 = length(cross(p1 - p0, p2 - p0)) * 0.5f, A2 = length(cross(p1 - p0, p3 - p0)) * 0.5f;
        bh_hbar.push_back((A1 + A2) / (3.0f * length(p0 - p1)));
        bh_k.push_back(meshes[vert_mesh[q[0]]].mat.area_bending_stiffness);
    }
    // stretch springs of the spring-model cloth meshes, one per edge with a free end
    // (init_sim_data.cpp:205-235, 336-365): rest length |x0 - x1|, stiffness thickness * mu
    for (uint32_t e = 0; e < ne; e++)
    {
        const uint32_t* q = &edges[2 * e];
        const lcsx_material& mt = meshes[edge_mesh[e]].mat;
        if (vert_body[q[0]] != ~0u || !mt.stretch_spring) continue;
        if (is_fixed[q[0]] && is_fixed[q[1]]) continue;
        sp.insert(sp.end(), q, q + 2);
        sp_rest.push_back(length(at(rest_x, q[0]) - at(rest_x, q[1])));
        double mu = mt.youngs_modulus / (2.0 * (1.0 + mt.poisson_ratio));
        sp_k.push_back((float)(mu * mt.thickness));
    }
    const uint32_t nsf = (uint32_t)(sf.size() / 3), nbh = (uint32_t)(bh.size() / 4), nsp = (uint32_t)(sp.size() / 2);
    if (std::max(std::max(nsf, nbh), nsp) >= (1u << 27))
        throw std::runtime_error("more than 2^27 stretch or bending elements");

    // material neighbour lists (sorted), reference CSR layout
    std::vector<std::vector<uint32_t>> adj(nv);
    auto add = [&](uint32_t a, uint32_t b) {
        auto& l = adj[a];
        if (std::find(l.begin(), l.end(), b) == l.end()) l.push_back(b);
    };
    for (uint32_t e = 0; e < nsp; e++)
    {
        add(sp[2 * e], sp[2 * e + 1]);
        add(sp[2 * e + 1], sp[2 * e]);
    }
    for (uint32_t f = 0; f < nsf; f++)
        for (int i = 0; i < 3; i++)
            for (int j = 0; j < 3; j++)
                if (i != j) add(sf[3 * f + i], sf[3 * f + j]);
    for (uint32_t e = 0; e < nbh; e++)
        for (int i = 0; i < 4; i++)
            for (int j = 0; j < 4; j++)
                if (i != j) add(bh[4 * e + i], bh[4 * e + j]);
    for (const Body& b : bodies)
        for (uint32_t i = 0; i < 4; i++)
            for (uint32_t j = 0; j < 4; j++)
                if (i != j) add(b.row0 + i, b.row0 + j);
    for (auto& l : adj)
    {
        std::sort(l.begin(), l.end());
        max_degree = std::max<uint32_t>(max_degree, (uint32_t)l.size());
    }
    csr.assign(nv + 1, 0);
    uint32_t cur = nv + 1;
    for (uint32_t i = 0; i < nv; i++)
    {
        csr[i] = cur;
        cur += (uint32_t)adj[i].size();
    }
    csr[nv] = cur;
    for (uint32_t i = 0; i < nv; i++) csr.insert(csr.end(), adj[i].begin(), adj[i].end());

    // vertex -> element gather lists in element order
    auto build_lists = [&](const std::vector<uint32_t>& el, int N, std::vector<uint32_t>& ptr, std::vector<uint32_t>& lst) {
        std::vector<uint32_t> cnt(nv + 1, 0);
        uint32_t              ne_ = (uint32_t)(el.size() / N);
        for (uint32_t e = 0; e < ne_; e++)
            for (int k = 0; k < N; k++) cnt[el[N * e + k] + 1]++;
        for (uint32_t i = 0; i < nv; i++) cnt[i + 1] += cnt[i];
        ptr = cnt;
        lst.assign(cnt[nv], 0);
        std::vector<uint32_t> fill(cnt.begin(), cnt.end() - 1);
        for (uint32_t e = 0; e < ne_; e++)
            for (int k = 0; k < N; k++) lst[fill[el[N * e + k]]++] = (e << 2) | (uint32_t)k;
    };
    build_lists(sp, 2, v_sp_ptr, v_sp);
    build_lists(sf, 3, v_sf_ptr, v_sf);
    build_lists(bh, 4, v_bh_ptr, v_bh);

    // SELL-16 layout
    nslices = (nv + kSlice - 1) / kSlice;
    sl_off.assign(nslices + 1, 0);
    for (uint32_t s = 0; s < nslices; s++)
    {
        uint32_t w = 0;
        for (uint32_t r = s * kSlice; r < std::min(nv, (s + 1) * kSlice); r++) w = std::max<uint32_t>(w, (uint32_t)adj[r].size());
        sl_off[s + 1] = sl_off[s] + w;
    }
    nblocks = sl_off[nslices] * kSlice;
    sell_col.assign(nblocks, 0);
    csr_to_sell.assign(csr.size(), 0xffffffffu);
    for (uint32_t s = 0; s < nslices; s++)
    {
        uint32_t w = sl_off[s + 1] - sl_off[s];
        for (uint32_t l = 0; l < (uint32_t)kSlice; l++)
        {
            uint32_t r = s * kSlice + l;
            for (uint32_t k = 0; k < w; k++)
            {
                uint32_t b = (sl_off[s] + k) * kSlice + l;
                if (r < nv && k < adj[r].size())
                {
                    sell_col[b]                  = adj[r][k];
                    csr_to_sell[csr[r] + k]      = b;
                }
                else
                    sell_col[b] = r < nv ? r : 0;  // padding: zero block against the row itself
            }
        }
    }
    // contributors per SELL block: springs of the row vertex in spring order, then faces, then
    // hinges (counted, then filled in the same visiting order). A spring's code is a hinge code
    // with both local indices 3, which no hinge block has (its two local indices differ).
    auto slot_of = [&](uint32_t r, uint32_t c) {
        const auto& l = adj[r];
        uint32_t    k = (uint32_t)(std::lower_bound(l.begin(), l.end(), c) - l.begin());
        return (sl_off[r / kSlice] + k) * kSlice + (r % kSlice);
    };
    auto visit = [&](auto&& emit) {
        for (uint32_t r = 0; r < nv; r++)
        {
            for (uint32_t p = v_sp_ptr[r]; p < v_sp_ptr[r + 1]; p++)
            {
                uint32_t e = v_sp[p] >> 2, a = v_sp[p] & 3;
                emit(slot_of(r, sp[2 * e + (a ^ 1u)]), 0x80000000u | (3u << 29) | (3u << 27) | e);
            }
            for (uint32_t p = v_sf_ptr[r]; p < v_sf_ptr[r + 1]; p++)
            {
                uint32_t f = v_sf[p] >> 2, a = v_sf[p] & 3;
                for (uint32_t b = 0; b < 3; b++)
                    if (b != a) emit(slot_of(r, sf[3 * f + b]), (a << 29) | (b << 27) | f);
            }
            for (uint32_t p = v_bh_ptr[r]; p < v_bh_ptr[r + 1]; p++)
            {
                uint32_t e = v_bh[p] >> 2, a = v_bh[p] & 3;
                for (uint32_t b = 0; b < 4; b++)
                    if (b != a) emit(slot_of(r, bh[4 * e + b]), 0x80000000u | (a << 29) | (b << 27) | e);
            }
        }
    };
    blk_ptr.assign(nblocks + 1, 0);
    visit([&](uint32_t blk, uint32_t) { blk_ptr[blk + 1]++; });
    for (uint32_t b = 0; b < nblocks; b++) blk_ptr[b + 1] += blk_ptr[b];
    blk_contrib.assign(blk_ptr[nblocks], 0);
    std::vector<uint32_t> fill(blk_ptr.begin(), blk_ptr.end() - 1);
    visit([&](uint32_t blk, uint32_t code) { blk_contrib[fill[blk]++] = code; });

    // affine bodies: mass matrix, orthogonality stiffness, SELL blocks of the body rows
    for (Body& b : bodies)
    {
        const uint32_t       mi = vert_mesh[b.v0];
        const lcsx_material& mt = meshes[mi].mat;
        float                m = 0.0f, mx[3] = {0, 0, 0}, mxx[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, vol = 0.0f;
        if (mt.body == 1)
            rigid_shell_mass(b, mi, vvol, body_vol, body_mass, m, mx, mxx, vol);
        else
            rigid_solid_mass(b, mi, face_mesh, m, mx, mxx, vol, mt.density);
        b.M[0] = m;
        for (int i = 0; i < 3; i++)
        {
            b.M[4 * (1 + i)] = mx[i];
            b.M[1 + i]       = mx[i];
            for (int j = 0; j < 3; j++) b.M[4 * (1 + i) + 1 + j] = mxx[i][j];
        }
        for (int i = 0; i < 4; i++) b.M[5 * i] = std::max(b.M[5 * i], 1.19209290E-7f);  // init_sim_data.cpp:694
        b.stiff = mt.rigid_stiffness * vol;
        int k   = 0;
        for (uint32_t ii = 0; ii < 4; ii++)
            for (uint32_t jj = 0; jj < 4; jj++)
                if (ii != jj) b.blk[k++] = slot_of(b.row0 + ii, b.row0 + jj);
    }
    cluster();
}

// Shell body (RigidMaterial is_shell, init_sim_data.cpp:600-640): mass carried by the vertices
// (the cloth vertex-mass rule), volume = area x thickness.
void Setup::rigid_shell_mass(const Body& b, uint32_t mi, const std::vector<float>& vvol, const std::vector<float>& body_vol,
                             const std::vector<float>& body_mass, float& m, float mx[3], float mxx[3][3], float& vol) const
{
    for (uint32_t i = b.v0; i < b.v1; i++)
    {
        float vm   = (vvol[i] / body_vol[mi]) * body_mass[mi];
        float X[3] = {rest_x[3 * i], rest_x[3 * i + 1], rest_x[3 * i + 2]};
        m += vm;
        for (int a = 0; a < 3; a++)
        {
            mx[a] += vm * X[a];
            for (int c = 0; c < 3; c++) mxx[a][c] = mxx[a][c] + vm * (X[a] * X[c]);
        }
    }
    vol = body_vol[mi];
}

// Solid body (compute_trimesh_dyadic_mass, init_sim_data.cpp:51-188): mass and moments of the
// enclosed solid by surface integrals over its triangles, volume likewise.
void Setup::rigid_solid_mass(const Body& b, uint32_t mi, const std::vector<uint32_t>& face_mesh_, float& m, float mx[3],
                             float mxx[3][3], float& vol, float rho) const
{
    (void)b;
    auto P = [&](uint32_t v) { return mk(rest_x[3 * v], rest_x[3 * v + 1], rest_x[3 * v + 2]); };
    for (uint32_t f = 0; f < nf; f++)
    {
        if (face_mesh_[f] != mi) continue;
        const f3 p0 = P(faces[3 * f]), p1 = P(faces[3 * f + 1]), p2 = P(faces[3 * f + 2]);
        const f3 N  = cross(p1 - p0, p2 - p0);
        m += rho * dot(p0, N) / 6.0;
        vol += dot(p0, N) / 6.0f;
        const float a0[3] = {p0.x, p0.y, p0.z}, a1[3] = {p1.x, p1.y, p1.z}, a2[3] = {p2.x, p2.y, p2.z};
        const float n[3]  = {N.x, N.y, N.z};
        for (int a = 0; a < 3; a++)
        {
            float V = 0.0;
            V += a0[a] * a0[a] / 12;
            V += a0[a] * a1[a] / 12;
            V += a0[a] * a2[a] / 12;
            V += a1[a] * a1[a] / 12;
            V += a1[a] * a2[a] / 12;
            V += a2[a] * a2[a] / 12;
            mx[a] += rho / 2 * n[a] * V;
        }
        for (int a = 0; a < 3; a++)
        {
            float V = 0.0;
            float s0 = a0[a] * a0[a], s1 = a1[a] * a1[a], s2 = a2[a] * a2[a];
            float c0 = s0 * a0[a], c1 = s1 * a1[a], c2 = s2 * a2[a];
            V += c0 / 20;
            V += s0 * a1[a] / 20;
            V += s0 * a2[a] / 20;
            V += a0[a] * s1 / 20;
            V += a0[a] * a1[a] * a2[a] / 20;
            V += a0[a] * s2 / 20;
            V += c1 / 20;
            V += s1 * a2[a] / 20;
            V += a1[a] * s2 / 20;
            V += c2 / 20;
            mxx[a][a] += rho / 3 * n[a] * V;
        }
        auto Q = [&](int a, int c) {
            float V = 0.0;
            float s0 = a0[a] * a0[a], s1 = a1[a] * a1[a], s2 = a2[a] * a2[a];
            V += s0 * a0[c] / 20;
            V += s0 * a1[c] / 60;
            V += s0 * a2[c] / 60;
            V += a0[a] * a0[c] * a1[a] / 30;
            V += a0[a] * a0[c] * a2[a] / 30;
            V += a0[a] * a1[a] * a1[c] / 30;
            V += a0[a] * a1[a] * a2[c] / 60;
            V += a0[a] * a1[c] * a2[a] / 60;
            V += a0[a] * a2[a] * a2[c] / 30;
            V += a0[c] * s1 / 60;
            V += a0[c] * a1[a] * a2[a] / 60;
            V += a0[c] * s2 / 60;
            V += s1 * a1[c] / 20;
            V += s1 * a2[c] / 60;
            V += a1[a] * a1[c] * a2[a] / 30;
            V += a1[a] * a2[a] * a2[c] / 30;
            V += a1[c] * s2 / 60;
            V += s2 * a2[c] / 20;
            return rho / 2 * n[a] * V;
        };
        mxx[0][1] += Q(0, 1);
        mxx[0][2] += Q(0, 2);
        mxx[1][2] += Q(1, 2);
        mxx[1][0] = mxx[0][1];
        mxx[2][0] = mxx[0][2];
        mxx[2][1] = mxx[1][2];
    }
}

}  // namespace lcsx
