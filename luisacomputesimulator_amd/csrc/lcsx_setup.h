// Host-side scene setup for the solver: topology, per-vertex quantities, culled elements,
// the material block-sparse structure (reference CSR + device SELL-64 layout) and the
// gather lists that let every output block be owned by exactly one thread.
#pragma once
#include <stdint.h>
#include <string>
#include <vector>
#include "../../include/lcsx.h"

namespace lcsx
{

struct MeshDesc
{
    std::vector<float>            x;     // world rest positions (3 per vertex)
    std::vector<int32_t>          tris;  // local indices
    lcsx_material                 mat;
    std::vector<uint32_t>         pinned;  // local ids in selection order
    std::vector<lcsx_fixed_anim>  anim;
    std::vector<float>            explicit_targets;  // optional (3 per pinned vertex)
    uint32_t                      scene = 0;  // batch member (meshes are added scene by scene)
};

constexpr int kSlice = 16;  // SELL slice height: 16 rows, read by one wavefront with 4 lanes per row

struct Setup
{
    uint32_t nv = 0, nf = 0, ne = 0, nh = 0;
    std::vector<float>    rest_x;                  // 3 nv
    std::vector<uint32_t> faces, edges, hinges;    // 3 nf, 2 ne, 4 nh (all elements, for collision)
    std::vector<uint32_t> vert_mesh, face_mesh, edge_mesh;
    std::vector<float>    face_area, edge_area, vert_area, vert_mass, offset, dhat;
    std::vector<uint8_t>  is_fixed;
    std::vector<uint32_t> fixed_verts;                   // pin order
    std::vector<uint32_t> fixed_mesh, fixed_local;        // mesh id and index in that mesh's pin list
    std::vector<lcsx_fixed_anim> fixed_anim;
    // culled material elements
    std::vector<uint32_t> sf;                      // 3 per stretch face
    std::vector<float>    sf_Dm, sf_area, sf_mu, sf_lambda;
    std::vector<uint32_t> sp;                      // stretch springs, 2 per spring (edge order)
    std::vector<float>    sp_rest, sp_k;           // rest length, stiffness
    std::vector<uint32_t> bh;                      // 4 per bending hinge
    std::vector<float>    bh_angle, bh_hbar, bh_k;
    // reference CSR of material neighbours: nv+1 prefixes (offset by nv+1), then sorted columns
    std::vector<uint32_t> csr;
    // vertex -> (element << 2 | local) gather lists, in element order
    std::vector<uint32_t> v_sf_ptr, v_sf, v_bh_ptr, v_bh, v_sp_ptr, v_sp;
    // SELL-64 layout of the off-diagonal blocks: slice s holds rows [64 s, 64 s + 64), width
    // sl_off[s+1] - sl_off[s]; block (row r, k-th neighbour) lives at (sl_off[s] + k) * 64 + (r % 64).
    uint32_t              nslices = 0, nblocks = 0;
    std::vector<uint32_t> sl_off, sell_col;
    std::vector<uint32_t> csr_to_sell;             // for each CSR slot (header slots: kInvalid)
    // per SELL block: contributors (bit 31 hinge, bits 29-30 local a, 27-28 local b, 0-26 element)
    std::vector<uint32_t> blk_ptr, blk_contrib;
    uint32_t              max_degree = 0;
    // batch of independent scenes: vertices, faces and edges of scene s are the ranges
    // [sc_v0[s], sc_v0[s+1]) etc. Row blocks of 256 vertices never straddle two scenes, so every
    // per-block partial sum belongs to one scene: block b covers rows [rb_row0[b], ..) of scene
    // rb_scene[b], and scene s owns blocks [sc_rb0[s], sc_rb0[s+1]).
    uint32_t              nscenes = 1;
    std::vector<uint32_t> sc_v0, sc_f0, sc_e0, sc_rb0, vert_scene, rb_scene, rb_row0;
    std::vector<uint32_t> sc_verts;  // vertex rows per scene (body rows excluded)
    uint32_t              n_rb = 0;
    // affine bodies: each rigid mesh is a body with four rows (p, a0, a1, a2) placed after the
    // vertex rows of its scene; its vertices keep rows of their own and follow x = p + A X.
    // row_kind: 0 soft vertex, 1 rigid vertex, 2 + k body row k.
    struct Body
    {
        uint32_t row0, v0, v1, fixed;
        float    stiff;    // kappa * volume
        float    M[16];    // 4x4 mass matrix (times I3)
        uint32_t blk[12];  // SELL blocks (ii, jj != ii), row-major
    };
    std::vector<Body>     bodies;
    std::vector<uint8_t>  row_kind;
    std::vector<uint32_t> vert_body;  // per row: body id (rigid vertex or body row) or ~0u
    std::vector<float>    body_X;     // per row: body-frame position of a rigid vertex (3)

    // an edge or a face listed twice (an edge of three or more faces is), or an element that names a vertex
    // twice: contacts of one row may then have equal vertex ids
    bool repeats = false;

    // points (rows of kind 0 and 1), faces and edges, mesh by mesh and along a Morton curve through each
    // mesh's rest pose: neighbours in these lists are neighbours in space, however a mesh moves. Every scene
    // is padded with kInvalid, to whole wavefronts of 64 points and whole blocks of kClusterLeaves elements;
    // _block: the first block of each scene, and the end.
    std::vector<uint32_t> cluster_v, cluster_f, cluster_e, cluster_f_block, cluster_e_block;
    bool cluster_f_use = true, cluster_e_use = true;  // whether the queries walk the blocks (cluster)

    void build(const std::vector<MeshDesc>& meshes);

private:
    void cluster();
    void rigid_shell_mass(const Body& b, uint32_t mi, const std::vector<float>& vvol, const std::vector<float>& body_vol,
                          const std::vector<float>& body_mass, float& m, float mx[3], float mxx[3][3], float& vol) const;
    void rigid_solid_mass(const Body& b, uint32_t mi, const std::vector<uint32_t>& face_mesh_, float& m, float mx[3],
                          float mxx[3][3], float& vol, float rho) const;
};

// Pinned-target animation (reference init_mesh_data.h:56-93, luisa::rotation axis-angle).
void animate_target(const lcsx_fixed_anim& a, float t, const float in[3], float out[3]);
void pin_by_method(MeshDesc& m, int method, float range, const lcsx_fixed_anim& anim);

}  // namespace lcsx
