// Newton-step kernels for gfx950: material evaluation and owner-computes assembly, DCD/CCD
// narrow phase, contact assembly, SELL-16 block SpMV, block-Jacobi PCG and line search.
// Reference counterparts are cited per kernel (paths relative to the reference root).
#include <hip/hip_ext.h>
#include <atomic>
#include <type_traits>
#include "lcsx_fp64.h"
#include "lcsx_internal.h"
#include "lcsx_kernels.h"
#include "lcsx_pcg_grid.h"
#include "lcsx_physics.h"

namespace lcsx
{

namespace
{
constexpr int kB = 256;

// Makes the kernel-argument values named here live in scalar registers from the kernel's first
// instructions. The compiler otherwise loads each argument where it is first used, and in a kernel
// whose work starts behind branches (row or contact block, one scene or several) those loads form
// a chain of scalar-memory round trips before the first vector load (about 1.5 us of a 10 us
// SpMV launch). An empty asm statement that takes the values as scalar operands makes all the
// argument loads issue together, with one wait.
LCSX_D void pin_sgpr(uint32_t v) { asm volatile("" ::"s"(v)); }
LCSX_D void pin_sgpr(float v) { asm volatile("" ::"s"(v)); }
LCSX_D void pin_sgpr(const void* p) { asm volatile("" ::"s"(p)); }
template <class T0, class T1, class... T>
LCSX_D void pin_sgpr(T0 v0, T1 v1, T... v)
{
    pin_sgpr(v0);
    pin_sgpr(v1, v...);
}

// Block-wide sum (256 threads); the result is valid in thread 0. Fixed order: wave butterflies,
// then the four wave sums in wave order.
LCSX_D float block_sum(float v, float* sh)
{
    v     = wave_sum(v);
    int w = threadIdx.x >> 6;
    if (lane_id() == 0) sh[w] = v;
    __syncthreads();
    float r = 0.0f;
    if (threadIdx.x == 0) r = ((sh[0] + sh[1]) + sh[2]) + sh[3];
    __syncthreads();
    return r;
}

// Sum of n partials in a fixed order (strided per thread, then block_sum), returned in every
// thread of the block. Every block of a launch computes the same value: the PCG scalars are
// reduced this way from the previous launch's partials instead of by a last-block hand-off,
// which would need device-scope fences (L2 write-back across XCDs) and a contended ticket.
LCSX_D float block_reduce_all(const float* __restrict__ part, uint32_t n, float* sh)
{
    __shared__ float bc;
    float            v = 0.0f;
    for (uint32_t i = threadIdx.x; i < n; i += kB) v = v + part[i];
    v = block_sum(v, sh);
    if (threadIdx.x == 0) bc = v;
    __syncthreads();
    v = bc;
    __syncthreads();
    return v;
}

// Sum of the partials [b0, e0) then [b1, e1), as block_reduce_all over their concatenation.
LCSX_D float block_reduce_ranges(const float* __restrict__ part, uint32_t b0, uint32_t e0, uint32_t b1, uint32_t e1,
                                 float* sh)
{
    __shared__ float bc;
    const uint32_t   n0 = e0 - b0, n = n0 + (e1 - b1);
    float            v  = 0.0f;
    for (uint32_t i = threadIdx.x; i < n; i += kB) v = v + part[i < n0 ? b0 + i : b1 + (i - n0)];
    v = block_sum(v, sh);
    if (threadIdx.x == 0) bc = v;
    __syncthreads();
    v = bc;
    __syncthreads();
    return v;
}

// block_reduce_ranges in two steps: the first kPre partials of each thread are requested first
// (before a flag or another wait), then summed with the rest in the same order, so the result is
// that of block_reduce_ranges.
constexpr int kPre = 4;
struct PrePartials
{
    float    v[kPre];
    uint32_t b0, n0, b1, n;
};
LCSX_D PrePartials prefetch_ranges(const float* __restrict__ part, uint32_t b0, uint32_t e0, uint32_t b1, uint32_t e1)
{
    PrePartials p;
    p.b0 = b0;
    p.n0 = e0 - b0;
    p.b1 = b1;
    p.n  = p.n0 + (e1 - b1);
#pragma unroll
    for (int u = 0; u < kPre; u++)
    {
        const uint32_t i = threadIdx.x + (uint32_t)u * kB;
        p.v[u]           = i < p.n ? part[i < p.n0 ? b0 + i : b1 + (i - p.n0)] : 0.0f;
    }
    return p;
}
LCSX_D float reduce_prefetched(const float* __restrict__ part, const PrePartials& p, float* sh)
{
    __shared__ float bc;
    float            v = 0.0f;
#pragma unroll
    for (int u = 0; u < kPre; u++)
        if (threadIdx.x + (uint32_t)u * kB < p.n) v = v + p.v[u];
    // the rest in batches, every load of a batch in flight (a long list of contact chunks)
    constexpr uint32_t kIn = 12u;
    for (uint32_t i = threadIdx.x + kPre * kB; i < p.n; i += kIn * kB)
    {
        float w[kIn];
#pragma unroll
        for (uint32_t u = 0; u < kIn; u++)
        {
            const uint32_t q = i + u * kB;
            w[u]             = q < p.n ? part[q < p.n0 ? p.b0 + q : p.b1 + (q - p.n0)] : 0.0f;
        }
#pragma unroll
        for (uint32_t u = 0; u < kIn; u++)
            if (i + u * kB < p.n) v = v + w[u];
    }
    v = block_sum(v, sh);
    if (threadIdx.x == 0) bc = v;
    __syncthreads();
    v = bc;
    __syncthreads();
    return v;
}

// Row block of a scene-aligned launch: its scene and this thread's row (valid below the end of
// the block or of the scene).
struct RowBlk
{
    uint32_t scene, row;
    bool     valid;
};
LCSX_D RowBlk row_blk(const SegView& g)
{
    RowBlk   r;
    uint32_t b = blockIdx.x;
    r.scene    = g.rb_scene[b];
    r.row      = g.rb_row0[b] + threadIdx.x;
    r.valid    = r.row < g.sc_v0[r.scene + 1];
    return r;
}

LCSX_D RowBlk row_blk_at(const SegView& g, uint32_t b)
{
    RowBlk r;
    r.scene = g.rb_scene[b];
    r.row   = g.rb_row0[b] + threadIdx.x;
    r.valid = r.row < g.sc_v0[r.scene + 1];
    return r;
}

// row_blk_at without memory reads when the launch holds one scene of n rows: its row blocks are
// then the consecutive 256-row blocks of [0, n), so the row operands can be requested at once
// instead of after the block's scene and first row arrive.
LCSX_D RowBlk row_blk_fast(const SegView& g, uint32_t n, uint32_t b)
{
    if (g.nscenes == 1u)
    {
        const uint32_t row = b * 256u + threadIdx.x;
        return RowBlk{0u, row, row < n};
    }
    return row_blk_at(g, b);
}

// [first, end) of scene sc's row blocks (sc_rb0), with no read for a single scene.
LCSX_D uint32_t scene_rb0(const SegView& g, uint32_t sc) { return g.nscenes == 1u ? (sc == 0u ? 0u : g.n_rb) : g.sc_rb0[sc]; }

// PCG direction vectors p: FP32 triples in 16-byte rows (the fourth word is zero).
LCSX_D f3 ld4(const float* p, uint32_t i)
{
    const float4 v = reinterpret_cast<const float4*>(p)[i];
    return mk(v.x, v.y, v.z);
}
LCSX_D void st4(float* p, uint32_t i, f3 v) { reinterpret_cast<float4*>(p)[i] = make_float4(v.x, v.y, v.z, 0.0f); }

// The flag read once per block (a launch may set it while other blocks start).
// A flag that no block of the current launch writes (set by an earlier launch): every thread reads
// it directly, without the barriers of block_flag, and all threads of a block see the same value.
LCSX_D bool launch_flag(const uint32_t* flag) { return *flag != 0u; }

LCSX_D bool block_flag(const uint32_t* flag)
{
    __shared__ uint32_t f;
    if (threadIdx.x == 0) f = *flag;
    __syncthreads();
    bool r = f != 0u;
    __syncthreads();
    return r;
}

LCSX_D m3 ld_planes(const float* __restrict__ P, size_t stride, size_t i)
{
    m3 a;
#pragma unroll
    for (int c = 0; c < 9; c++) a.m[c] = P[c * stride + i];
    return a;
}
LCSX_D void st_planes(float* __restrict__ P, size_t stride, size_t i, const m3& a)
{
#pragma unroll
    for (int c = 0; c < 9; c++) P[c * stride + i] = a.m[c];
}

// ---------------------------------------------------------------- frame
// solver_interface.cpp:130-162: pinned velocity = (target - x) / dt
__global__ void k_pin_velocity(uint32_t nfix, const uint32_t* __restrict__ ids, const float* __restrict__ targets,
                               const float* __restrict__ x, float* __restrict__ v, float dt)
{
    uint32_t k = blockIdx.x * kB + threadIdx.x;
    if (k >= nfix) return;
    uint32_t i = ids[k];
    st3(v, i, (ld3(targets, k) - ld3(x, i)) / dt);
}

// fn_predict_position, newton_solver.cpp:577-608
// (+ fn_abd_predict_position, newton_solver.cpp:640-675: gravity on a body's translation row only)
__global__ void k_predict(uint32_t nv, const float* __restrict__ x_step, const float* __restrict__ v,
                          const uint8_t* __restrict__ fixed, const uint8_t* __restrict__ kind, float h, f3 g,
                          float* __restrict__ x_iter, float* __restrict__ x_tilde, float* __restrict__ x)
{
    uint32_t i = blockIdx.x * kB + threadIdx.x;
    if (i >= nv) return;
    f3   xs   = ld3(x_step, i), vi = ld3(v, i);
    bool grav = kind[i] <= 2u;
    f3   vp   = fixed[i] ? vi : (grav ? vi + h * g : vi);
    st3(x_iter, i, xs);
    st3(x_tilde, i, xs + h * vp);
    st3(x, i, xs);
}

// fn_update_velocity, newton_solver.cpp:610-636
__global__ void k_frame_end(uint32_t nv, float* __restrict__ x_step, const float* __restrict__ x, float* __restrict__ v,
                            float h, float damp)
{
    uint32_t i = blockIdx.x * kB + threadIdx.x;
    if (i >= nv) return;
    f3 xe = ld3(x, i);
    st3(v, i, ((xe - ld3(x_step, i)) / h) * damp);
    st3(x_step, i, xe);
}

// ---------------------------------------------------------------- material
// fn_evaluate_spring, newton_solver.cpp:1002-1048. Staging per spring (16 floats): the gradient of
// its first vertex (the second's is the negation), then the row-major block He (the diagonal
// blocks of both vertices are He, the off-diagonal ones -He). The length is clamped below at
// FLT_EPSILON and the Hessian's lateral term at 0 (a compressed spring keeps its PSD part).
constexpr float kSpringMinLength = 1.19209290e-7f;
__global__ __launch_bounds__(kB) void k_spring_stage(uint32_t nsp, const uint32_t* __restrict__ sp,
                                                      const float2* __restrict__ c, const float* __restrict__ x,
                                                      float* __restrict__ stage)
{
    uint32_t e = blockIdx.x * kB + threadIdx.x;
    if (e >= nsp) return;
    const f3     diff = ld3(x, sp[2 * e]) - ld3(x, sp[2 * e + 1]);
    const float2 rk   = c[e];
    const float  l    = fmaxf(sqrtf(dot(diff, diff)), kSpringMinLength);
    const float  C    = l - rk.x;
    const f3     dir  = diff / l;
    const float  xinv = 1.0f / l, xsi = xinv * xinv;
    const f3     g    = (rk.y * dir) * C;
    const float  s1 = rk.y * xsi, s2 = rk.y * fmaxf(1.0f - rk.x * xinv, 0.0f);
    const float  d[3] = {diff.x, diff.y, diff.z};
    float*       S    = stage + 16 * (size_t)e;
    S[0] = g.x;
    S[1] = g.y;
    S[2] = g.z;
    for (int r = 0; r < 3; r++)
        for (int cc = 0; cc < 3; cc++)
        {
            const float o    = d[r] * d[cc];
            S[3 + 3 * r + cc] = s1 * o + s2 * ((r == cc ? 1.0f : 0.0f) - xsi * o);
        }
}

// fn_evaluate_stretch_face, newton_solver.cpp:1053-1100. Staging per face (64 floats):
// g0 g1 g2 | H00 H11 H22 | H01 H02 H12 (row-major 3x3 blocks), 1 float pad.
__global__ __launch_bounds__(kB) void k_face_stage(uint32_t nsf, const uint32_t* __restrict__ sf,
                                                    const float4* __restrict__ Dm, const float4* __restrict__ c,
                                                    const float* __restrict__ x, float* __restrict__ stage)
{
    uint32_t f = blockIdx.x * kB + threadIdx.x;
    if (f >= nsf) return;
    float4  d4 = Dm[f], c4 = c[f];
    float   d[4] = {d4.x, d4.y, d4.z, d4.w};
    FaceOut o;
    bw_face(ld3(x, sf[3 * f]), ld3(x, sf[3 * f + 1]), ld3(x, sf[3 * f + 2]), d, c4.y, c4.z, c4.x, o);
    float out[64];
    for (int a = 0; a < 3; a++)
    {
        out[3 * a] = o.g[a].x;
        out[3 * a + 1] = o.g[a].y;
        out[3 * a + 2] = o.g[a].z;
    }
    for (int a = 0; a < 3; a++)
        for (int k = 0; k < 9; k++) out[9 + 9 * a + k] = o.H[a][a].m[k];
    for (int k = 0; k < 9; k++)
    {
        out[36 + k] = o.H[0][1].m[k];
        out[45 + k] = o.H[0][2].m[k];
        out[54 + k] = o.H[1][2].m[k];
    }
    out[63]   = 0.0f;
    float4* S = reinterpret_cast<float4*>(stage + 64 * (size_t)f);
#pragma unroll
    for (int k = 0; k < 16; k++) S[k] = make_float4(out[4 * k], out[4 * k + 1], out[4 * k + 2], out[4 * k + 3]);
}

// fn_evaluate_bending, newton_solver.cpp:1102-1172. Staging per hinge (16 floats):
// dtheta/dx_0..3 (12), stiff, stiff * (theta - theta_rest), 2 pad.
__global__ __launch_bounds__(kB) void k_hinge_stage(uint32_t nbh, const uint32_t* __restrict__ bh,
                                                     const float4* __restrict__ c, float scaling,
                                                     const float* __restrict__ x, float* __restrict__ stage)
{
    uint32_t e = blockIdx.x * kB + threadIdx.x;
    if (e >= nbh) return;
    f3 p0 = ld3(x, bh[4 * e]), p1 = ld3(x, bh[4 * e + 1]), p2 = ld3(x, bh[4 * e + 2]), p3 = ld3(x, bh[4 * e + 3]);
    f3 g[4];
    float  ang = dihedral_angle(p0, p1, p2, p3);
    dihedral_grad(p0, p1, p2, p3, g);
    float4 cc    = c[e];  // rest angle, h_bar, stiffness
    float  stiff = (cc.z * scaling) * cc.y;
    float  coef  = stiff * (ang - cc.x);
    float4* S    = reinterpret_cast<float4*>(stage + 16 * (size_t)e);
    S[0]         = make_float4(g[0].x, g[0].y, g[0].z, g[1].x);
    S[1]         = make_float4(g[1].y, g[1].z, g[2].x, g[2].y);
    S[2]         = make_float4(g[2].z, g[3].x, g[3].y, g[3].z);
    S[3]         = make_float4(stiff, coef, 0.0f, 0.0f);
}

LCSX_D f3 hinge_g(const float* H, uint32_t a) { return mk(H[3 * a], H[3 * a + 1], H[3 * a + 2]); }

// Inertia (fn_evaluate_inertia 819-850), ground barrier (883-950) and the per-vertex part of the
// assembly (compile_assembly 705-814): gradient and diagonal block, faces then hinges in order.
__global__ __launch_bounds__(kB) void k_vert_assemble(VertArgs a)
{
    uint32_t i = blockIdx.x * kB + threadIdx.x;
    if (i >= a.nv) return;
    const uint8_t kind = a.row_kind[i];
    if (kind >= 2u) return;  // body rows: k_abd_material
    if (kind == 1u)
    {
        // a rigid vertex follows its body: an identity row that solves to dx = 0
        m3 I = m3_zero();
        I.m[0] = I.m[4] = I.m[8] = 1.0f;
        st3(a.cgB, i, mk(0.0f, 0.0f, 0.0f));
        st_planes(a.diag, a.nv, i, I);
        if (a.diag_mat) st_planes(a.diag_mat, a.nv, i, I);
        return;
    }
    float m    = a.mass[i];
    f3    grad = ((-m) * a.h2inv) * (ld3(a.x, i) - ld3(a.x_tilde, i));
    m3    H    = m3_zero();
    float d    = (1.0f * m) * a.h2inv;
    H.m[0] = H.m[4] = H.m[8] = d;
    bool fixed = a.fixed[i] != 0;
    if (fixed)
    {
        grad = grad + a.kD * grad;
        for (int k = 0; k < 9; k++) H.m[k] = H.m[k] + a.kD * H.m[k];
    }
    if (a.use_floor && !fixed)
    {
        float dh = a.dhat[i], th = a.offset[i], dist = a.x[3 * (size_t)i + 1] - a.floor_y;
        if (dist - th < dh)
        {
            float k1, k2;
            ground_k(a.quadratic, dist, th, dh, a.kappa * a.area[i], k1, k2);
            grad.y = grad.y - k1;
            H.m[4] = H.m[4] + k2;
        }
    }
    for (uint32_t p = a.v_sp_ptr[i]; p < a.v_sp_ptr[i + 1]; p++)
    {
        uint32_t     e = a.v_sp[p] >> 2, l = a.v_sp[p] & 3u;
        const float* S = a.spring_stage + 16 * (size_t)e;
        const f3     g = mk(S[0], S[1], S[2]);
        grad           = grad + (l == 0 ? -g : g);
        for (int k = 0; k < 9; k++) H.m[k] = H.m[k] + S[3 + k];
    }
    for (uint32_t p = a.v_sf_ptr[i]; p < a.v_sf_ptr[i + 1]; p++)
    {
        uint32_t     f = a.v_sf[p] >> 2, l = a.v_sf[p] & 3u;
        const float* S = a.face_stage + 64 * (size_t)f;
        grad           = grad + (-mk(S[3 * l], S[3 * l + 1], S[3 * l + 2]));
        for (int k = 0; k < 9; k++) H.m[k] = H.m[k] + S[9 + 9 * l + k];
    }
    for (uint32_t p = a.v_bh_ptr[i]; p < a.v_bh_ptr[i + 1]; p++)
    {
        uint32_t     e = a.v_bh[p] >> 2, l = a.v_bh[p] & 3u;
        const float* S = a.hinge_stage + 16 * (size_t)e;
        f3           g = hinge_g(S, l);
        float        stiff = S[12], coef = S[13];
        grad               = grad + (-(coef * g));
        float gv[3]        = {g.x, g.y, g.z};
        for (int r = 0; r < 3; r++)
            for (int cc = 0; cc < 3; cc++) H.m[3 * r + cc] = H.m[3 * r + cc] + stiff * (gv[r] * gv[cc]);
    }
    st3(a.cgB, i, grad);
    st_planes(a.diag, a.nv, i, H);
    if (a.diag_mat) st_planes(a.diag_mat, a.nv, i, H);
}

// Off-diagonal blocks: one thread per SELL block sums its contributors in order
// (faces of the row vertex, then hinges) and writes the block once.
__global__ __launch_bounds__(kB) void k_offdiag(uint32_t nblocks, const uint32_t* __restrict__ ptr,
                                                 const uint32_t* __restrict__ con, const float* __restrict__ spring_stage,
                                                 const float* __restrict__ face_stage,
                                                 const float* __restrict__ hinge_stage, float* __restrict__ val)
{
    uint32_t b = blockIdx.x * kB + threadIdx.x;
    if (b >= nblocks) return;
    m3 H = m3_zero();
    for (uint32_t p = ptr[b]; p < ptr[b + 1]; p++)
    {
        uint32_t c = con[p], el = c & 0x07ffffffu, la = (c >> 29) & 3u, lb = (c >> 27) & 3u;
        if ((c & 0x80000000u) && la == 3u && lb == 3u)
        {
            // a spring (no hinge block pairs a local index with itself)
            const float* S = spring_stage + 16 * (size_t)el;
            for (int k = 0; k < 9; k++) H.m[k] = H.m[k] + (-S[3 + k]);
        }
        else if (c & 0x80000000u)
        {
            const float* S = hinge_stage + 16 * (size_t)el;
            f3    ga = hinge_g(S, la), gb = hinge_g(S, lb);
            float st = S[12];
            float u[3] = {ga.x, ga.y, ga.z}, w[3] = {gb.x, gb.y, gb.z};
            for (int r = 0; r < 3; r++)
                for (int cc = 0; cc < 3; cc++) H.m[3 * r + cc] = H.m[3 * r + cc] + st * (u[r] * w[cc]);
        }
        else
        {
            const float* S   = face_stage + 64 * (size_t)el;
            uint32_t     lo  = la < lb ? la : lb, hi = la < lb ? lb : la;
            uint32_t     off = 36 + 9 * (lo == 0 ? (hi == 1 ? 0 : 1) : 2);
            if (la < lb)
                for (int k = 0; k < 9; k++) H.m[k] = H.m[k] + S[off + k];
            else
                for (int r = 0; r < 3; r++)
                    for (int cc = 0; cc < 3; cc++) H.m[3 * r + cc] = H.m[3 * r + cc] + S[off + 3 * cc + r];
        }
    }
    st_planes(val, nblocks, b, H);
}

// ---------------------------------------------------------------- affine bodies
LCSX_D m3 m3_diag(float d)
{
    m3 a   = m3_zero();
    a.m[0] = a.m[4] = a.m[8] = d;
    return a;
}
LCSX_D m3 m3_add(const m3& a, const m3& b)
{
    m3 o;
    for (int k = 0; k < 9; k++) o.m[k] = a.m[k] + b.m[k];
    return o;
}
LCSX_D m3 m3_scale(float s, const m3& a)
{
    m3 o;
    for (int k = 0; k < 9; k++) o.m[k] = s * a.m[k];
    return o;
}
LCSX_D m3 m3_outer(f3 u, f3 v)
{
    float a[3] = {u.x, u.y, u.z}, b[3] = {v.x, v.y, v.z};
    m3    o;
    for (int r = 0; r < 3; r++)
        for (int c = 0; c < 3; c++) o.m[3 * r + c] = a[r] * b[c];
    return o;
}
LCSX_D m3 m3_transpose(const m3& a)
{
    m3 o;
    for (int r = 0; r < 3; r++)
        for (int c = 0; c < 3; c++) o.m[3 * r + c] = a.m[3 * c + r];
    return o;
}

// One thread per body: fn_evaluate_abd_inertia (newton_solver.cpp:1176-1245), _orthogonality
// (1246-1335), _ground_collision over the body's vertices (1336-1413) and the assembly of its 16
// blocks (fn_material_energy_assembly_affine_body, 803-813): cgB = -gradient, the four diagonal
// blocks, the twelve off-diagonal blocks into the SELL planes. Block order: diagonal blocks,
// then (ii, jj != ii) row-major.
__global__ __launch_bounds__(kB) void k_abd_material(AbdArgs a)
{
    uint32_t bi = blockIdx.x * kB + threadIdx.x;
    if (bi >= a.nb) return;
    const BodyDev& B = a.bodies[bi];
    f3             q[4], dq[4], g[4];
    for (int k = 0; k < 4; k++)
    {
        q[k]  = ld3(a.x, B.row0 + k);
        dq[k] = q[k] - ld3(a.x_tilde, B.row0 + k);
        g[k]  = mk(0.0f, 0.0f, 0.0f);
    }
    for (int ii = 0; ii < 4; ii++)
        for (int jj = 0; jj < 4; jj++) g[ii] = g[ii] + B.M[4 * ii + jj] * dq[jj];
    const float ah = (B.fixed ? (1.0f + a.kD) : 1.0f) * a.h2inv;
    f3          G[4];
    m3          H[16];
    for (int k = 0; k < 4; k++)
    {
        G[k] = ah * g[k];
        H[k] = m3_diag(ah * B.M[5 * k]);
    }
    int idx = 4;
    for (int ii = 0; ii < 4; ii++)
        for (int jj = 0; jj < 4; jj++)
            if (ii != jj) H[idx++] = m3_diag(ah * B.M[4 * ii + jj]);
    // orthogonality of A = (a0 a1 a2): 4 kappa V (sum_j (a_i . a_j) a_j - a_i) and exact Hessian
    const f3 A[3] = {q[1], q[2], q[3]};
    const float s4 = 4.0f * B.stiff;
    for (int ii = 0; ii < 3; ii++)
    {
        f3 grad = -1.0f * A[ii];
        for (int jj = 0; jj < 3; jj++) grad = grad + dot(A[ii], A[jj]) * A[jj];
        G[1 + ii] = G[1 + ii] + s4 * grad;
    }
    m3 oh[6];
    int o = 0;
    for (int ii = 0; ii < 3; ii++)
        for (int jj = ii; jj < 3; jj++)
        {
            m3 h;
            if (ii == jj)
            {
                h = m3_add(m3_outer(A[ii], A[ii]), m3_diag(dot(A[ii], A[ii]) - 1.0f));
                for (int kk = 0; kk < 3; kk++) h = m3_add(h, m3_outer(A[kk], A[kk]));
            }
            else
                h = m3_add(m3_outer(A[jj], A[ii]), m3_diag(dot(A[ii], A[jj])));
            oh[o++] = m3_add(m3_zero(), m3_scale(s4, h));
        }
    H[1]  = m3_add(H[1], oh[0]);
    H[8]  = m3_add(H[8], oh[1]);
    H[9]  = m3_add(H[9], oh[2]);
    H[11] = m3_add(H[11], m3_transpose(oh[1]));
    H[2]  = m3_add(H[2], oh[3]);
    H[12] = m3_add(H[12], oh[4]);
    H[14] = m3_add(H[14], m3_transpose(oh[2]));
    H[15] = m3_add(H[15], m3_transpose(oh[4]));
    H[3]  = m3_add(H[3], oh[5]);
    // ground barrier of the body's free vertices, lifted with weights (1, X)
    if (a.use_floor)
        for (uint32_t v = B.v0; v < B.v1; v++)
        {
            if (a.fixed[v]) continue;
            float dist = a.x[3 * (size_t)v + 1] - a.floor_y, th = a.offset[v], dh = a.dhat[v];
            if (!(dist - th < dh)) continue;
            const f3    n     = mk(0.0f, 1.0f, 0.0f);
            float       k1, k2;
            ground_k(a.quadratic, dist, th, dh, a.kappa * a.area[v], k1, k2);
            f3          gr    = k1 * n;
            m3          hs    = m3_scale(k2, m3_outer(n, n));
            const float w[4]  = {1.0f, a.body_X[3 * (size_t)v], a.body_X[3 * (size_t)v + 1], a.body_X[3 * (size_t)v + 2]};
            int         id    = 4;
            for (int ii = 0; ii < 4; ii++)
            {
                G[ii] = G[ii] + w[ii] * gr;
                for (int jj = 0; jj < 4; jj++)
                {
                    m3 hh = m3_scale(w[ii] * w[jj], hs);
                    if (ii == jj) H[ii] = m3_add(H[ii], hh);
                    else
                    {
                        H[id] = m3_add(H[id], hh);
                        id++;
                    }
                }
            }
        }
    for (int k = 0; k < 4; k++)
    {
        uint32_t r = B.row0 + k;
        st3(a.cgB, r, -G[k]);
        st_planes(a.diag, a.n_rows, r, H[k]);
        if (a.diag_mat) st_planes(a.diag_mat, a.n_rows, r, H[k]);
    }
    for (int k = 0; k < 12; k++) st_planes(a.sell_val, a.nblocks, B.blk[k], H[4 + k]);
}

// fn_apply_dx_affine_bodies (newton_solver.cpp:505-526): x = A X + p for every rigid vertex.
__global__ __launch_bounds__(kB) void k_rigid_positions(uint32_t n, const uint8_t* __restrict__ kind,
                                                         const uint32_t* __restrict__ vert_body,
                                                         const BodyDev* __restrict__ bodies, const float* __restrict__ body_X,
                                                         float* __restrict__ x)
{
    uint32_t i = blockIdx.x * kB + threadIdx.x;
    if (i >= n || kind[i] != 1u) return;
    uint32_t r  = bodies[vert_body[i]].row0;
    f3       p  = ld3(x, r), a0 = ld3(x, r + 1), a1 = ld3(x, r + 2), a2 = ld3(x, r + 3);
    f3       X  = ld3(body_X, i);
    st3(x, i, ((X.x * a0 + X.y * a1) + X.z * a2) + p);
}

// ---------------------------------------------------------------- narrow phase
// Contact record (the reference's CollisionPairTemplate, collision_data.h:48-127):
// idx (type bit 31 in idx.z for VF, idx.w for EE), (n, k2), weights, (k1, area*kappa, bary0, bary1).
// Appends the block's emitted contacts with one atomic on the shared counter (one per wavefront was
// what the DCD waited for in contact: 474 us for 0.7M contacts, now 173). Called by all threads of
// the block; `turn` alternates from call to call, so one call's LDS words outlive the next one's start.
LCSX_D void push_contact(const ContactBuf& cb, bool emit, uint4 idx, f3 n, float k1, float k2, float ak, float b0,
                         float b1, float4 w, uint32_t turn)
{
    __shared__ uint32_t cnt[2][4], base[2];
    const uint32_t      wv   = threadIdx.x >> 6, o = turn & 1u;
    const uint64_t      mask = __ballot(emit);
    if (lane_id() == 0) cnt[o][wv] = (uint32_t)__popcll(mask);
    __syncthreads();
    if (threadIdx.x == 0)
    {
        const uint32_t tot = cnt[o][0] + cnt[o][1] + cnt[o][2] + cnt[o][3];
        base[o]            = tot ? count_reserve(cb.count, tot) : 0u;
    }
    __syncthreads();
    uint32_t slot = base[o] + (uint32_t)__popcll(mask & lanemask_lt());
    for (uint32_t k = 0; k < wv; k++) slot += cnt[o][k];
    if (emit && slot < cb.capacity)
    {
        cb.idx[slot] = idx;
        cb.nk[slot]  = make_float4(n.x, n.y, n.z, k2);
        cb.w[slot]   = w;
        cb.aux[slot] = make_float4(k1, ak, b0, b1);
    }
}

// fn_narrow_phase_vf_dcd_query, narrow_phase.cpp:771-933 (barrier energy). FP64 (the mixed
// forms: distance, normal and barrier in double) is a template parameter, as in k_ccd, so the
// FP32 instance is allocated the registers of its own path.
template <bool FP64>
__global__ __launch_bounds__(kB) void k_dcd_vf(DcdArgs a)
{
    uint32_t n = min(*a.pair_count, a.pair_capacity);
    uint32_t turn = 0u;
    for (uint32_t first = blockIdx.x * kB; first < n; first += gridDim.x * kB, turn++)
    {
        const bool     in = first + threadIdx.x < n;
        const uint32_t p  = in ? first + threadIdx.x : n - 1u;
        uint32_t vid = a.pairs[2 * (size_t)p], fid = a.pairs[2 * (size_t)p + 1];
        uint32_t f0 = a.faces[3 * fid], f1 = a.faces[3 * fid + 1], f2 = a.faces[3 * fid + 2];
        // shared vertex, or both sides on one rigid body (narrow_phase.cpp:806-807)
        bool     skip = !in || (vid == f0 || vid == f1 || vid == f2) ||
                    (a.vert_body && a.vert_body[vid] != kInvalid && a.vert_body[vid] == a.vert_body[f0]);
        bool     emit = false;
        uint4    idx  = make_uint4(vid, f0, f1 | 0x80000000u, f2);
        f3       nrm  = mk(0.0f, 0.0f, 0.0f);
        float    k1 = 0.0f, k2 = 0.0f, ak = 0.0f;
        f3       b  = mk(0.0f, 0.0f, 0.0f);
        if (!skip && FP64)
        {
            // mixed-precision mode: barycentrics, distance and barrier in double
            using namespace fp64;
            d3     P = wide(ld3(a.x, vid)), t0 = wide(ld3(a.x, f0)), t1 = wide(ld3(a.x, f1)), t2 = wide(ld3(a.x, f2));
            d3     bd = pt_coeff_unclassified(P, t0, t1, t2);
            d3     X  = (bd.x * (P - t0) + bd.y * (P - t1)) + bd.z * (P - t2);
            double d2 = fp64::dot(X, X);
            double dh = ((double)a.dhat[vid] + (double)a.dhat[f0]) * 0.5;
            double th = (double)a.offset[vid] + (double)a.offset[f0];
            b         = mk((float)bd.x, (float)bd.y, (float)bd.z);
            if (d2 < (th + dh) * (th + dh))
            {
                double d  = sqrt(d2);
                d3     nd = X / d;
                nrm       = mk((float)nd.x, (float)nd.y, (float)nd.z);
                double aa = 0.5 * ((double)a.area_a[vid] + (double)a.area_b[fid]), dk1, dk2;
                fp64::pair_k(a.quadratic, d, th, dh, aa, (double)a.kappa, dk1, dk2);
                k1        = (float)dk1;
                k2        = (float)dk2;
                ak        = (float)(aa * (double)a.kappa);
                emit      = true;
            }
        }
        else if (!skip)
        {
            f3 P = ld3(a.x, vid), t0 = ld3(a.x, f0), t1 = ld3(a.x, f1), t2 = ld3(a.x, f2);
            b         = pt_coeff_unclassified(P, t0, t1, t2);
            f3    X   = (b.x * (P - t0) + b.y * (P - t1)) + b.z * (P - t2);
            float d2  = dot(X, X);
            float dh  = (a.dhat[vid] + a.dhat[f0]) * 0.5f;
            float th  = a.offset[vid] + a.offset[f0];
            if (d2 < (th + dh) * (th + dh))
            {
                float d  = sqrtf(d2);
                nrm      = X / d;
                float aa = 0.5f * (a.area_a[vid] + a.area_b[fid]);
                pair_k(a.quadratic, d, th, dh, aa, a.kappa, k1, k2);
                ak       = aa * a.kappa;
                emit     = true;
            }
        }
        push_contact(a.out, emit, idx, nrm, k1, k2, ak, b.x, b.y, make_float4(1.0f, -b.x, -b.y, (b.x + b.y) - 1.0f),
                     turn);
    }
}

// fn_narrow_phase_ee_dcd_query, narrow_phase.cpp:935-1098
template <bool FP64>
__global__ __launch_bounds__(kB) void k_dcd_ee(DcdArgs a)
{
    uint32_t n = min(*a.pair_count, a.pair_capacity);
    uint32_t turn = 0u;
    for (uint32_t first = blockIdx.x * kB; first < n; first += gridDim.x * kB, turn++)
    {
        const bool     in = first + threadIdx.x < n;
        const uint32_t p  = in ? first + threadIdx.x : n - 1u;
        uint32_t l = a.pairs[2 * (size_t)p], r = a.pairs[2 * (size_t)p + 1];
        uint32_t a0 = a.edges[2 * l], a1 = a.edges[2 * l + 1], b0 = a.edges[2 * r], b1 = a.edges[2 * r + 1];
        // shared vertex, or both edges on one rigid body (narrow_phase.cpp:972-974)
        bool     skip = !in || (a0 == b0 || a0 == b1 || a1 == b0 || a1 == b1) ||
                    (a.vert_body && a.vert_body[a0] != kInvalid && a.vert_body[a0] == a.vert_body[b0]);
        bool     emit = false;
        uint4    idx  = make_uint4(a0, a1, b0, b1 | 0x80000000u);
        f3       nrm  = mk(0.0f, 0.0f, 0.0f);
        float    k1 = 0.0f, k2 = 0.0f, ak = 0.0f;
        c4       c  = {{0.0f, 0.0f, 0.0f, 0.0f}};
        if (!skip && FP64)
        {
            using namespace fp64;
            d3     pa0 = wide(ld3(a.x, a0)), pa1 = wide(ld3(a.x, a1)), pb0 = wide(ld3(a.x, b0)), pb1 = wide(ld3(a.x, b1));
            dc4    cd  = ee_coeff_unclassified(pa0, pa1, pb0, pb1);
            d3     X   = (cd.v[0] * pa0 + cd.v[1] * pa1) - (cd.v[2] * pb0 + cd.v[3] * pb1);
            double d2  = fp64::dot(X, X);
            double dh  = ((double)a.dhat[a0] + (double)a.dhat[b0]) * 0.5;
            double th  = (double)a.offset[a0] + (double)a.offset[b0];
            for (int k = 0; k < 4; k++) c.v[k] = (float)cd.v[k];
            if (d2 < (th + dh) * (th + dh))
            {
                double d  = sqrt(d2);
                d3     nd = X / d;
                nrm       = mk((float)nd.x, (float)nd.y, (float)nd.z);
                double aa = 0.5 * ((double)a.area_a[l] + (double)a.area_b[r]), dk1, dk2;
                fp64::pair_k(a.quadratic, d, th, dh, aa, (double)a.kappa, dk1, dk2);
                k1        = (float)dk1;
                k2        = (float)dk2;
                ak        = (float)(aa * (double)a.kappa);
                emit      = true;
            }
        }
        else if (!skip)
        {
            f3 pa0 = ld3(a.x, a0), pa1 = ld3(a.x, a1), pb0 = ld3(a.x, b0), pb1 = ld3(a.x, b1);
            c          = ee_coeff_unclassified(pa0, pa1, pb0, pb1);
            f3    X    = (c.v[0] * pa0 + c.v[1] * pa1) - (c.v[2] * pb0 + c.v[3] * pb1);
            float d2   = dot(X, X);
            float dh   = (a.dhat[a0] + a.dhat[b0]) * 0.5f;
            float th   = a.offset[a0] + a.offset[b0];
            if (d2 < (th + dh) * (th + dh))
            {
                float d  = sqrtf(d2);
                nrm      = X / d;
                float aa = 0.5f * (a.area_a[l] + a.area_b[r]);
                pair_k(a.quadratic, d, th, dh, aa, a.kappa, k1, k2);
                ak       = aa * a.kappa;
                emit     = true;
            }
        }
        push_contact(a.out, emit, idx, nrm, k1, k2, ak, c.v[0], c.v[2],
                     make_float4(c.v[0], 1.0f - c.v[0], -c.v[2], c.v[2] - 1.0f), turn);
    }
}

// Post-step gap of one candidate pair or vertex (device_post_dist_check, newton_solver.cpp:
// 3364-3375): the DCD's FP64 distance (unclassified barycentrics) minus the pair's offsets, or the
// vertex's height above the floor minus its offset. Every wavefront takes one contiguous stretch of
// the list and keeps its lanes' smallest gap and counts in registers, with one set of atomics per
// stretch and scene (pairs of one scene are mostly contiguous): a set per 64 pairs, all on the same
// three words, made the launch wait for the atomics (672 us for the cloth tube's 0.9M edge pairs, now
// 115 us).
__global__ __launch_bounds__(kB) void k_gap_check(GapArgs a)
{
    using namespace fp64;
    const uint32_t n = a.kind == 2 ? a.nv : min(*a.pair_count, a.pair_capacity);
    const uint32_t waves = gridDim.x * (kB / 64u), w = blockIdx.x * (kB / 64u) + (threadIdx.x >> 6);
    const uint32_t per   = ((n + waves - 1u) / waves + 63u) & ~63u;  // a wavefront's stretch
    uint32_t       cur = kInvalid, np = 0u, nc = 0u;  // the scene of the lanes' sums (uniform)
    unsigned long long best = ~0ull;
    auto flush = [&]() {
        if (cur == kInvalid) return;
        for (int o = 32; o > 0; o >>= 1)
        {
            const unsigned long long t = __shfl_xor(best, o);
            best                       = t < best ? t : best;
            np += __shfl_xor(np, o);
            nc += __shfl_xor(nc, o);
        }
        if (lane_id() == 0)
        {
            atomicMin(&a.out[cur].min_key, best);
            if (np) atomicAdd(&a.out[cur].n_pen, np);
            atomicAdd(&a.out[cur].n_checked, nc);
        }
        np = nc = 0u;
        best    = ~0ull;
    };
    const uint64_t begin = (uint64_t)w * per, end = begin + per < n ? begin + per : n;
    for (uint64_t base = begin; base < end; base += 64u)
    {
        const uint32_t p     = (uint32_t)base + lane_id();
        bool           valid = p < n;
        double         gap   = 0.0;
        uint32_t       v0    = 0;
        if (valid && a.kind == 0)
        {
            uint32_t vid = a.pairs[2 * (size_t)p], fid = a.pairs[2 * (size_t)p + 1];
            uint32_t f0 = a.faces[3 * fid], f1 = a.faces[3 * fid + 1], f2 = a.faces[3 * fid + 2];
            valid = !(vid == f0 || vid == f1 || vid == f2) &&
                    !(a.vert_body[vid] != kInvalid && a.vert_body[vid] == a.vert_body[f0]);
            if (valid)
            {
                d3 P = wide(ld3(a.x, vid)), t0 = wide(ld3(a.x, f0)), t1 = wide(ld3(a.x, f1)), t2 = wide(ld3(a.x, f2));
                d3 bd = pt_coeff_unclassified(P, t0, t1, t2);
                d3 X  = (bd.x * (P - t0) + bd.y * (P - t1)) + bd.z * (P - t2);
                gap   = sqrt(fp64::dot(X, X)) - ((double)a.offset[vid] + (double)a.offset[f0]);
                v0    = vid;
            }
        }
        else if (valid && a.kind == 1)
        {
            uint32_t l = a.pairs[2 * (size_t)p], r = a.pairs[2 * (size_t)p + 1];
            uint32_t a0 = a.edges[2 * l], a1 = a.edges[2 * l + 1], b0 = a.edges[2 * r], b1 = a.edges[2 * r + 1];
            valid = !(a0 == b0 || a0 == b1 || a1 == b0 || a1 == b1) &&
                    !(a.vert_body[a0] != kInvalid && a.vert_body[a0] == a.vert_body[b0]);
            if (valid)
            {
                d3  pa0 = wide(ld3(a.x, a0)), pa1 = wide(ld3(a.x, a1)), pb0 = wide(ld3(a.x, b0)), pb1 = wide(ld3(a.x, b1));
                dc4 cd  = ee_coeff_unclassified(pa0, pa1, pb0, pb1);
                d3  X   = (cd.v[0] * pa0 + cd.v[1] * pa1) - (cd.v[2] * pb0 + cd.v[3] * pb1);
                gap     = sqrt(fp64::dot(X, X)) - ((double)a.offset[a0] + (double)a.offset[b0]);
                v0      = a0;
            }
        }
        else if (valid)
        {
            // ground: free vertex rows (soft or rigid), as the ground barrier (newton_solver.cpp:883-950)
            valid = a.row_kind[p] < 2u && !a.fixed[p];
            if (valid)
            {
                gap = ((double)a.x[3 * (size_t)p + 1] - (double)a.floor_y) - (double)a.offset[p];
                v0  = p;
            }
        }
        const uint32_t           sc  = valid ? a.vert_scene[v0] : kInvalid;
        const unsigned long long key = valid ? d2ord(gap) : ~0ull;
        for (uint64_t todo = __ballot(valid); todo != 0ull;)
        {
            const uint32_t s0   = __shfl(sc, __ffsll((unsigned long long)todo) - 1);
            const bool     mine = valid && sc == s0;
            if (s0 != cur)
            {
                flush();
                cur = s0;
            }
            if (mine)
            {
                best = key < best ? key : best;
                np += gap <= 0.0 ? 1u : 0u;
                nc++;
            }
            todo &= ~__ballot(mine);
        }
    }
    flush();
}

__global__ void k_reset_gap(GapStatus* g, uint32_t nscenes)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nscenes) g[i] = GapStatus{~0ull, 0u, 0u};
}

__global__ void k_fill_u32(uint32_t* a, uint32_t n, uint32_t v)
{
    uint32_t i = blockIdx.x * kB + threadIdx.x;
    if (i < n) a[i] = v;
}

// ---------------------------------------------------------------- contact adjacency
// Generalized DOFs of a contact (narrow_phase.cpp:2600-2670): each side is either soft (its
// vertices with their weights) or one rigid body (its four rows with the weights sum_side w (1, X)).
__global__ __launch_bounds__(kB) void k_contact_lift(ContactView c, const uint32_t* __restrict__ vert_body,
                                                      const BodyDev* __restrict__ bodies, const float* __restrict__ body_X,
                                                      uint4* __restrict__ gr, float4* __restrict__ gw)
{
    uint32_t n = min(*c.count, c.capacity);
    for (uint32_t k = blockIdx.x * kB + threadIdx.x; k < n; k += gridDim.x * kB)
    {
        uint4    id     = c.idx[k];
        float4   w4     = c.w[k];
        bool     vf     = (id.z & 0x80000000u) != 0u;
        uint32_t ids[4] = {id.x & 0x7fffffffu, id.y & 0x7fffffffu, id.z & 0x7fffffffu, id.w & 0x7fffffffu};
        float    w[4]   = {w4.x, w4.y, w4.z, w4.w};
        uint32_t r[8];
        float    g[8];
        int      ng = 0;
        for (int side = 0; side < 2; side++)
        {
            int      k0 = vf ? (side == 0 ? 0 : 1) : 2 * side, k1 = vf ? (side == 0 ? 1 : 4) : 2 * side + 2;
            uint32_t b  = vert_body ? vert_body[ids[k0]] : kInvalid;
            if (b == kInvalid)
            {
                for (int j = k0; j < k1; j++)
                {
                    r[ng] = ids[j];
                    g[ng] = w[j];
                    ng++;
                }
                continue;
            }
            float aw[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            for (int j = k0; j < k1; j++)
            {
                f3 X  = ld3(body_X, ids[j]);
                aw[0] = aw[0] + w[j] * 1.0f;
                aw[1] = aw[1] + w[j] * X.x;
                aw[2] = aw[2] + w[j] * X.y;
                aw[3] = aw[3] + w[j] * X.z;
            }
            uint32_t r0 = bodies[b].row0;
            for (int j = 0; j < 4; j++)
            {
                r[ng] = r0 + j;
                g[ng] = aw[j];
                ng++;
            }
        }
        for (int j = ng; j < 8; j++)
        {
            r[j] = kInvalid;
            g[j] = 0.0f;
        }
        gr[2 * (size_t)k]     = make_uint4(r[0], r[1], r[2], r[3]);
        gr[2 * (size_t)k + 1] = make_uint4(r[4], r[5], r[6], r[7]);
        gw[2 * (size_t)k]     = make_float4(g[0], g[1], g[2], g[3]);
        gw[2 * (size_t)k + 1] = make_float4(g[4], g[5], g[6], g[7]);
    }
}

// Entries [4 half, 4 half + 4) of contact k's generalized DOFs. Without bodies (gr null) they are the
// contact's own four vertices and weights.
LCSX_D void gdofs4(const ContactView& c, uint32_t k, uint32_t half, uint32_t r[4], float w[4])
{
    uint4  a = make_uint4(kInvalid, kInvalid, kInvalid, kInvalid);
    float4 u = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (c.gr)
    {
        a = c.gr[2 * (size_t)k + half];
        u = c.gw[2 * (size_t)k + half];
    }
    else if (half == 0u)
    {
        a = c.idx[k];
        u = c.w[k];
        a = make_uint4(a.x & 0x7fffffffu, a.y & 0x7fffffffu, a.z & 0x7fffffffu, a.w & 0x7fffffffu);
    }
    r[0] = a.x; r[1] = a.y; r[2] = a.z; r[3] = a.w;
    w[0] = u.x; w[1] = u.y; w[2] = u.z; w[3] = u.w;
}
LCSX_D void gdofs(const ContactView& c, uint32_t k, uint32_t r[8], float w[8])
{
    gdofs4(c, k, 0u, r, w);
    gdofs4(c, k, 1u, r + 4, w + 4);
}
LCSX_D float gweight(const ContactView& c, uint32_t k, uint32_t j)
{
    const float4   u = c.gr ? c.gw[2 * (size_t)k + (j >> 2)] : c.w[k];
    const uint32_t l = j & 3u;
    return l == 0 ? u.x : (l == 1 ? u.y : (l == 2 ? u.z : u.w));
}

// ---------------------------------------------------------------- contact triplets (on demand)
// The contact Hessian's off-diagonal blocks as the reference's sorted contact triplets
// (NarrowPhasesDetector::device_sort_contact_triplet / device_assemble_contact_triplet,
// narrow_phase.cpp:1434-1758, 1883-2323): for every ordered pair (a, b), a != b, of a contact's
// generalized DOFs, the Gauss-Newton block (k2 w_a) w_b n n^T; sorted by (row, column) and summed
// per (row, column). The PCG does not use them (its contact product is matrix-free); they are for
// callers that take the assembled contact matrix.
__global__ __launch_bounds__(kB) void k_ct_count(ContactView c, uint32_t* __restrict__ cnt)
{
    const uint32_t n = min(*c.count, c.capacity);
    for (uint32_t k = blockIdx.x * kB + threadIdx.x; k < n; k += gridDim.x * kB)
    {
        uint32_t r[8];
        float    w[8];
        gdofs(c, k, r, w);
        uint32_t ng = 0;
        for (int j = 0; j < 8; j++) ng += r[j] != kInvalid ? 1u : 0u;
        cnt[k] = ng * (ng - (ng ? 1u : 0u));
    }
}
__global__ __launch_bounds__(kB) void k_ct_fill(ContactView c, const uint32_t* __restrict__ ptr, uint32_t* __restrict__ row,
                                                uint32_t* __restrict__ col, uint32_t* __restrict__ idx,
                                                float* __restrict__ blk)
{
    const uint32_t n = min(*c.count, c.capacity);
    for (uint32_t k = blockIdx.x * kB + threadIdx.x; k < n; k += gridDim.x * kB)
    {
        uint32_t r[8];
        float    w[8];
        gdofs(c, k, r, w);
        const float4 nk = c.nk[k];
        const float  nv[3] = {nk.x, nk.y, nk.z};
        uint32_t     t     = ptr[k];
        for (int a = 0; a < 8; a++)
        {
            if (r[a] == kInvalid) continue;
            const float ka = nk.w * w[a];
            for (int b = 0; b < 8; b++)
            {
                if (b == a || r[b] == kInvalid) continue;
                const float s = ka * w[b];
                row[t] = r[a];
                col[t] = r[b];
                idx[t] = t;
#pragma unroll
                for (int i = 0; i < 3; i++)
#pragma unroll
                    for (int j = 0; j < 3; j++) blk[9 * (size_t)t + 3 * i + j] = s * (nv[i] * nv[j]);
                t++;
            }
        }
    }
}
// head[t] = 1 where the sorted (row, column) differs from the previous entry's
__global__ __launch_bounds__(kB) void k_ct_heads(uint32_t n, const uint32_t* __restrict__ row, const uint32_t* __restrict__ col,
                                                 uint32_t* __restrict__ head)
{
    const uint32_t t = blockIdx.x * kB + threadIdx.x;
    if (t < n) head[t] = (t == 0 || row[t] != row[t - 1] || col[t] != col[t - 1]) ? 1u : 0u;
}
// one thread per distinct (row, column): the sum of its blocks in sorted order (the stable sort keeps
// the contacts' order within a key)
__global__ __launch_bounds__(kB) void k_ct_reduce(uint32_t n, const uint32_t* __restrict__ head,
                                                  const uint32_t* __restrict__ pos, const uint32_t* __restrict__ row,
                                                  const uint32_t* __restrict__ col, const uint32_t* __restrict__ idx,
                                                  const float* __restrict__ blk, uint32_t* __restrict__ out_rc,
                                                  float* __restrict__ out_blk)
{
    const uint32_t t = blockIdx.x * kB + threadIdx.x;
    if (t >= n || head[t] == 0u) return;
    float acc[9];
#pragma unroll
    for (int i = 0; i < 9; i++) acc[i] = 0.0f;
    for (uint32_t u = t; u < n && (u == t || head[u] == 0u); u++)
    {
        const size_t b = 9 * (size_t)idx[u];
#pragma unroll
        for (int i = 0; i < 9; i++) acc[i] = acc[i] + blk[b + i];
    }
    const uint32_t o = pos[t];
    out_rc[2 * (size_t)o]     = row[t];
    out_rc[2 * (size_t)o + 1] = col[t];
#pragma unroll
    for (int i = 0; i < 9; i++) out_blk[9 * (size_t)o + i] = acc[i];
}

// Per-row lists of (contact << 3 | entry), built once per Newton iteration after the DCD, so that
// contact terms are gathered by the rows that own them instead of scattered with atomics.
__global__ __launch_bounds__(kB) void k_vc_count(ContactView c, uint32_t* __restrict__ cnt)
{
    uint32_t n = min(*c.count, c.capacity);
    for (uint32_t k = blockIdx.x * kB + threadIdx.x; k < n; k += gridDim.x * kB)
    {
        uint32_t r[8];
        float    w[8];
        gdofs(c, k, r, w);
        for (int j = 0; j < 8; j++)
            if (r[j] != kInvalid) atomicAdd(&cnt[r[j]], 1u);
    }
}

// Exclusive scan of n 32-bit counts into out[0..n] (out[n] = total; out may equal in) in three
// launches: tile sums, a scan of the tile sums in one workgroup, then each tile rescanned from its
// offset. Tiles of kScanTile values, 1024 threads x 4 consecutive values.
constexpr uint32_t kScanTile = 4096;

// Exclusive scan over the block of one value per thread (1024 threads); returns the block total.
LCSX_D uint32_t block_scan_1024(uint32_t v, uint32_t& excl)
{
    __shared__ uint32_t wsum[16];
    const uint32_t      lane = lane_id(), w = threadIdx.x >> 6;
    uint32_t            x    = v;
    for (int off = 1; off < 64; off <<= 1)
    {
        uint32_t y = __shfl_up(x, off);
        if ((int)lane >= off) x += y;
    }
    if (lane == 63u) wsum[w] = x;
    __syncthreads();
    uint32_t before = 0, total = 0;
    for (uint32_t k = 0; k < 16u; k++)
    {
        if (k < w) before += wsum[k];
        total += wsum[k];
    }
    __syncthreads();
    excl = before + x - v;
    return total;
}

__global__ __launch_bounds__(1024) void k_scan_tiles(const uint32_t* __restrict__ in, uint32_t n, uint32_t* __restrict__ part)
{
    const uint32_t base = blockIdx.x * kScanTile + 4u * threadIdx.x;
    uint32_t       v    = 0;
    for (uint32_t k = 0; k < 4u; k++)
        if (base + k < n) v += in[base + k];
    uint32_t excl;
    uint32_t tot = block_scan_1024(v, excl);
    if (threadIdx.x == 0) part[blockIdx.x] = tot;
}

// part[0..m) -> exclusive offsets, part[m] = total (one workgroup, m <= 1024 * chunk)
__global__ __launch_bounds__(1024) void k_scan_parts(uint32_t* __restrict__ part, uint32_t m)
{
    const uint32_t per = (m + 1023u) / 1024u;
    const uint32_t b = min(m, threadIdx.x * per), e = min(m, b + per);
    uint32_t       v = 0;
    for (uint32_t i = b; i < e; i++) v += part[i];
    uint32_t excl;
    uint32_t tot = block_scan_1024(v, excl);
    for (uint32_t i = b; i < e; i++)
    {
        uint32_t x = part[i];
        part[i]    = excl;
        excl += x;
    }
    if (threadIdx.x == 0) part[m] = tot;
}

__global__ __launch_bounds__(1024) void k_scan_apply(const uint32_t* in, uint32_t n, const uint32_t* __restrict__ part,
                                                      uint32_t* out)
{
    const uint32_t base = blockIdx.x * kScanTile + 4u * threadIdx.x;
    uint32_t       x[4], v = 0;
    for (uint32_t k = 0; k < 4u; k++)
    {
        x[k] = base + k < n ? in[base + k] : 0u;
        v += x[k];
    }
    uint32_t excl;
    block_scan_1024(v, excl);  // every read of this tile happens before the barrier inside
    uint32_t run = part[blockIdx.x] + excl;
    for (uint32_t k = 0; k < 4u; k++)
        if (base + k < n)
        {
            out[base + k] = run;
            run += x[k];
        }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) out[n] = part[gridDim.x];
}

// The three steps for up to kScanPasses tiles in one workgroup: pass i covers values 4096 i .. of which
// thread t holds four; every value is loaded before the first wait.
constexpr uint32_t kScanPasses = 9;
template <int kP>
__global__ __launch_bounds__(1024) void k_scan_one(const uint32_t* in, uint32_t n, uint32_t* out)
{
    __shared__ uint32_t tot[kP * 16 + 1];
    const uint32_t      t = threadIdx.x, w = t >> 6, lane = t & 63u;
    uint32_t            x[kP][4], inc[kP];
#pragma unroll
    for (int i = 0; i < kP; i++)
#pragma unroll
        for (uint32_t k = 0; k < 4u; k++)
        {
            const uint32_t at = (uint32_t)i * kScanTile + 4u * t + k;
            x[i][k]           = at < n ? in[at] : 0u;
        }
#pragma unroll
    for (int i = 0; i < kP; i++)
    {
        inc[i] = ((x[i][0] + x[i][1]) + x[i][2]) + x[i][3];
        for (int o = 1; o < 64; o <<= 1)
        {
            const uint32_t u = __shfl_up(inc[i], o);
            if ((int)lane >= o) inc[i] += u;
        }
        if (lane == 63u) tot[16 * i + w] = inc[i];
    }
    __syncthreads();
    if (t < 64u)
    {
        // exclusive scan of the wavefronts' totals, kP / 4 consecutive ones per lane
        constexpr int kPer = (kP * 16 + 63) / 64;
        uint32_t      v[kPer], s = 0u;
        for (int k = 0; k < kPer; k++)
        {
            const uint32_t at = kPer * t + (uint32_t)k;
            v[k]              = at < kP * 16u ? tot[at] : 0u;
            s += v[k];
        }
        uint32_t run = s;
        for (int o = 1; o < 64; o <<= 1)
        {
            const uint32_t u = __shfl_up(run, o);
            if ((int)lane >= o) run += u;
        }
        if (t == 63u) tot[kP * 16] = run;
        run -= s;
        for (int k = 0; k < kPer; k++)
        {
            const uint32_t at = kPer * t + (uint32_t)k;
            if (at < kP * 16u) tot[at] = run;
            run += v[k];
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kP; i++)
    {
        uint32_t run = tot[16 * i + w] + inc[i] - (((x[i][0] + x[i][1]) + x[i][2]) + x[i][3]);
#pragma unroll
        for (uint32_t k = 0; k < 4u; k++)
        {
            const uint32_t at = (uint32_t)i * kScanTile + 4u * t + k;
            if (at < n) out[at] = run;
            run += x[i][k];
        }
    }
    if (t == 0) out[n] = tot[kP * 16];
}

__global__ __launch_bounds__(kB) void k_vc_fill(ContactView c, const uint32_t* __restrict__ ptr, uint32_t* __restrict__ cursor,
                                                 uint32_t* __restrict__ list, uint32_t* __restrict__ row)
{
    uint32_t n = min(*c.count, c.capacity);
    for (uint32_t k = blockIdx.x * kB + threadIdx.x; k < n; k += gridDim.x * kB)
    {
        uint32_t r[8];
        float    w[8];
        gdofs(c, k, r, w);
        for (uint32_t j = 0; j < 8; j++)
        {
            uint32_t v = r[j];
            if (v == kInvalid) continue;
            uint32_t pos = ptr[v] + atomicAdd(&cursor[v], 1u);
            list[pos]    = (k << 3) | j;
            row[pos]     = v;
        }
    }
}

// Each row's slots in a fixed order: by the contact's vertex ids (with the type bit). The narrow phase
// appends contacts with atomics, so contact ids differ from run to run;
// ordering the slots by content makes every per-row sum (contact gradient and Hessian, the SpMV's
// contact runs) add its terms in the same order in every run, so a state and its contact set give
// the same rounding. A slot's place is its rank among its row's slots. One
// thread per slot walks a short row by itself; the slots of a longer one (a collider vertex has
// hundreds) are compared by their wavefront together, 64 of the row's keys at a time from registers
// (2.8M slots: 678 us when every thread walked its row, now 316).
// kTies: meshes that list an edge or a face twice, or an element that names a vertex twice
// (Setup::repeats), give slots of one row with equal ids. Those are ordered by their entry, their
// contact's k2 (the listings differ in area) and the contact's id, so every slot still has a place of its own.
LCSX_D bool tie_less(const ContactView& c, uint32_t y, uint32_t x)
{
    if ((y & 7u) != (x & 7u)) return (y & 7u) < (x & 7u);
    const uint32_t ky = __float_as_uint(c.nk[y >> 3].w), kx = __float_as_uint(c.nk[x >> 3].w);
    return ky != kx ? ky < kx : y < x;
}
template <bool kTies>
__global__ __launch_bounds__(kB) void k_vc_rank(ContactView c, const uint32_t* __restrict__ ptr,
                                                 const uint32_t* __restrict__ row, const uint32_t* __restrict__ total,
                                                 const uint32_t* __restrict__ list, uint32_t* __restrict__ out)
{
    constexpr uint32_t kShort = 32u;
    const uint32_t     n = *total, lane = lane_id();
    for (uint32_t e0 = blockIdx.x * kB + (threadIdx.x & ~63u); e0 < n; e0 += gridDim.x * kB)
    {
        const bool     on = e0 + lane < n;
        const uint32_t e  = on ? e0 + lane : n - 1u;
        const uint32_t v = row[e], b = ptr[v], m = ptr[v + 1] - b, x = list[e];
        const uint4    kx = c.idx[x >> 3];
        const uint64_t hx = ((uint64_t)kx.x << 32) | kx.y, lx = ((uint64_t)kx.z << 32) | kx.w;
        auto less = [&](uint64_t hy, uint64_t ly) { return (hy < hx) | ((hy == hx) & (ly < lx)); };
        uint32_t rank = 0u;
        if (kTies && on)
            for (uint32_t t = 0; t < m; t++)
            {
                const uint32_t y  = list[b + t];
                const uint4    ky = c.idx[y >> 3];
                const uint64_t hy = ((uint64_t)ky.x << 32) | ky.y, ly = ((uint64_t)ky.z << 32) | ky.w;
                if (less(hy, ly) || (hy == hx && ly == lx && y != x && tie_less(c, y, x))) rank++;
            }
        if (!kTies && on && m <= kShort)
            for (uint32_t t = 0; t < m; t++)
            {
                const uint4 ky = c.idx[list[b + t] >> 3];
                rank += less(((uint64_t)ky.x << 32) | ky.y, ((uint64_t)ky.z << 32) | ky.w) ? 1u : 0u;
            }
        for (uint64_t todo = __ballot(!kTies && on && m > kShort); todo != 0ull;)
        {
            const int      lead = __ffsll((unsigned long long)todo) - 1;
            const uint32_t rb = (uint32_t)__builtin_amdgcn_readlane((int)b, lead);
            const uint32_t rm = (uint32_t)__builtin_amdgcn_readlane((int)m, lead);
            const bool     mine = on && b == rb;  // rows with slots start at different places
            for (uint32_t u0 = 0; u0 < rm; u0 += 64u)
            {
                const uint4 ky = u0 + lane < rm ? c.idx[list[rb + u0 + lane] >> 3] : make_uint4(0u, 0u, 0u, 0u);
                const uint32_t cnt = min(64u, rm - u0);
                for (uint32_t s = 0; s < cnt; s++)
                {
                    auto rl = [&](uint32_t q) { return (uint32_t)__builtin_amdgcn_readlane((int)q, (int)s); };
                    const uint64_t hy = ((uint64_t)rl(ky.x) << 32) | rl(ky.y), ly = ((uint64_t)rl(ky.z) << 32) | rl(ky.w);
                    rank += (mine & less(hy, ly)) ? 1u : 0u;
                }
            }
            todo &= ~__ballot(mine);
        }
        if (on) out[b + rank] = x;
    }
}

// fn_perPair_assemble_gradient_hessian, narrow_phase.cpp:2550-2676 (soft bodies), gathered per
// vertex: cgB_i += k1 w_j n and diag_i += k2 w_j^2 n n^T over the vertex's contact slots.
__global__ __launch_bounds__(kB) void k_contact_assemble(ContactView c, VertContacts vc, float* __restrict__ cgB,
                                                          float* __restrict__ diag, uint32_t nv)
{
    // One wavefront per row: 64 slots' twelve terms (gradient 3, block 9) at a time into LDS, lane by
    // lane one slot, then added in slot order, twelve lanes one entry each. (A thread per row was a chain
    // of as many round trips as the row has slots: 543 us with 2.8M slots, now 91.)
    __shared__ float term[kB / 64][12][64 + 1];
    const uint32_t   lane = lane_id(), w = threadIdx.x >> 6, waves = gridDim.x * (kB / 64u);
    for (uint32_t i = blockIdx.x * (kB / 64u) + w; i < nv; i += waves)
    {
        const uint32_t e0 = vc.ptr[i], e1 = vc.ptr[i + 1];
        if (e0 == e1) continue;
        float sum = 0.0f;
        for (uint32_t e = e0; e < e1; e += 64u)
        {
            const uint32_t cnt = min(64u, e1 - e);
            if (lane < cnt)
            {
                const uint32_t ent = vc.list[e + lane], k = ent >> 3;
                const float4   nk  = c.nk[k];
                const float    ax = c.aux[k].x, wj = gweight(c, k, ent & 7u), gs = ax * wj, s = (nk.w * wj) * wj;
                const float    n3[3] = {nk.x, nk.y, nk.z};
#pragma unroll
                for (int r = 0; r < 3; r++)
                {
                    term[w][r][lane] = gs * n3[r];
#pragma unroll
                    for (int cc = 0; cc < 3; cc++) term[w][3 + 3 * r + cc][lane] = s * (n3[r] * n3[cc]);
                }
            }
            __builtin_amdgcn_wave_barrier();
            if (lane < 12u)
                for (uint32_t q = 0; q < cnt; q++) sum = sum + term[w][lane][q];
            __builtin_amdgcn_wave_barrier();
        }
        if (lane < 3u) cgB[3 * (size_t)i + lane] = cgB[3 * (size_t)i + lane] + sum;
        else if (lane < 12u) diag[(lane - 3u) * (size_t)nv + i] = diag[(lane - 3u) * (size_t)nv + i] + sum;
    }
}

// Per-slot coefficient a = k2 w_j n (the contact's id in .w), in list order. With the contact
// diagonal blocks left out of the SpMV's diagonal, the contact part of (A p)_i
// (narrow_phase.cpp:2730-2775) is sum over the row's slots of a t_c, t_c = sum_jj w_jj n.p_jj.
__global__ __launch_bounds__(kB) void k_vc_coeffs(ContactView c, const uint32_t* __restrict__ ptr, uint32_t nv,
                                                   const uint32_t* __restrict__ ranked, uint32_t* __restrict__ list,
                                                   float4* __restrict__ coef)
{
    uint32_t total = ptr[nv];
    for (uint32_t e = blockIdx.x * kB + threadIdx.x; e < total; e += gridDim.x * kB)
    {
        uint32_t ent = ranked[e], k = ent >> 3, j = ent & 7u;
        list[e]      = ent;
        float4   nk = c.nk[k];
        f3       a  = (nk.w * gweight(c, k, j)) * mk(nk.x, nk.y, nk.z);
        coef[e]       = make_float4(a.x, a.y, a.z, __uint_as_float(k));
    }
}

// Scene-aligned 256-slot chunks of the slot list: scene s's slots [ptr[v0_s], ptr[v0_{s+1}])
// are cut into ceil(slots / 256) chunks (one workgroup).
__global__ __launch_bounds__(1024) void k_chunk_table(SegView g, const uint32_t* __restrict__ ptr,
                                                       uint32_t* __restrict__ sc_cb0, uint32_t* __restrict__ cb_scene,
                                                       uint32_t* __restrict__ cb_slot0)
{
    __shared__ uint32_t part[1024];
    const uint32_t t   = threadIdx.x, S = g.nscenes;
    const uint32_t per = (S + 1023u) / 1024u;
    const uint32_t b   = min(S, t * per), e = min(S, b + per);
    auto nch = [&](uint32_t sc) { return (ptr[g.sc_v0[sc + 1]] - ptr[g.sc_v0[sc]] + 255u) / 256u; };
    uint32_t sum = 0;
    for (uint32_t sc = b; sc < e; sc++) sum += nch(sc);
    part[t] = sum;
    __syncthreads();
    for (uint32_t off = 1; off < 1024u; off <<= 1)
    {
        uint32_t v = t >= off ? part[t - off] : 0u;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    uint32_t run = part[t] - sum;
    for (uint32_t sc = b; sc < e; sc++)
    {
        sc_cb0[sc] = run;
        run += nch(sc);
    }
    const uint32_t total = part[1023];
    if (t == 1023u) sc_cb0[S] = total;
    __threadfence_block();
    __syncthreads();
    // the chunks, all threads over all scenes' (a scene's chunks by one thread: 430 us for one scene
    // with 11,000)
    for (uint32_t c = t; c < total; c += 1024u)
    {
        uint32_t lo = 0u, hi = S - 1u;  // the last scene whose first chunk is not after c
        while (lo < hi)
        {
            const uint32_t m = (lo + hi + 1u) / 2u;
            if (sc_cb0[m] <= c) lo = m;
            else hi = m - 1u;
        }
        cb_scene[c] = lo;
        cb_slot0[c] = ptr[g.sc_v0[lo]] + 256u * (c - sc_cb0[lo]);
    }
}

// t_c = sum_j w_j n.p_j over the contact's generalized DOFs, with p given by pfun.
template <class PF>
LCSX_D float contact_t1(const ContactView& c, uint32_t k, PF pfun)
{
    uint32_t r[8];
    float    w[8];
    gdofs4(c, k, 0u, r, w);
    float4 nk = c.nk[k];
    f3     nn = mk(nk.x, nk.y, nk.z);
    if (!c.gr)
    {
        // four vertices: their rows are requested together
        const f3 p0 = pfun(r[0]), p1 = pfun(r[1]), p2 = pfun(r[2]), p3 = pfun(r[3]);
        return ((w[0] * dot(nn, p0) + w[1] * dot(nn, p1)) + w[2] * dot(nn, p2)) + w[3] * dot(nn, p3);
    }
    gdofs4(c, k, 1u, r + 4, w + 4);
    float t = w[0] * dot(nn, pfun(r[0]));
    for (int j = 1; j < 8; j++)
        if (r[j] != kInvalid) t = t + w[j] * dot(nn, pfun(r[j]));
    return t;
}

// t_c for every contact, with p given by pfun.
template <class PF>
LCSX_D void contact_t(const ContactView& c, float* __restrict__ tc, PF pfun)
{
    uint32_t n = min(*c.count, c.capacity);
    for (uint32_t k = blockIdx.x * kB + threadIdx.x; k < n; k += gridDim.x * kB) tc[k] = contact_t1(c, k, pfun);
}

// One 64-slot chunk per wavefront, starting at `base`: slot contributions a t_c are summed over
// each run of equal rows by a segmented shuffle scan (slots are in row order); the last lane of
// a run returns true with the run's row and sum. Called by all 64 lanes.
template <class TF>
LCSX_D bool slot_chunk(const VertContacts& vc, uint32_t base, uint32_t end, uint32_t& row, f3& sum, TF tcf)
{
    const uint32_t lane = lane_id();
    uint32_t       e    = base + lane;
    bool           ok   = e < end;
    row                 = 0xffffffffu;
    float vx = 0.0f, vy = 0.0f, vz = 0.0f;
    if (ok)
    {
        float4 C = vc.coef[e];
        float  t = tcf(__float_as_uint(C.w));
        row      = vc.row[e];
        vx       = C.x * t;
        vy       = C.y * t;
        vz       = C.z * t;
    }
    for (int off = 1; off < 64; off <<= 1)
    {
        float    ux = __shfl_up(vx, off), uy = __shfl_up(vy, off), uz = __shfl_up(vz, off);
        uint32_t ur = __shfl_up(row, off);
        if ((int)lane >= off && ur == row)
        {
            vx = vx + ux;
            vy = vy + uy;
            vz = vz + uz;
        }
    }
    uint32_t rn = __shfl_down(row, 1);
    sum         = mk(vx, vy, vz);
    return ok && (lane == 63u || rn != row);
}
LCSX_D bool slot_chunk(const VertContacts& vc, uint32_t base, uint32_t end, uint32_t& row, f3& sum)
{
    return slot_chunk(vc, base, end, row, sum, [&](uint32_t c) { return vc.tc[c]; });
}

// Adds row i's contact runs to y in slot order. The wavefronts that summed the runs start at
// s0 + 64 m, so the row's runs end at every wavefront end s0 + 64 m + 63 inside its slots
// [ptr[i], ptr[i + 1]) and at its last slot. No atomics: the sum does not depend on which
// wavefront finished first.
template <class RF>
LCSX_D f3 fold_runs_of(f3 y, RF runsum, const uint32_t* __restrict__ ptr, uint32_t i, uint32_t s0)
{
    const uint32_t b = ptr[i], e = ptr[i + 1];
    if (e <= b) return y;
    for (uint32_t w = s0 + ((b - s0) & ~63u) + 63u;; w += 64u)
    {
        const uint32_t end = min(w, e - 1u);
        y                  = y + runsum(end);
        if (end == e - 1u) break;
    }
    return y;
}
LCSX_D f3 fold_runs(f3 y, const float4* __restrict__ runsum, const uint32_t* __restrict__ ptr, uint32_t i, uint32_t s0)
{
    return fold_runs_of(
        y,
        [&](uint32_t e) {
            const float4 R = runsum[e];
            return mk(R.x, R.y, R.z);
        },
        ptr, i, s0);
}

// Scalars of PCG iteration k (precond_cg.cpp:681-726 and the loop of 118-330): r.z from the
// previous launch's partials, the convergence test (every check_every iterations: r.z below the
// absolute tolerance, or below rel^2 r0.z0, or NaN) and beta = r.z / r.z_old (0 below 1e-10).
struct IterScalars
{
    float rz, beta;
    bool  stop;
};
// The inputs of iter_scalars, read before the converged flag: the scene's r.z partials of the
// previous update and the stored r.z of the previous iteration and of the first one.
struct IterInputs
{
    PrePartials rz;
    float       rz0, rz_old;
};
LCSX_D IterInputs iter_inputs(const PcgArgs& a, uint32_t scene)
{
    IterInputs      in;
    const PcgState* st = a.s + scene;
    in.rz              = prefetch_ranges(a.part_rz, scene_rb0(a.seg, scene), scene_rb0(a.seg, scene + 1), 0u, 0u);
    in.rz0             = a.k == 0 ? 0.0f : st->rz0;
    in.rz_old          = a.k == 0 ? 0.0f : st->rz[(a.k - 1u) & 1u];
    return in;
}
LCSX_D IterScalars iter_scalars(const PcgArgs& a, const IterInputs& in, float* sh)
{
    IterScalars o;
    o.rz         = reduce_prefetched(a.part_rz, in.rz, sh);
    float rz0    = a.k == 0 ? o.rz : in.rz0;
    bool  check  = (a.k % a.check_every) == 0u;
    o.stop       = !(o.rz == o.rz) || (check && (o.rz < a.abs_tol || o.rz <= a.rel2 * rz0));
    float rz_old = in.rz_old;
    o.beta       = rz_old < 1e-10f ? 0.0f : o.rz / rz_old;
    return o;
}

__global__ __launch_bounds__(kB) void k_contact_t_plain(ContactView c, const float* __restrict__ p, float* __restrict__ tc)
{
    contact_t(c, tc, [&](uint32_t v) { return ld3(p, v); });
}

// ---------------------------------------------------------------- PCG
// precond_cg.cpp:118-331, 626-771. State scalars live on the device; kernels early-exit once
// the solve has converged, so the host can enqueue iterations in chunks without reading back.
// One iteration is three launches: the direction (k_pcg_dir: r.z, the convergence test, beta,
// p = z + beta p and the contacts' t_c), the product (k_spmv_pcg: q = A p and p.q) and the update
// (k_pcg_update: alpha, x, r, z and r.z). Kernel boundaries order them; every block re-reduces the
// previous launch's per-block partials in the same fixed order, so all blocks agree on the scalars.
__global__ __launch_bounds__(kB) void k_pcg_init(PcgArgs a)
{
    __shared__ float sh[4];
    const uint32_t   rbi = xcd_block(blockIdx.x, a.seg.n_rb);
    const RowBlk     rb  = row_blk_fast(a.seg, a.n, rbi);
    const uint32_t   i   = rb.row;
    float            loc = 0.0f;
    if (rb.valid)
    {
        m3 D = ld_planes(a.diag, a.n, i);
        // 3x3 inverse by cofactors
        const float* m   = D.m;
        float        c00 = m[4] * m[8] - m[5] * m[7];
        float        c01 = m[5] * m[6] - m[3] * m[8];
        float        c02 = m[3] * m[7] - m[4] * m[6];
        float        det = m[0] * c00 + m[1] * c01 + m[2] * c02;
        float        inv = 1.0f / det;
        m3           Mi;
        Mi.m[0] = c00 * inv;
        Mi.m[1] = (m[2] * m[7] - m[1] * m[8]) * inv;
        Mi.m[2] = (m[1] * m[5] - m[2] * m[4]) * inv;
        Mi.m[3] = c01 * inv;
        Mi.m[4] = (m[0] * m[8] - m[2] * m[6]) * inv;
        Mi.m[5] = (m[2] * m[3] - m[0] * m[5]) * inv;
        Mi.m[6] = c02 * inv;
        Mi.m[7] = (m[1] * m[6] - m[0] * m[7]) * inv;
        Mi.m[8] = (m[0] * m[4] - m[1] * m[3]) * inv;
        st_planes(a.minv, a.n, i, Mi);
        f3 r = ld3(a.b, i);
        st3(a.r, i, r);
        f3 z = mul(Mi, r);
        st3(a.z, i, z);
        st3(a.x, i, mk(0.0f, 0.0f, 0.0f));
        st4(a.p_old, i, mk(0.0f, 0.0f, 0.0f));
        loc = dot(r, z);
    }
    float bs = block_sum(loc, sh);
    if (threadIdx.x == 0)
    {
        a.part_rz[rbi] = bs;
        if (rbi == scene_rb0(a.seg, rb.scene))
        {
            // a scene whose Newton loop has stopped starts converged: its blocks do no work
            PcgState* st = a.s + rb.scene;
            bool      on = a.seg.active == nullptr || a.seg.active[rb.scene] != 0;
            st->converged = on ? 0u : 1u;
            st->iters     = 0u;
            st->nan       = 0u;
            st->fail      = 0u;
            st->rz[0] = st->rz[1] = st->rz0 = 0.0f;
        }
    }
}

// Direction of iteration k (precond_cg.cpp:118-160, 681-726): r.z from the update's partials, the
// convergence test (every check_every iterations), beta = r.z / r.z_old, p_new = z + beta p_old per
// row (FP32 triples in 16-byte rows, so the product gathers one aligned 16-byte load per column),
// and t_c = sum_j w_j n.(z_j + beta p_old_j) per contact (p_new of other rows is not complete
// within this launch). Blocks [0, n_rb) are the rows; the rest the contacts: CT 1 one thread per
// contact (one scene), CT 2 one block per scene-aligned 256-slot chunk, for the contacts whose first
// slot lies in it (batches, each with its scene's beta).
template <int CT>
__global__ __launch_bounds__(kB) void k_pcg_dir(PcgArgs a, ContactView c, VertContacts vc)
{
    __shared__ float sh[4];
    const uint32_t   n_rb = a.seg.n_rb;
    // the contact blocks (a multiple of 8) come first: their dependent gathers start with the
    // launch instead of after the row blocks
    const uint32_t   nc   = gridDim.x - n_rb;
    const bool       rows = blockIdx.x >= nc;
    const uint32_t   rbi  = rows ? xcd_block(blockIdx.x - nc, n_rb) : 0u;
    const uint32_t   ch   = blockIdx.x;
    pin_sgpr(a.n, a.seg.nscenes, a.seg.rb_scene, a.seg.rb_row0, a.seg.sc_v0, a.z, a.p_old, a.p_new, a.s, a.part_rz,
             a.k, a.check_every, a.abs_tol, a.rel2);
    uint32_t         scene = 0;
    if (rows) scene = a.seg.nscenes == 1u ? 0u : a.seg.rb_scene[rbi];
    else if (CT == 2)
    {
        if (ch >= a.seg.sc_cb0[a.seg.nscenes]) return;
        scene = a.seg.cb_scene[ch];
    }
    PcgState* st = a.s + scene;
    // a row block loads its z and p_old rows before the flag and the partials (overlapped latencies)
    RowBlk rb{};
    f3     zr = mk(0.0f, 0.0f, 0.0f), pr = zr;
    if (rows)
    {
        rb = row_blk_fast(a.seg, a.n, rbi);
        if (rb.valid)
        {
            zr = ld3(a.z, rb.row);
            pr = ld4(a.p_old, rb.row);
        }
    }
    const IterInputs in = iter_inputs(a, scene);
    if (block_flag(&st->converged)) return;
    IterScalars sc = iter_scalars(a, in, sh);
    if (rows && rbi == scene_rb0(a.seg, scene) && threadIdx.x == 0)
    {
        st->rz[a.k & 1u] = sc.rz;
        if (a.k == 0) st->rz0 = sc.rz;
        if (sc.stop)
        {
            st->iters     = a.k;
            st->nan       = (sc.rz == sc.rz) ? 0u : 1u;
            st->converged = 1u;
        }
    }
    if (sc.stop) return;
    const float beta = sc.beta;
    if (rows)
    {
        if (rb.valid) st4(a.p_new, rb.row, zr + beta * pr);
        return;
    }
    auto pf = [&](uint32_t v) { return ld3(a.z, v) + beta * ld4(a.p_old, v); };
    if (CT == 1)
    {
        const uint32_t n = min(*c.count, c.capacity);
        for (uint32_t k = ch * kB + threadIdx.x; k < n; k += nc * kB) vc.tc[k] = contact_t1(c, k, pf);
    }
    else
    {
        const uint32_t e = a.seg.cb_slot0[ch] + threadIdx.x;
        if (e >= vc.ptr[a.seg.sc_v0[scene + 1]]) return;
        const uint32_t ent = vc.list[e];
        if ((ent & 7u) != 0u) return;
        const uint32_t k = ent >> 3;
        vc.tc[k]         = contact_t1(c, k, pf);
    }
}

// One 16-bit entry of a packed mixed-precision block as float (BF16: the high half of an FP32).
template <int LP>
LCSX_D float half_entry(uint32_t bits)
{
    if (LP == 2) return __uint_as_float(bits << 16);
    return __half2float(__ushort_as_half((unsigned short)bits));
}

// Block b of the SELL planes. FP32: the nine planes. 16-bit (LP 1 FP16, 2 BF16): the five packed
// words are requested first (sell_words) and decoded after the column gathers (sell_unpack), so
// the decision on a block kept in FP32 (an affine body's rows) waits for nothing else: the packed
// loads of all the pass's blocks are in flight together.
LCSX_D m3 sell_block32(const SellView& A, size_t b)
{
    m3 M;
#pragma unroll
    for (int c = 0; c < 9; c++) M.m[c] = A.val[c * (size_t)A.nblocks + b];
    return M;
}
struct PackedBlock
{
    uint32_t w[5];
};
LCSX_D PackedBlock sell_words(const SellView& A, size_t b)
{
    PackedBlock P;
#pragma unroll
    for (int c = 0; c < 5; c++) P.w[c] = A.val_p[c * (size_t)A.nblocks + b];
    return P;
}
template <int LP>
LCSX_D m3 sell_unpack(const SellView& A, size_t b, const PackedBlock& P)
{
    const int ex = (int)(int8_t)((P.w[4] >> 16) & 0xffu);
    if (ex == kKeepFp32) return sell_block32(A, b);
    m3          M;
    const float sc = __uint_as_float((uint32_t)(127 + ex) << 23);
#pragma unroll
    for (int c = 0; c < 4; c++)
    {
        M.m[2 * c]     = half_entry<LP>(P.w[c] & 0xffffu) * sc;
        M.m[2 * c + 1] = half_entry<LP>(P.w[c] >> 16) * sc;
    }
    M.m[8] = half_entry<LP>(P.w[4] & 0xffffu) * sc;
    return M;
}

// q = A p for PCG iteration k (newton_solver.cpp:259-472 / 3397-3427 semantics), p.q in the same
// launch. Row blocks (4 n_rb of them: 256 threads = 64 rows, a quarter of a scene-aligned 256-row
// block): each wavefront holds 16 rows of one SELL-16 slice with 4 lanes per row (lane = 16 j + l);
// lane j takes the row's blocks j, j + 4, j + 8, ... so each 64-lane load of a block entry is
// contiguous. A pass issues the column indices, the entries and the 16-byte p gathers of U blocks
// before using any of them; with UNC every lane issues all of its pass's loads (a block past the
// row's width rereads the pass's first block and its product is dropped by a select), so the
// compiler has no branch to sink the later blocks' loads into. Every mapping adds the blocks in
// the order j, j + 4, j + 8, ..., so all give the same bits. The four partial sums of a row are
// combined by two butterflies; lane 0 of the row adds the diagonal block. Contact blocks: one
// scene-aligned 256-slot chunk each, every run of slots of one row summed by a segmented scan and
// stored at the run's last slot (folded into q by the update, fold_runs). p.q partials: four per
// row block, then one per chunk. `cf` > 0 (a multiple of 8) places the chunk blocks first in the
// launch, so their dependent loads overlap the row blocks' streaming instead of trailing it.
template <int LP, int U, bool UNC>
__global__ __launch_bounds__(kB) void k_spmv_pcg(PcgArgs a, SellView A, VertContacts vc, uint32_t cf)
{
    __shared__ float sh[4];
    const uint32_t   n_rb = a.seg.n_rb;
    const uint32_t   lane = lane_id();
    float            loc  = 0.0f;
    const bool       rows = cf ? blockIdx.x >= cf : blockIdx.x < 4u * n_rb;
    pin_sgpr(a.n, n_rb, a.seg.nscenes, a.seg.rb_scene, a.seg.rb_row0, a.seg.sc_v0, A.sl_off, A.col,
             LP ? (const void*)A.val_p : (const void*)A.val, A.diag, A.nblocks, a.p_new, a.q, a.part_pq, a.s);
    if (rows)
    {
        const uint32_t sb    = xcd_block(blockIdx.x - cf, 4u * n_rb);
        const uint32_t rbi   = sb >> 2;
        // one scene: row block rbi starts at row 256 rbi and the rows end at n, with nothing to read
        const bool     one   = a.seg.nscenes == 1u;
        const uint32_t scene = one ? 0u : a.seg.rb_scene[rbi];
        const uint32_t row0  = one ? rbi * 256u : a.seg.rb_row0[rbi];
        const uint32_t j = lane >> 4;
        const uint32_t i = row0 + (sb & 3u) * 64u + (threadIdx.x >> 6) * 16u + (lane & 15u);
        const bool     valid = i < (one ? a.n : a.seg.sc_v0[scene + 1]) && i < row0 + 256u;
        // the slice offsets and the row's own p and diagonal block are read before the converged
        // flag, so their latency overlaps the flag's
        const uint32_t s = i >> 4, l = i & 15u;
        uint32_t       k0 = 0u, wd = 0u;
        f3             y = mk(0.0f, 0.0f, 0.0f), pi = mk(0.0f, 0.0f, 0.0f);
        m3             D;
        if (valid)
        {
            k0 = A.sl_off[s];
            wd = A.sl_off[s + 1] - k0;
            if (j == 0u)
            {
                pi = ld4(a.p_new, i);
                D  = ld_planes(A.diag, a.n, i);
            }
        }
        if (launch_flag(&a.s[scene].converged)) return;
        if (valid)
        {
            if (j == 0u) y = mul(D, pi);
            for (uint32_t kk = j; kk < wd; kk += 4u * U)
            {
                uint32_t cl[U];
                bool     on[U];
                size_t   bb[U];
#pragma unroll
                for (int u = 0; u < U; u++)
                {
                    const uint32_t k = kk + 4u * (uint32_t)u;
                    on[u]            = k < wd;
                    if (UNC)
                    {
                        bb[u] = (size_t)(k0 + (on[u] ? k : kk)) * kSellH + l;
                        cl[u] = A.col[bb[u]];
                    }
                    else
                    {
                        bb[u] = (size_t)(k0 + (on[u] ? k : 0u)) * kSellH + l;
                        cl[u] = on[u] ? A.col[bb[u]] : i;
                    }
                }
                m3          M[U];
                PackedBlock W[U];
#pragma unroll
                for (int u = 0; u < U; u++)
                {
                    if (LP) W[u] = sell_words(A, bb[u]);
                    else M[u] = sell_block32(A, bb[u]);
                }
                f3 pc[U];
#pragma unroll
                for (int u = 0; u < U; u++) pc[u] = ld4(a.p_new, cl[u]);
                if (LP)
                {
#pragma unroll
                    for (int u = 0; u < U; u++) M[u] = sell_unpack<LP>(A, bb[u], W[u]);
                }
#pragma unroll
                for (int u = 0; u < U; u++)
                {
                    if (UNC)
                    {
                        const f3 yy = y + mul(M[u], pc[u]);
                        y.x         = on[u] ? yy.x : y.x;
                        y.y         = on[u] ? yy.y : y.y;
                        y.z         = on[u] ? yy.z : y.z;
                    }
                    else if (on[u])
                        y = y + mul(M[u], pc[u]);
                }
            }
        }
        // the row's four lanes hold partial sums: lanes l, l + 16, l + 32, l + 48
        y = xor_add<32>(xor_add<16>(y));
        if (valid && j < 3u) a.q[3 * (size_t)i + j] = get(y, (int)j);
        if (valid && j == 0u) loc = dot(pi, y);
        const float bs = block_sum(loc, sh);
        if (threadIdx.x == 0) a.part_pq[sb] = bs;
        return;
    }
    // contact slots: chunk ch of 256 slots
    const uint32_t ch = cf ? blockIdx.x : blockIdx.x - 4u * n_rb;
    if (ch >= a.seg.sc_cb0[a.seg.nscenes]) return;
    const uint32_t scene = a.seg.cb_scene[ch];
    if (launch_flag(&a.s[scene].converged)) return;
    uint32_t row;
    f3       sum;
    const uint32_t base = a.seg.cb_slot0[ch] + (threadIdx.x & ~63u);
    if (slot_chunk(vc, base, vc.ptr[a.seg.sc_v0[scene + 1]], row, sum))
    {
        vc.runsum[base + lane] = make_float4(sum.x, sum.y, sum.z, 0.0f);
        loc                    = dot(ld4(a.p_new, row), sum);
    }
    const float bs = block_sum(loc, sh);
    if (threadIdx.x == 0) a.part_pq[4u * n_rb + ch] = bs;
}

__global__ void k_fill_f64(double* a, uint32_t n)
{
    uint32_t i = blockIdx.x * kB + threadIdx.x;
    if (i < n) a[i] = 0.0;
}

// ---------------------------------------------------------------- energy (line search)
// solver_interface.cpp:499-873 (inertia, ground, stretch face, bending, affine-body inertia and
// orthogonality) and narrow_phase.cpp:2964-3070 (the iteration's contact list at the current x).
// Each element in FP32 as the reference (the barrier terms in FP64 in the mixed form), the sums
// in double: per block when the block's elements are of one scene, else per element.
LCSX_D void scene_add(double e, uint32_t scene, double* __restrict__ out)
{
    __shared__ uint32_t s0;
    __shared__ double   sd[kB / 64];
    if (threadIdx.x == 0) s0 = kInvalid;
    __syncthreads();
    if (scene != kInvalid) s0 = scene;  // any one of the block's scenes
    __syncthreads();
    const uint32_t g = s0;
    if (__syncthreads_and(scene == kInvalid || scene == g))
    {
        for (int off = 32; off > 0; off >>= 1) e += __shfl_xor(e, off);
        if (lane_id() == 0) sd[threadIdx.x >> 6] = e;
        __syncthreads();
        if (threadIdx.x == 0 && g != kInvalid) atomicAdd(out + g, ((sd[0] + sd[1]) + sd[2]) + sd[3]);
    }
    else if (scene != kInvalid && e != 0.0)
        atomicAdd(out + scene, e);
}

__global__ __launch_bounds__(kB) void k_energy_rows(EnergyArgs a)
{
    const uint32_t i  = blockIdx.x * kB + threadIdx.x;
    double         e  = 0.0;
    uint32_t       sc = kInvalid;
    if (i < a.nv && a.row_kind[i] < 2u)
    {
        sc = a.vert_scene[i];
        const f3 xi = ld3(a.x, i);
        if (a.row_kind[i] == 0u)
        {
            f3    d  = xi - ld3(a.x_tilde, i);
            float ei = ((a.h2inv * dot(d, d)) * a.mass[i]) / 2.0f;
            if (a.fixed[i]) ei = a.kD * ei;
            e += (double)ei;
        }
        if (a.use_floor && !a.fixed[i])
        {
            const float dist = xi.y - a.floor_y, th = a.offset[i], dh = a.dhat[i];
            if (dist - th < dh)
            {
                const float stiff = a.kappa * a.vert_area[i];
                e += a.fp64 ? fp64::ground_e(a.quadratic, (double)dist, (double)th, (double)dh, (double)stiff)
                            : (double)ground_e(a.quadratic, dist, th, dh, stiff);
            }
        }
    }
    scene_add(e, sc, a.out);
}

__global__ __launch_bounds__(kB) void k_energy_faces(EnergyArgs a)
{
    const uint32_t f  = blockIdx.x * kB + threadIdx.x;
    double         e  = 0.0;
    uint32_t       sc = kInvalid;
    if (f < a.nsf)
    {
        const uint32_t v0 = a.sf[3 * f], v1 = a.sf[3 * f + 1], v2 = a.sf[3 * f + 2];
        sc                = a.vert_scene[v0];
        const float4 D = a.sf_Dm[f], c = a.sf_c[f];
        const f3     e0 = ld3(a.x, v1) - ld3(a.x, v0), e1 = ld3(a.x, v2) - ld3(a.x, v0);
        const f3     Fu = e0 * D.x + e1 * D.y, Fv = e0 * D.z + e1 * D.w;
        const float  su = sqrtf(dot(Fu, Fu)) - 1.0f, sv = sqrtf(dot(Fv, Fv)) - 1.0f, i6 = dot(Fu, Fv);
        e = (double)(c.x * (0.5f * c.y * (su * su + sv * sv) + 0.5f * c.z * (i6 * i6)));
    }
    scene_add(e, sc, a.out);
}

// fn_calc_energy_spring, solver_interface.cpp:603-630: 1/2 k (|x1 - x0| - L)^2
__global__ __launch_bounds__(kB) void k_energy_springs(EnergyArgs a)
{
    const uint32_t e  = blockIdx.x * kB + threadIdx.x;
    double         en = 0.0;
    uint32_t       sc = kInvalid;
    if (e < a.nsp)
    {
        const uint32_t v0 = a.sp[2 * e], v1 = a.sp[2 * e + 1];
        sc                = a.vert_scene[v0];
        const f3     diff = ld3(a.x, v1) - ld3(a.x, v0);
        const float2 rk   = a.sp_c[e];
        const float  C    = sqrtf(dot(diff, diff)) - rk.x;
        en                = (double)(((0.5f * rk.y) * C) * C);
    }
    scene_add(en, sc, a.out);
}

__global__ __launch_bounds__(kB) void k_energy_hinges(EnergyArgs a)
{
    const uint32_t h  = blockIdx.x * kB + threadIdx.x;
    double         e  = 0.0;
    uint32_t       sc = kInvalid;
    if (h < a.nbh)
    {
        const uint32_t* q = a.bh + 4 * (size_t)h;
        sc                = a.vert_scene[q[0]];
        const float4 c    = a.bh_c[h];
        const float  d    = dihedral_angle(ld3(a.x, q[0]), ld3(a.x, q[1]), ld3(a.x, q[2]), ld3(a.x, q[3])) - c.x;
        e                 = (double)(((((0.5f * c.z) * a.scaling) * c.y) * d) * d);
    }
    scene_add(e, sc, a.out);
}

__global__ __launch_bounds__(kB) void k_energy_bodies(EnergyArgs a)
{
    const uint32_t b  = blockIdx.x * kB + threadIdx.x;
    double         e  = 0.0;
    uint32_t       sc = kInvalid;
    if (b < a.nb)
    {
        const BodyDev& B = a.bodies[b];
        sc               = a.vert_scene[B.row0];
        f3 dq[4], A[3];
        for (int k = 0; k < 4; k++) dq[k] = ld3(a.x, B.row0 + k) - ld3(a.x_tilde, B.row0 + k);
        for (int k = 0; k < 3; k++) A[k] = ld3(a.x, B.row0 + 1 + k);
        float ei = 0.0f;
        for (int ii = 0; ii < 4; ii++)
            for (int jj = 0; jj < 4; jj++) ei = ei + ((a.h2inv * dot(dq[ii], dq[jj])) * B.M[4 * ii + jj]) / 2.0f;
        if (B.fixed) ei = ei * a.kD;
        float o = 0.0f;
        for (int ii = 0; ii < 3; ii++)
            for (int jj = 0; jj < 3; jj++)
            {
                float t = dot(A[ii], A[jj]) - (ii == jj ? 1.0f : 0.0f);
                o       = o + t * t;
            }
        e = (double)ei + (double)(o * B.stiff);
    }
    scene_add(e, sc, a.out);
}

__global__ __launch_bounds__(kB) void k_energy_contacts(EnergyArgs a)
{
    const uint32_t n = min(*a.c.count, a.c.capacity);
    for (uint32_t base = blockIdx.x * kB; base < n; base += gridDim.x * kB)
    {
        const uint32_t k  = base + threadIdx.x;
        double         e  = 0.0;
        uint32_t       sc = kInvalid;
        if (k < n)
        {
            const uint4  I  = a.c.idx[k];
            const float4 w  = a.c.w[k];
            const float  ak = a.c.aux[k].y;
            const uint32_t i0 = I.x & 0x7fffffffu, i1 = I.y & 0x7fffffffu, i2 = I.z & 0x7fffffffu, i3 = I.w & 0x7fffffffu;
            sc                = a.vert_scene[i0];
            const f3    diff = ((w.x * ld3(a.x, i0) + w.y * ld3(a.x, i1)) + w.z * ld3(a.x, i2)) + w.w * ld3(a.x, i3);
            const float d    = sqrtf(dot(diff, diff));
            const float dh   = 0.5f * (a.dhat[i0] + a.dhat[i2]);
            const float th   = a.offset[i0] + a.offset[i2];
            if (d < th + dh)
                e = a.fp64 ? fp64::pair_e(a.quadratic, (double)d, (double)th, (double)dh, (double)ak)
                           : (double)pair_e(a.quadratic, d, th, dh, ak);
        }
        scene_add(e, sc, a.out);
    }
}


// BF16 of a finite float, rounded to nearest even (the upper 16 bits of the rounded float).
LCSX_D uint16_t float_to_bf16_rn(float x)
{
    const uint32_t u = __float_as_uint(x);
    return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

// Mixed precision: FP16 copy of the off-diagonal blocks, each block scaled by 2^-e with 2^e the
// smallest power of two above its largest magnitude (entries in (-1, 1), 11 significant bits).
// One thread per SELL row (rows past n are slice padding): each block as nine 16-bit entries times
// 2^e, e the exponent of the block's largest magnitude, packed into five 32-bit planes (SellView).
// An affine body's rows keep their FP32 blocks (exponent kKeepFp32): its 12x12 system couples the
// orthogonality stiffness with the rotational inertia, eigenvalues about six orders of magnitude
// apart, which 11 bits cannot hold.
__global__ __launch_bounds__(kB) void k_pack_fp16(uint32_t nslices, uint32_t n, const uint32_t* __restrict__ sl_off,
                                                   uint32_t nb, const float* __restrict__ val,
                                                   const uint8_t* __restrict__ row_kind, uint32_t* __restrict__ vp,
                                                   int bf16)
{
    uint32_t r = blockIdx.x * kB + threadIdx.x;
    if (r >= nslices * kSellH) return;
    const uint32_t s = r / kSellH, l = r % kSellH;
    const bool     keep = r < n && row_kind != nullptr && row_kind[r] >= 2;
    for (uint32_t k = sl_off[s]; k < sl_off[s + 1]; k++)
    {
        const size_t b = (size_t)k * kSellH + l;
        if (keep)
        {
            vp[4 * (size_t)nb + b] = (uint32_t)(uint8_t)kKeepFp32 << 16;
            continue;
        }
        float v[9], m = 0.0f;
#pragma unroll
        for (int c = 0; c < 9; c++)
        {
            v[c] = val[c * (size_t)nb + b];
            m    = fmaxf(m, fabsf(v[c]));
        }
        int e = 0;
        if (m > 0.0f) frexpf(m, &e);  // m = f 2^e, f in [0.5, 1)
        e        = max(-100, min(100, e));
        float    sc = __int_as_float((127 - e) << 23);
        uint32_t h[9];
#pragma unroll
        for (int c = 0; c < 9; c++)
            h[c] = bf16 ? (uint32_t)float_to_bf16_rn(v[c] * sc)
                        : (uint32_t)__half_as_ushort(__float2half_rn(v[c] * sc));
#pragma unroll
        for (int c = 0; c < 4; c++) vp[c * (size_t)nb + b] = h[2 * c] | (h[2 * c + 1] << 16);
        vp[4 * (size_t)nb + b] = h[8] | ((uint32_t)(uint8_t)(int8_t)e << 16);
    }
}

// Knuth's TwoSum: s + e = a + b exactly.
LCSX_D void two_sum(float a, float b, float& s, float& e)
{
    s        = a + b;
    float bb = s - a;
    e        = (a - (s - bb)) + (b - bb);
}

// Residual replacement of the mixed-precision PCG: r = b - y with y = A x from the FP32 blocks (the
// true residual), z = Minv r, and the block's r.z summed pairwise with TwoSum, the rounding errors
// carried alongside: part_rz[block] = sum + error (read by the next iteration), part_res[2 block]
// = (sum, error) for the host's double total.
__global__ __launch_bounds__(kB) void k_residual(SegView g, const float* __restrict__ b, const float* __restrict__ y,
                                                  const float* __restrict__ minv, float* __restrict__ r,
                                                  float* __restrict__ z, float* __restrict__ part_rz,
                                                  float* __restrict__ part_res)
{
    __shared__ float ss[kB], se[kB];
    const RowBlk     rb = row_blk(g);
    const uint32_t   i  = rb.row, n = g.sc_v0[g.nscenes];
    float            s = 0.0f, e = 0.0f;
    if (rb.valid)
    {
        f3 ri = ld3(b, i) - ld3(y, i);
        st3(r, i, ri);
        f3 zi = mul(ld_planes(minv, n, i), ri);
        st3(z, i, zi);
        float p0 = ri.x * zi.x, p1 = ri.y * zi.y, p2 = ri.z * zi.z;
        float t, u;
        two_sum(p0, p1, s, e);
        two_sum(s, p2, t, u);
        s = t;
        e = e + u;
    }
    ss[threadIdx.x] = s;
    se[threadIdx.x] = e;
    __syncthreads();
    for (uint32_t h = kB / 2; h > 0; h >>= 1)
    {
        if (threadIdx.x < h)
        {
            float t, u;
            two_sum(ss[threadIdx.x], ss[threadIdx.x + h], t, u);
            ss[threadIdx.x] = t;
            se[threadIdx.x] = (se[threadIdx.x] + se[threadIdx.x + h]) + u;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0)
    {
        part_rz[blockIdx.x]          = ss[0] + se[0];
        part_res[2 * blockIdx.x]     = ss[0];
        part_res[2 * blockIdx.x + 1] = se[0];
    }
}

// y = A p: rows (diagonal and material blocks, FP32 or the packed 16-bit ones) in one launch, then
// the contact slots added to y.
template <int LP>
__global__ __launch_bounds__(kB) void k_spmv_plain(uint32_t n, SellView A, const float* __restrict__ p, float* __restrict__ y)
{
    uint32_t i = blockIdx.x * kB + threadIdx.x;
    if (i >= n) return;
    f3       out = mul(ld_planes(A.diag, n, i), ld3(p, i));
    uint32_t s   = i / kSellH, l = i % kSellH;
    for (uint32_t k = A.sl_off[s]; k < A.sl_off[s + 1]; k++)
    {
        size_t b = (size_t)k * kSellH + l;
        const m3 M = LP ? sell_unpack<LP>(A, b, sell_words(A, b)) : sell_block32(A, b);
        out        = out + mul(M, ld3(p, A.col[b]));
    }
    st3(y, i, out);
}

__global__ __launch_bounds__(kB) void k_slots_plain(VertContacts vc)
{
    uint32_t       row;
    f3             sum;
    const uint32_t base = blockIdx.x * kB + (threadIdx.x & ~63u);
    if (slot_chunk(vc, base, *vc.total, row, sum)) vc.runsum[base + lane_id()] = make_float4(sum.x, sum.y, sum.z, 0.0f);
}
__global__ __launch_bounds__(kB) void k_fold_plain(VertContacts vc, uint32_t n, float* __restrict__ y)
{
    const uint32_t i = blockIdx.x * kB + threadIdx.x;
    if (i < n) st3(y, i, fold_runs(ld3(y, i), vc.runsum, vc.ptr, i, 0u));
}

__global__ __launch_bounds__(kB) void k_pcg_update(PcgArgs a)
{
    __shared__ float sh[4];
    const uint32_t rbi = xcd_block(blockIdx.x, a.seg.n_rb);
    pin_sgpr(a.n, a.seg.nscenes, a.seg.rb_scene, a.seg.rb_row0, a.seg.sc_v0, a.p_new, a.x, a.q, a.r, a.z, a.minv,
             a.runsum, a.vc_ptr, a.s, a.part_pq, a.part_rz, a.k);
    const RowBlk   rb  = row_blk_fast(a.seg, a.n, rbi);
    PcgState*    st = a.s + rb.scene;
    const uint32_t i = rb.row;
    // the row's operands do not depend on alpha: they are loaded before the converged flag and the
    // p.q partials are read, so the latencies of the three reads overlap
    f3 pn = mk(0.0f, 0.0f, 0.0f), x0 = pn, q = pn, r0 = pn;
    m3 Mi;
    if (rb.valid)
    {
        pn = ld4(a.p_new, i);
        x0 = ld3(a.x, i);
        q  = ld3(a.q, i);
        if (a.runsum) q = fold_runs(q, a.runsum, a.vc_ptr, i, a.vc_ptr[a.seg.nscenes == 1u ? 0u : a.seg.sc_v0[rb.scene]]);
        r0 = ld3(a.r, i);
        Mi = ld_planes(a.minv, a.n, i);
    }
    const SegView&    g   = a.seg;
    const PrePartials pre = prefetch_ranges(a.part_pq, 4u * scene_rb0(g, rb.scene), 4u * scene_rb0(g, rb.scene + 1),
                                            4u * g.n_rb + g.sc_cb0[rb.scene], 4u * g.n_rb + g.sc_cb0[rb.scene + 1]);
    const float       rz  = st->rz[a.k & 1u];
    if (launch_flag(&st->converged)) return;
    const float    pq    = reduce_prefetched(a.part_pq, pre, sh);
    const float    alpha = pq < 1e-10f ? 0.0f : rz / pq;
    float          loc   = 0.0f;
    if (rb.valid)
    {
        st3(a.x, i, x0 + alpha * pn);
        f3 r = r0 - alpha * q;
        st3(a.r, i, r);
        f3 z = mul(Mi, r);
        st3(a.z, i, z);
        loc = dot(r, z);
    }
    float bs = block_sum(loc, sh);
    if (threadIdx.x == 0) a.part_rz[rbi] = bs;
}

// ---------------------------------------------------------------- PCG in one launch (lcsx_pcg_grid.h)
// The SELL-16 matrix and the contact slots as k_pcg_grid reads them.
template <int LP>
struct GridSell
{
    SellView A;
    uint32_t n;
    struct Row
    {
        uint32_t b0, count;  // block k at b0 + 16 k
        bool     ok;
    };
    using Raw = typename std::conditional<LP != 0, PackedBlock, m3>::type;
    LCSX_D Row row(uint32_t i) const
    {
        const uint32_t s = i >> 4, k0 = A.sl_off[s];
        return Row{k0 * kSellH + (i & 15u), A.sl_off[s + 1] - k0, true};
    }
    LCSX_D uint32_t col(const Row& r, uint32_t k) const { return A.col[r.b0 + kSellH * k]; }
    LCSX_D Raw      load(const Row& r, uint32_t k) const
    {
        if constexpr (LP != 0) return sell_words(A, r.b0 + kSellH * k);
        else return sell_block32(A, r.b0 + kSellH * k);
    }
    LCSX_D m3 get(const Raw& w, uint32_t i, uint32_t k, bool on) const
    {
        if constexpr (LP != 0)
        {
            // a block kept in FP32 (an affine body's row) is read from its planes
            const bool keep = (int)(int8_t)((w.w[4] >> 16) & 0xffu) == kKeepFp32;
            return sell_unpack<LP>(A, on && keep ? (size_t)(A.sl_off[i >> 4] + k) * kSellH + (i & 15u) : 0, w);
        }
        else
            return w;
    }
    LCSX_D m3   diag(uint32_t i) const { return ld_planes(A.diag, n, i); }
    LCSX_D m3   minv(const float* P, uint32_t i) const { return ld_planes(P, n, i); }
    LCSX_D void bad_column() const {}
    // keeps the decoding of 16-bit blocks inside the iteration: hoisted out of it, the decoded blocks
    // would take nearly twice the registers
    template <int U, int K>
    LCSX_D void opaque(Raw (&W)[U][K]) const
    {
        if constexpr (LP != 0)
        {
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int k = 0; k < K; k++)
#pragma unroll
                    for (int c = 0; c < 5; c++) asm volatile("" : "+v"(W[u][k].w[c]));
        }
    }
};
struct GridContacts
{
    ContactView  c;
    VertContacts vc;
    uint32_t     c0 = 0, nch = 0, s0 = 0, end = 0, part = 0, parts = 1;  // the scene's chunks and slots
    LCSX_D void  begin(const PcgArgs& a, uint32_t scene, uint32_t part_, uint32_t parts_)
    {
        c0    = a.seg.nscenes == 1u ? 0u : a.seg.sc_cb0[scene];
        nch   = a.seg.sc_cb0[scene + 1] - c0;
        s0    = vc.ptr[a.seg.nscenes == 1u ? 0u : a.seg.sc_v0[scene]];
        end   = vc.ptr[a.seg.nscenes == 1u ? a.n : a.seg.sc_v0[scene + 1]];
        part  = part_;
        parts = parts_;
    }
    LCSX_D uint32_t first() const { return c0; }
    LCSX_D uint32_t chunks() const { return nch; }
    // p = z + beta p_old of four rows at once (kInvalid: none), every load in flight before the first is
    // used
    struct P4
    {
        f3 p[4];
    };
    LCSX_D P4 rows4(const PcgArgs& a, const grid::Word* zx, bool first, uint32_t zep, const float* p_old, float beta,
                    const uint32_t (&r)[4], uint32_t& bad) const
    {
        P4 o;
        if (first)
        {
#pragma unroll
            for (int j = 0; j < 4; j++)
            {
                const uint32_t v = r[j] != kInvalid ? r[j] : 0u;
                o.p[j]           = ld3(a.z, v) + beta * ld4(p_old, v);
            }
            return o;
        }
        f3 po[4];
#pragma unroll
        for (int j = 0; j < 4; j++) po[j] = grid::ld_row(p_old, r[j] != kInvalid ? r[j] : 0u);
        for (uint32_t tries = 0;; tries++)
        {
            grid::Word w[4][3];
#pragma unroll
            for (int j = 0; j < 4; j++)
            {
                const uint32_t v = r[j] != kInvalid ? r[j] : 0u;
#pragma unroll
                for (int d = 0; d < 3; d++) w[j][d] = grid::peek(zx + d * (size_t)a.n + v);
            }
            bool ok = true;
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int d = 0; d < 3; d++) ok = ok && (r[j] == kInvalid || grid::epoch_of(w[j][d]) == zep);
            if (!ok && tries > grid::kPolls) bad = 1u;
            if (ok || *(volatile uint32_t*)&bad != 0u)
            {
#pragma unroll
                for (int j = 0; j < 4; j++)
                    o.p[j] = mk(grid::value_of(w[j][0]), grid::value_of(w[j][1]), grid::value_of(w[j][2])) + beta * po[j];
                return o;
            }
        }
    }
    // The runs of this workgroup's 256-slot chunks and their p.q partials. p of other workgroups' rows
    // is z + beta p_old again, and every slot evaluates its contact's t_c itself (contact_t1's
    // expression, so the same bits): a wait of all workgroups for the t_c would cost more than the
    // repetition as long as the contacts are few (the limit in Solver::pcg_run).
    LCSX_D void slots(const PcgArgs& a, const grid::Word* zx, bool first, uint32_t zep, const float* p_old, float beta,
                      grid::Word* words, uint32_t epoch, float* sh, uint32_t& bad) const
    {
        const uint32_t gpw = blockDim.x >> 8, grp = threadIdx.x >> 8, wv = threadIdx.x >> 6;
        for (uint32_t base = part * gpw; base < nch; base += parts * gpw)
        {
            const uint32_t ch  = base + grp;
            float          loc = 0.0f;
            if (ch < nch)
            {
                uint32_t       row;
                f3             sum, pr = mk(0.0f, 0.0f, 0.0f);
                const uint32_t b = s0 + 256u * ch + (threadIdx.x & 192u);
                auto           tf = [&](uint32_t k) {
                    const float4   nk  = c.nk[k];
                    const f3       nn  = mk(nk.x, nk.y, nk.z);
                    const uint32_t own = vc.row[b + lane_id()];
                    uint32_t       ra[4], rb[4];
                    float          fa[4], fb[4];
                    gdofs4(c, k, 0u, ra, fa);
                    gdofs4(c, k, 1u, rb, fb);
                    const P4       A = rows4(a, zx, first, zep, p_old, beta, ra, bad);
                    float          t = fa[0] * dot(nn, A.p[0]);
#pragma unroll
                    for (int j = 0; j < 4; j++)
                    {
                        if (j > 0 && ra[j] != kInvalid) t = t + fa[j] * dot(nn, A.p[j]);
                        if (ra[j] == own) pr = A.p[j];
                    }
                    if (rb[0] != kInvalid || rb[1] != kInvalid || rb[2] != kInvalid || rb[3] != kInvalid)
                    {
                        const P4 B = rows4(a, zx, first, zep, p_old, beta, rb, bad);
#pragma unroll
                        for (int j = 0; j < 4; j++)
                        {
                            if (rb[j] != kInvalid) t = t + fb[j] * dot(nn, B.p[j]);
                            if (rb[j] == own) pr = B.p[j];
                        }
                    }
                    return t;
                };
                if (slot_chunk(vc, b, end, row, sum, tf))
                {
                    grid::st_row(reinterpret_cast<float*>(vc.runsum), b + lane_id(), sum);
                    loc = dot(pr, sum);
                }
            }
            loc = wave_sum(loc);
            if (lane_id() == 0) sh[wv] = loc;
            grid::stores_done();  // the runs' sums, before the word that announces them
            __syncthreads();
            if ((threadIdx.x & 255u) == 0u && ch < nch)
                grid::post(words + c0 + ch, ((sh[wv] + sh[wv + 1]) + sh[wv + 2]) + sh[wv + 3], epoch);
            __syncthreads();
        }
    }
    LCSX_D void poison(grid::Word* words) const
    {
        const uint32_t gpw = blockDim.x >> 8;
        for (uint32_t base = part * gpw; base < nch; base += parts * gpw)
            for (uint32_t ch = base; ch < min(base + gpw, nch); ch++) grid::post(words + c0 + ch, 0.0f, grid::kPoison);
    }
    LCSX_D f3 fold(f3 q, uint32_t i) const
    {
        return fold_runs_of(
            q, [&](uint32_t e) { return grid::ld_row(reinterpret_cast<const float*>(vc.runsum), e); }, vc.ptr, i,
            s0);
    }
};
__global__ void k_grid_clear(unsigned long long* w, size_t n)
{
    for (size_t i = blockIdx.x * kB + threadIdx.x; i < n; i += (size_t)gridDim.x * kB) w[i] = 0ull;
}

// Standalone narrow phase: the pair count and the CCD's rest count and step bound of one call.
__global__ void k_narrow_init(uint32_t* cnt, uint32_t n_pairs, SceneStatus* st)
{
    if (blockIdx.x == 0 && threadIdx.x == 0)
    {
        cnt[0] = n_pairs;
        cnt[1] = 0u;
        if (st) *st = SceneStatus{f2ord(1.0f), 0u, 0u, 0u};
    }
}
__global__ void k_toi_out(const SceneStatus* st, float* toi)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) toi[0] = ord2f(st->toi_bits);
}

// ---------------------------------------------------------------- line search
__global__ void k_apply_dx(uint32_t nv, const float* __restrict__ x_iter, const float* __restrict__ dx, float* __restrict__ x,
                           const SceneStatus* __restrict__ sst, float alpha_const, SegView g)
{
    uint32_t i = blockIdx.x * kB + threadIdx.x;
    if (i >= nv) return;
    uint32_t sc    = g.vert_scene[i];
    float    alpha = sst ? ord2f(sst[sc].toi_bits) : alpha_const;
    if (g.active && g.active[sc] == 0) alpha = 0.0f;
    st3(x, i, ld3(x_iter, i) + alpha * ld3(dx, i));
}

// fn_gound_collision_ccd, newton_solver.cpp:952-1000 (+ NaN check of dx and max |dx|)
__global__ __launch_bounds__(kB) void k_ground_ccd_maxdx(LsArgs a)
{
    __shared__ float sh[4][2];
    const RowBlk     rb = row_blk(a.seg);
    const uint32_t   i  = rb.row;
    float            toi = 1.0f, mdx = 0.0f;
    if (rb.valid)
    {
        f3 d = ld3(a.dx, i);
        mdx  = length(d);
        if (!(mdx == mdx)) atomicOr(&a.st->nan, 1u);
        if (a.use_floor && !a.fixed[i] && a.row_kind[i] < 2u)
        {
            float off = a.offset[i], cy = a.x[3 * (size_t)i + 1];
            if (cy - off < a.floor_y)
            {
                float iy = a.x_iter[3 * (size_t)i + 1];
                toi      = ((iy - off) - a.floor_y) / (iy - cy) / kLineSearchMaxT;
            }
        }
    }
    toi   = wave_min(toi);
    mdx   = wave_max(mdx);
    int w = threadIdx.x >> 6;
    if (lane_id() == 0)
    {
        sh[w][0] = toi;
        sh[w][1] = mdx;
    }
    __syncthreads();
    if (threadIdx.x == 0)
    {
        float t = fminf(fminf(sh[0][0], sh[1][0]), fminf(sh[2][0], sh[3][0]));
        float m = fmaxf(fmaxf(sh[0][1], sh[1][1]), fmaxf(sh[2][1], sh[3][1]));
        if (t != 1.0f) atomicMin(&a.sst[rb.scene].toi_bits, f2ord(t));
        atomicMax(&a.sst[rb.scene].maxdx_bits, __float_as_uint(m));
    }
}

// fn_narrow_phase_{vf,ee}_ccd_query, narrow_phase.cpp:293-593: min over pairs of toi / 1.25.
// One instance per pair kind (KIND: 0 vertex-face, 1 edge-edge) and arithmetic (FP64: the double
// ACCD of the mixed forms), so each is allocated the registers of its own ACCD loop: the double
// loop needs about twice those of the FP32 one, and a kernel holding both ran at two wavefronts
// per SIMD.
template <bool FP64, int KIND>
__global__ __launch_bounds__(kB) void k_ccd(CcdArgs a)
{
    __shared__ float    sh[4];
    __shared__ uint32_t s_any;
    uint32_t         n    = a.rest ? min(*a.rest_count, a.pair_capacity) : min(*a.pair_count, a.pair_capacity);
    // smallest step bound of this thread's pairs, per run of pairs of one scene (pairs of one
    // scene are mostly contiguous in the list)
    uint32_t         cs   = kInvalid;
    float            cmin = 1.0f;
    if (threadIdx.x == 0) s_any = kInvalid;
    for (uint32_t idx = blockIdx.x * kB + threadIdx.x; idx < n; idx += gridDim.x * kB)
    {
        uint32_t p = a.rest ? a.rest_list[idx] : idx;
        uint32_t q = a.pairs[2 * (size_t)p], o = a.pairs[2 * (size_t)p + 1];
        uint32_t v[4];
        if (KIND == 0)
        {
            v[0] = q;
            v[1] = a.faces[3 * o];
            v[2] = a.faces[3 * o + 1];
            v[3] = a.faces[3 * o + 2];
            if (v[0] == v[1] || v[0] == v[2] || v[0] == v[3]) continue;
            if (a.vert_body && a.vert_body[v[0]] != kInvalid && a.vert_body[v[0]] == a.vert_body[v[1]]) continue;  // narrow_phase.cpp:324-325
        }
        else
        {
            v[0] = a.edges[2 * q];
            v[1] = a.edges[2 * q + 1];
            v[2] = a.edges[2 * o];
            v[3] = a.edges[2 * o + 1];
            if (v[0] == v[2] || v[0] == v[3] || v[1] == v[2] || v[1] == v[3]) continue;
            if (a.vert_body && a.vert_body[v[0]] != kInvalid && a.vert_body[v[0]] == a.vert_body[v[2]]) continue;  // narrow_phase.cpp:471-472
        }
        f3 x0[4], x1[4];
        for (int k = 0; k < 4; k++)
        {
            x0[k] = ld3(a.x0, v[k]);
            x1[k] = ld3(a.x1, v[k]);
        }
        float off  = a.offset[v[0]] + a.offset[KIND == 0 ? v[1] : v[2]];
        bool  done = true;
        float b    = 1.0f;
        if (FP64)
        {
            // double ACCD on the FP32 positions; its step bound toi / 1.25 rounded toward zero, so
            // the FP32 bound is never later than the double one
            fp64::d3 d0[4], d1[4];
            for (int k = 0; k < 4; k++)
            {
                d0[k] = fp64::wide(x0[k]);
                d1[k] = fp64::wide(x1[k]);
            }
            double t = fp64::accd_budget(d0, d1, (double)a.offset[v[0]] + (double)a.offset[KIND == 0 ? v[1] : v[2]],
                                         KIND, a.rest ? 0x7fffffff : a.budget, &done);
            if (done) b = __double2float_rd(t / fp64::kMaxT);
        }
        else
        {
            // FP32: toi / 1.25 (the minimum of the quotients is the quotient of the minimum)
            float t = accd_budget(x0, x1, off, KIND, a.rest ? 0x7fffffff : a.budget, &done);
            if (done && t != kLineSearchMaxT) b = t / kLineSearchMaxT;
        }
        uint32_t slot = wave_append(a.rest_count, !done);
        if (!done && slot < a.pair_capacity) a.rest_list[slot] = p;
        uint32_t sc = a.vert_scene ? a.vert_scene[v[0]] : 0u;
        if (sc != cs)
        {
            if (cs != kInvalid && cmin < 1.0f) atomicMin(&a.sst[cs].toi_bits, f2ord(cmin));
            cs   = sc;
            cmin = 1.0f;
        }
        cmin = fminf(cmin, b);
    }
    // one scene in the whole block (always with one scene): a block minimum and one atomic
    __syncthreads();
    if (cs != kInvalid) s_any = cs;
    __syncthreads();
    const uint32_t s0 = s_any;
    if (__syncthreads_and(cs == kInvalid || cs == s0))
    {
        float bound = wave_min(cmin);
        int   w     = threadIdx.x >> 6;
        if (lane_id() == 0) sh[w] = bound;
        __syncthreads();
        if (threadIdx.x == 0)
        {
            float t = fminf(fminf(sh[0], sh[1]), fminf(sh[2], sh[3]));
            if (s0 != kInvalid && t < 1.0f) atomicMin(&a.sst[s0].toi_bits, f2ord(t));
        }
    }
    else if (cs != kInvalid && cmin < 1.0f)
        atomicMin(&a.sst[cs].toi_bits, f2ord(cmin));
}

// max |x - x_tilde| over pinned vertices (line_search, newton_solver.cpp:3860-3882)
__global__ void k_pin_delta(uint32_t nfix, const uint32_t* __restrict__ ids, const float* __restrict__ x,
                            const float* __restrict__ x_tilde, SceneStatus* __restrict__ sst,
                            const uint32_t* __restrict__ vert_scene)
{
    uint32_t k  = blockIdx.x * kB + threadIdx.x;
    float    d  = 0.0f;
    uint32_t sc = kInvalid;
    if (k < nfix)
    {
        uint32_t i = ids[k];
        d          = length(ld3(x, i) - ld3(x_tilde, i));
        sc         = vert_scene[i];
    }
    uint32_t s0 = __shfl(sc, 0);
    if (__ballot(sc != kInvalid && sc != s0) == 0ull)
    {
        d = wave_max(d);
        if (lane_id() == 0 && s0 != kInvalid) atomicMax(&sst[s0].pin_bits, __float_as_uint(d));
    }
    else if (sc != kInvalid)
        atomicMax(&sst[sc].pin_bits, __float_as_uint(d));
}

__global__ void k_reset_ls(Status* st, SceneStatus* sst, uint32_t nscenes)
{
    uint32_t i = blockIdx.x * kB + threadIdx.x;
    if (i == 0) st->n_vf_ccd = st->n_ee_ccd = 0;
    if (i < nscenes) sst[i] = SceneStatus{f2ord(1.0f), 0u, 0u, 0u};
}

__global__ void k_reset_status(Status* st, SceneStatus* sst, uint32_t nscenes)
{
    uint32_t i = blockIdx.x * kB + threadIdx.x;
    if (i == 0)
    {
        // the CCD counts stay: the next DCD may run on the last line search's candidates (the
        // line search resets them before its own broad phase)
        st->n_vf = st->n_ee = st->n_contacts = st->overflow = 0;
        st->nan = 0;
    }
    if (i < nscenes) sst[i] = SceneStatus{f2ord(1.0f), 0u, 0u, 0u};
}
}  // namespace

// ---------------------------------------------------------------- launchers
uint32_t scan_tmp_words(uint32_t n) { return (n + kScanTile - 1) / kScanTile + 1; }
void launch_scan_excl_u32(const uint32_t* in, uint32_t* out, uint32_t n, uint32_t* tmp, hipStream_t s)
{
    const uint32_t m = (n + kScanTile - 1) / kScanTile;
    if (m == 0)
    {
        k_fill_u32<<<1, kB, 0, s>>>(out, 1, 0u);
        return;
    }
    if (m == 1) k_scan_one<1><<<1, 1024, 0, s>>>(in, n, out);
    else if (m <= 4) k_scan_one<4><<<1, 1024, 0, s>>>(in, n, out);
    else if (m <= kScanPasses) k_scan_one<kScanPasses><<<1, 1024, 0, s>>>(in, n, out);
    else
    {
        k_scan_tiles<<<m, 1024, 0, s>>>(in, n, tmp);
        k_scan_parts<<<1, 1024, 0, s>>>(tmp, m);
        k_scan_apply<<<m, 1024, 0, s>>>(in, n, tmp, out);
    }
}
void launch_fill_u32(uint32_t* a, uint32_t n, uint32_t v, hipStream_t s)
{
    if (n) k_fill_u32<<<grid_for(n, kB), kB, 0, s>>>(a, n, v);
}
void launch_pin_velocity(uint32_t nfix, const uint32_t* ids, const float* targets, const float* x, float* v, float dt, hipStream_t s)
{
    if (nfix) k_pin_velocity<<<grid_for(nfix, kB), kB, 0, s>>>(nfix, ids, targets, x, v, dt);
}
void launch_predict(uint32_t nv, const float* x_step, const float* v, const uint8_t* fixed, const uint8_t* row_kind,
                    float h, const float g[3], float* x_iter, float* x_tilde, float* x, hipStream_t s)
{
    k_predict<<<grid_for(nv, kB), kB, 0, s>>>(nv, x_step, v, fixed, row_kind, h, mk(g[0], g[1], g[2]), x_iter, x_tilde, x);
}
void launch_frame_end(uint32_t nv, float* x_step, const float* x, float* v, float h, float damp, hipStream_t s)
{
    k_frame_end<<<grid_for(nv, kB), kB, 0, s>>>(nv, x_step, x, v, h, damp);
}
void launch_face_stage(uint32_t nsf, const uint32_t* sf, const float4* Dm, const float4* c, const float* x, float* stage,
                       hipStream_t s)
{
    if (nsf) k_face_stage<<<grid_for(nsf, kB), kB, 0, s>>>(nsf, sf, Dm, c, x, stage);
}
void launch_hinge_stage(uint32_t nbh, const uint32_t* bh, const float4* c, float scaling, const float* x, float* stage,
                        hipStream_t s)
{
    if (nbh) k_hinge_stage<<<grid_for(nbh, kB), kB, 0, s>>>(nbh, bh, c, scaling, x, stage);
}
void launch_vert_assemble(const VertArgs& a, hipStream_t s) { k_vert_assemble<<<grid_for(a.nv, kB), kB, 0, s>>>(a); }
void launch_spring_stage(uint32_t nsp, const uint32_t* sp, const float2* c, const float* x, float* stage, hipStream_t s)
{
    if (nsp) k_spring_stage<<<grid_for(nsp, kB), kB, 0, s>>>(nsp, sp, c, x, stage);
}
void launch_offdiag(uint32_t nblocks, const uint32_t* ptr, const uint32_t* con, const float* ss, const float* fs, const float* hs,
                    float* val, hipStream_t s)
{
    if (nblocks) k_offdiag<<<grid_for(nblocks, kB), kB, 0, s>>>(nblocks, ptr, con, ss, fs, hs, val);
}
void launch_abd_material(const AbdArgs& a, hipStream_t s)
{
    if (a.nb) k_abd_material<<<grid_for(a.nb, kB), kB, 0, s>>>(a);
}
void launch_rigid_positions(uint32_t n_rows, const uint8_t* row_kind, const uint32_t* vert_body, const BodyDev* bodies,
                            const float* body_X, float* x, hipStream_t s)
{
    k_rigid_positions<<<grid_for(n_rows, kB), kB, 0, s>>>(n_rows, row_kind, vert_body, bodies, body_X, x);
}
void launch_contact_lift(const ContactView& c, unsigned grid, const uint32_t* vert_body, const BodyDev* bodies,
                         const float* body_X, uint4* gr, float4* gw, hipStream_t s)
{
    k_contact_lift<<<grid, kB, 0, s>>>(c, vert_body, bodies, body_X, gr, gw);
}
void launch_dcd(const DcdArgs& a, int kind, unsigned grid, hipStream_t s)
{
    if (kind == 0)
    {
        if (a.fp64) k_dcd_vf<true><<<grid, kB, 0, s>>>(a);
        else k_dcd_vf<false><<<grid, kB, 0, s>>>(a);
    }
    else if (a.fp64) k_dcd_ee<true><<<grid, kB, 0, s>>>(a);
    else k_dcd_ee<false><<<grid, kB, 0, s>>>(a);
}
void launch_contact_adjacency(const ContactView& c, uint32_t nv, unsigned grid, uint32_t* cnt, uint32_t* ptr,
                              uint32_t* list, uint32_t* row, float4* coef, uint32_t* tmp, const SegView& g,
                              uint32_t* sc_cb0, uint32_t* cb_scene, uint32_t* cb_slot0, bool repeats, hipStream_t s)
{
    k_fill_u32<<<grid_for(nv + 1, kB), kB, 0, s>>>(cnt, nv + 1, 0u);
    k_vc_count<<<grid, kB, 0, s>>>(c, cnt);
    launch_scan_excl_u32(cnt, ptr, nv, list, s);  // list: scratch for the tile sums (refilled below)
    k_fill_u32<<<grid_for(nv + 1, kB), kB, 0, s>>>(cnt, nv + 1, 0u);
    k_vc_fill<<<grid, kB, 0, s>>>(c, ptr, cnt, list, row);
    if (repeats) k_vc_rank<true><<<4 * grid, kB, 0, s>>>(c, ptr, row, ptr + nv, list, tmp);
    else k_vc_rank<false><<<4 * grid, kB, 0, s>>>(c, ptr, row, ptr + nv, list, tmp);
    k_vc_coeffs<<<4 * grid, kB, 0, s>>>(c, ptr, nv, tmp, list, coef);
    k_chunk_table<<<1, 1024, 0, s>>>(g, ptr, sc_cb0, cb_scene, cb_slot0);
}
uint32_t launch_contact_triplets(const ContactView& c, uint32_t n_contacts, unsigned grid, ContactTripletBufs& b,
                                 hipStream_t s)
{
    if (n_contacts == 0) return 0;
    k_ct_count<<<grid, kB, 0, s>>>(c, b.cnt);
    launch_scan_excl_u32(b.cnt, b.ptr, n_contacts, b.scan_tmp, s);
    uint32_t total = 0;
    LCSX_HIP(hipMemcpyAsync(&total, b.ptr + n_contacts, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
    LCSX_HIP(hipStreamSynchronize(s));
    if (total == 0) return 0;
    b.reserve(total, s);
    k_ct_fill<<<grid, kB, 0, s>>>(c, b.ptr, b.row[0], b.col[0], b.idx[0], b.blk);
    const int cur = launch_sort_key_pairs(b.col, b.row, b.idx, total, 32, 32, b.hist, b.sort_tmp, s);
    k_ct_heads<<<grid_for(total, kB), kB, 0, s>>>(total, b.row[cur], b.col[cur], b.head);
    launch_scan_excl_u32(b.head, b.pos, total, b.scan_tmp2, s);
    uint32_t unique = 0;
    LCSX_HIP(hipMemcpyAsync(&unique, b.pos + total, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
    LCSX_HIP(hipStreamSynchronize(s));
    b.out_rc.alloc(2 * (size_t)std::max(unique, 1u));
    b.out_blk.alloc(9 * (size_t)std::max(unique, 1u));
    k_ct_reduce<<<grid_for(total, kB), kB, 0, s>>>(total, b.head, b.pos, b.row[cur], b.col[cur], b.idx[cur], b.blk,
                                                   b.out_rc.p, b.out_blk.p);
    LCSX_HIP(hipGetLastError());
    return unique;
}
void launch_contact_assemble(const ContactView& c, const VertContacts& vc, float* cgB, float* diag, uint32_t nv,
                             hipStream_t s)
{
    k_contact_assemble<<<std::min(8192u, grid_for(nv, kB / 64u)), kB, 0, s>>>(c, vc, cgB, diag, nv);
}
void launch_pcg_init(const PcgArgs& a, hipStream_t s) { k_pcg_init<<<a.seg.n_rb, kB, 0, s>>>(a); }
void launch_pcg_dir(const PcgArgs& a, const ContactView& c, const VertContacts& vc, unsigned max_chunks,
                    bool per_contact, hipStream_t s)
{
    // the contact blocks first, rounded up to a multiple of 8 (the row blocks keep their XCD mapping)
    if (!vc.ptr || !max_chunks) k_pcg_dir<0><<<a.seg.n_rb, kB, 0, s>>>(a, c, vc);
    // contacts <= slots / 4 <= 64 max_chunks
    else if (per_contact && a.seg.nscenes == 1)
        k_pcg_dir<1><<<a.seg.n_rb + ((max_chunks / 4u + 1u + 7u) & ~7u), kB, 0, s>>>(a, c, vc);
    else k_pcg_dir<2><<<a.seg.n_rb + ((max_chunks + 7u) & ~7u), kB, 0, s>>>(a, c, vc);
}
// SpMV mappings (kSpmvShapes): shape % 3 selects the blocks per pass and load form (0: three,
// unconditional; 1: three, predicated on the row's width; 2: two, unconditional); shapes 3-5 put
// the contact chunks first in the launch.
template <int LP>
static void spmv_shape_launch(int shape, dim3 g, uint32_t cf, const PcgArgs& a, const SellView& A,
                              const VertContacts& vc, hipStream_t s, hipEvent_t start, hipEvent_t stop)
{
    auto go = [&](auto kern) {
        if (start) hipExtLaunchKernelGGL(kern, g, dim3(kB), 0, s, start, stop, 0, a, A, vc, cf);
        else kern<<<g, kB, 0, s>>>(a, A, vc, cf);
    };
    switch (shape % 3)
    {
        case 1: go(k_spmv_pcg<LP, 3, false>); break;
        case 2: go(k_spmv_pcg<LP, 2, true>); break;
        default: go(k_spmv_pcg<LP, 3, true>); break;
    }
}
void launch_pcg_spmv(const PcgArgs& a, const SellView& A, const VertContacts& vc, unsigned max_chunks, int shape,
                     hipStream_t s, hipEvent_t start, hipEvent_t stop)
{
    const uint32_t nch = vc.ptr ? max_chunks : 0u;
    const uint32_t cf  = shape >= 3 && nch ? (nch + 7u) & ~7u : 0u;
    const dim3     g(4u * a.seg.n_rb + (cf ? cf : nch));
    if (A.val_p && A.bf16) spmv_shape_launch<2>(shape, g, cf, a, A, vc, s, start, stop);
    else if (A.val_p) spmv_shape_launch<1>(shape, g, cf, a, A, vc, s, start, stop);
    else spmv_shape_launch<0>(shape, g, cf, a, A, vc, s, start, stop);
}
void launch_energy(const EnergyArgs& a, unsigned contact_grid, uint32_t nscenes, hipStream_t s)
{
    k_fill_f64<<<grid_for(nscenes, kB), kB, 0, s>>>(a.out, nscenes);
    if (a.nv) k_energy_rows<<<grid_for(a.nv, kB), kB, 0, s>>>(a);
    if (a.nsp) k_energy_springs<<<grid_for(a.nsp, kB), kB, 0, s>>>(a);
    if (a.nsf) k_energy_faces<<<grid_for(a.nsf, kB), kB, 0, s>>>(a);
    if (a.nbh) k_energy_hinges<<<grid_for(a.nbh, kB), kB, 0, s>>>(a);
    if (a.nb) k_energy_bodies<<<grid_for(a.nb, kB), kB, 0, s>>>(a);
    if (a.c.count && contact_grid) k_energy_contacts<<<contact_grid, kB, 0, s>>>(a);
}
void launch_pack_fp16(uint32_t nslices, uint32_t n, const uint32_t* sl_off, uint32_t nblocks, const float* val,
                      const uint8_t* row_kind, uint32_t* val_p, int bf16, hipStream_t s)
{
    if (nblocks)
        k_pack_fp16<<<grid_for(nslices * kSellH, kB), kB, 0, s>>>(nslices, n, sl_off, nblocks, val, row_kind, val_p, bf16);
}
void launch_residual(const SegView& g, const float* b, const float* y, const float* minv, float* r, float* z,
                     float* part_rz, float* part_res, hipStream_t s)
{
    k_residual<<<g.n_rb, kB, 0, s>>>(g, b, y, minv, r, z, part_rz, part_res);
}
void launch_pcg_update(const PcgArgs& a, hipStream_t s) { k_pcg_update<<<a.seg.n_rb, kB, 0, s>>>(a); }
void launch_grid_clear(unsigned long long* w, size_t n, hipStream_t s)
{
    if (n) k_grid_clear<<<std::min(1024u, grid_for(n, kB)), kB, 0, s>>>(w, n);
}
// A workgroup takes one row block (256 rows) while one launch holds them all, otherwise two: a wait for
// more workgroups costs more than the second block's product, and a batch needs half the launches.
// Blocks per thread and row (K, four threads a row) are what fits 256 registers beside the rows'
// vectors.
GridPlan grid_plan(uint32_t n_rb_most, uint32_t n_rb, uint32_t width, uint32_t wgs)
{
    GridPlan  p;
    const int K = width <= 12u ? 3 : (width <= 16u ? 4 : (width <= 32u ? 8 : 0));
    const int U = n_rb <= wgs || K > 3 ? 2 : 4;
    if (K == 0 || n_rb == 0 || n_rb_most > wgs * (uint32_t)(U / 2)) return p;
    p.U = U;
    p.K = K;
    return p;
}
template <class Mat, class Ct, bool CT>
static void grid_go(const GridPlan& p, unsigned wgs, const PcgArgs& a, const Mat& A, const Ct& ct, const GridSync& g, uint32_t len,
                    hipStream_t s)
{
    auto go = [&](auto kern) { kern<<<wgs, kGridThreads, 0, s>>>(a, A, ct, g, len); };
    if (p.U == 4) go(k_pcg_grid<Mat, 4, 3, CT, Ct>);
    else if (p.K == 3) go(k_pcg_grid<Mat, 2, 3, CT, Ct>);
    else if (p.K == 4) go(k_pcg_grid<Mat, 2, 4, CT, Ct>);
    else go(k_pcg_grid<Mat, 2, 8, CT, Ct>);
    LCSX_HIP(hipGetLastError());
}
template <int LP>
static void grid_lp(const GridPlan& p, unsigned wgs, const PcgArgs& a, const SellView& A, const ContactView& c,
                    const VertContacts& vc, const GridSync& g, uint32_t len, hipStream_t s)
{
    const GridSell<LP> M{A, a.n};
    if (vc.ptr)
    {
        GridContacts ct;
        ct.c  = c;
        ct.vc = vc;
        grid_go<GridSell<LP>, GridContacts, true>(p, wgs, a, M, ct, g, len, s);
    }
    else
        grid_go<GridSell<LP>, NoContacts, false>(p, wgs, a, M, NoContacts{}, g, len, s);
}
void launch_pcg_grid(const GridPlan& p, unsigned wgs, const PcgArgs& a, const SellView& A, const ContactView& c,
                     const VertContacts& vc, const GridSync& g, uint32_t len, hipStream_t s)
{
    if (A.val_p && A.bf16) grid_lp<2>(p, wgs, a, A, c, vc, g, len, s);
    else if (A.val_p) grid_lp<1>(p, wgs, a, A, c, vc, g, len, s);
    else grid_lp<0>(p, wgs, a, A, c, vc, g, len, s);
}
namespace
{
constexpr int kGridDevices = 64;
struct GridDevice
{
    std::atomic<bool>     busy{false};
    std::atomic<uint32_t> cus{0};            // 0: not asked yet
    std::atomic<uint32_t> skip{0}, back{0};  // solves without a lease still to come, and after the next wait
    std::atomic<uint64_t> one{0}, unfit{0}, waited{0}, refused{0};
};
GridDevice g_grid[kGridDevices];
}  // namespace
uint32_t grid_wgs(int device)
{
    if (device < 0 || device >= kGridDevices) return 0u;
    uint32_t cus = g_grid[device].cus.load();
    if (!cus)
    {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || n <= 0) return 0u;
        cus = (uint32_t)n;
        g_grid[device].cus.store(cus);
    }
    return std::min(cus, kGridWgs);
}
bool GridLease::take(int device)
{
    if (device < 0 || device >= kGridDevices) return false;
    GridDevice& d = g_grid[device];
    uint32_t    s = d.skip.load();
    while (s && !d.skip.compare_exchange_weak(s, s - 1u)) {}
    if (s || d.busy.exchange(true))
    {
        d.refused++;
        return false;
    }
    dev = device;
    return true;
}
void GridLease::outcome(uint32_t fail, bool remember)
{
    if (dev < 0) return;
    GridDevice& d = g_grid[dev];
    if (!fail) d.one++;
    else if (fail & kGridUnfit) d.unfit++;
    else
    {
        d.waited++;
        if (!remember) return;
        const uint32_t b = std::max(d.back.load(), 1024u);
        d.skip.store(b);
        d.back.store(std::min(2u * b, 1u << 20));
    }
}
GridLease::~GridLease()
{
    if (dev >= 0) g_grid[dev].busy.store(false);
}
GridCounts grid_counts(int device)
{
    if (device < 0 || device >= kGridDevices) return GridCounts{};
    const GridDevice& d = g_grid[device];
    return GridCounts{d.one.load(), d.unfit.load(), d.waited.load(), d.refused.load()};
}
void launch_spmv(const SellView& A, const ContactView& c, const VertContacts& vc, unsigned contact_grid, const float* p,
                 float* y, uint32_t n, hipStream_t s)
{
    if (A.val_p && A.bf16) k_spmv_plain<2><<<grid_for(n, kB), kB, 0, s>>>(n, A, p, y);
    else if (A.val_p) k_spmv_plain<1><<<grid_for(n, kB), kB, 0, s>>>(n, A, p, y);
    else k_spmv_plain<0><<<grid_for(n, kB), kB, 0, s>>>(n, A, p, y);
    if (vc.ptr && vc.nslots)
    {
        k_contact_t_plain<<<contact_grid, kB, 0, s>>>(c, p, vc.tc);
        k_slots_plain<<<grid_for(vc.nslots, kB), kB, 0, s>>>(vc);
        k_fold_plain<<<grid_for(n, kB), kB, 0, s>>>(vc, n, y);
    }
}
void launch_apply_dx(uint32_t nv, const float* x_iter, const float* dx, float* x, const SceneStatus* sst,
                     float alpha_const, const SegView& g, hipStream_t s)
{
    k_apply_dx<<<grid_for(nv, kB), kB, 0, s>>>(nv, x_iter, dx, x, sst, alpha_const, g);
}
void launch_ground_ccd_maxdx(const LsArgs& a, hipStream_t s) { k_ground_ccd_maxdx<<<a.seg.n_rb, kB, 0, s>>>(a); }
void launch_ccd(const CcdArgs& a, unsigned grid, hipStream_t s)
{
    if (a.fp64)
    {
        if (a.kind == 0) k_ccd<true, 0><<<grid, kB, 0, s>>>(a);
        else k_ccd<true, 1><<<grid, kB, 0, s>>>(a);
    }
    else if (a.kind == 0) k_ccd<false, 0><<<grid, kB, 0, s>>>(a);
    else k_ccd<false, 1><<<grid, kB, 0, s>>>(a);
}
void launch_pin_delta(uint32_t nfix, const uint32_t* ids, const float* x, const float* x_tilde, SceneStatus* sst,
                      const uint32_t* vert_scene, hipStream_t s)
{
    if (nfix) k_pin_delta<<<grid_for(nfix, kB), kB, 0, s>>>(nfix, ids, x, x_tilde, sst, vert_scene);
}
void launch_reset_status(Status* st, SceneStatus* sst, uint32_t nscenes, hipStream_t s)
{
    k_reset_status<<<grid_for(nscenes, kB), kB, 0, s>>>(st, sst, nscenes);
}
void launch_reset_line_search(Status* st, SceneStatus* sst, uint32_t nscenes, hipStream_t s)
{
    k_reset_ls<<<grid_for(nscenes, kB), kB, 0, s>>>(st, sst, nscenes);
}
void launch_reset_gap(GapStatus* g, uint32_t nscenes, hipStream_t s)
{
    k_reset_gap<<<grid_for(nscenes, kB), kB, 0, s>>>(g, nscenes);
}
void launch_gap_check(const GapArgs& a, unsigned grid, hipStream_t s)
{
    if (a.kind == 2) grid = std::max(1u, std::min(grid, grid_for(a.nv, kB)));
    grid = std::min(grid, 1024u);  // four workgroups per CU: a stretch of at least a few hundred pairs
    k_gap_check<<<grid, kB, 0, s>>>(a);
}


// The narrow phase on a caller's pair list (one scene, no affine bodies): CCD's step bound and the
// DCD's contacts. `work` holds 2 + n_pairs words and one SceneStatus (16 B), device memory.
void narrow_ccd(int kind, const uint32_t* pairs, uint32_t n_pairs, const uint32_t* prims, const float* x0,
                const float* x1, const float* offset, int fp64, int budget, float* toi, uint32_t* work, hipStream_t s)
{
    SceneStatus* st = reinterpret_cast<SceneStatus*>(work);
    uint32_t*    cnt = work + 4;
    k_narrow_init<<<1, 64, 0, s>>>(cnt, n_pairs, st);
    CcdArgs c{};
    c.kind          = kind;
    c.pairs         = pairs;
    c.pair_count    = cnt;
    c.pair_capacity = n_pairs;
    c.x0            = x0;
    c.x1            = x1;
    c.faces         = prims;
    c.edges         = prims;
    c.offset        = offset;
    c.budget        = budget;
    c.fp64          = fp64;
    c.rest_list     = cnt + 2;
    c.rest_count    = cnt + 1;
    c.sst           = st;
    const unsigned grid = std::max(1u, std::min(4096u, grid_for(n_pairs, kB)));
    if (n_pairs)
    {
        c.rest = 0;
        launch_ccd(c, grid, s);
        c.rest = 1;
        launch_ccd(c, std::min(1024u, grid), s);
    }
    k_toi_out<<<1, 64, 0, s>>>(st, toi);
}

void narrow_dcd(int kind, const uint32_t* pairs, uint32_t n_pairs, const uint32_t* prims, const float* x,
                const float* area_a, const float* area_b, const float* offset, const float* dhat, float kappa,
                int quadratic, int fp64, const ContactBuf& out, uint32_t* work, hipStream_t s)
{
    k_narrow_init<<<1, 64, 0, s>>>(work, n_pairs, nullptr);
    DcdArgs a{};
    a.pairs         = pairs;
    a.pair_count    = work;
    a.pair_capacity = n_pairs;
    a.x             = x;
    a.faces         = prims;
    a.edges         = prims;
    a.area_a        = area_a;
    a.area_b        = area_b;
    a.offset        = offset;
    a.dhat          = dhat;
    a.kappa         = kappa;
    a.fp64          = fp64;
    a.quadratic     = quadratic;
    a.out           = out;
    if (n_pairs) launch_dcd(a, kind, std::max(1u, std::min(4096u, grid_for(n_pairs, kB))), s);
}

}  // namespace lcsx
