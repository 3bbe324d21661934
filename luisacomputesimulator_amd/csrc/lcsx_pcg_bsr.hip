// Standalone block-Jacobi PCG on a caller's block-CSR system (device pointers), the counterpart of
// ConjugateGradientSolver::device_solve (Solver/LinearSolver/precond_cg.h:38-47,
// precond_cg.cpp:626-771) for a caller that assembles its own matrix: 3x3 diagonal blocks (also the
// preconditioner, inverted per row) and off-diagonal blocks in block-CSR order.
//
// The iteration is the reference's: x0 = 0, r = b, z = M^-1 r, beta = r.z / r.z_old (0 when r.z_old
// is below 1e-10), p = z + beta p, q = A p, alpha = r.z / p.q (0 when p.q is below 1e-10),
// x += alpha p, r -= alpha q; the solve stops when r.z < abs_tol (or r.z <= rel_tol^2 r0.z0, or
// NaN), tested every check_every iterations, or after max_iters iterations. A system that fits runs in
// one launch (k_pcg_grid, lcsx_pcg_grid.h); otherwise, or where that form gives up, each iteration is
// three launches (direction, product, update), whose blocks re-reduce the previous launch's per-block
// partials in a fixed order. Both give the same bits, and results do not depend on scheduling.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

#include "../../include/lcsx.h"
#include "lcsx_common.h"
#include "lcsx_internal.h"
#include "lcsx_kernels.h"
#include "lcsx_pcg_grid.h"

namespace lcsx
{
namespace
{
constexpr int      kB       = 256;  // rows per block of the row-wise kernels
constexpr int      kProdB   = 256;  // product: 64 rows per block, 4 lanes per row
constexpr uint32_t kAlign   = 64;   // scratch regions start on 256-byte boundaries (floats)
constexpr uint32_t kNoAllocRows = 131072;  // largest system of lcsx_pcg_solve_bsr_noalloc

using BsrState = PcgState;  // scalars shared between launches

// Scratch of one solve (device pointers into one allocation).
struct BsrWork
{
    uint32_t  n, nb;  // rows, row blocks of kB rows
    float*    minv;   // 9 per row
    float*    r;      // 3 per row
    float*    z;      // 3 per row
    float*    p[2];   // 4 per row
    float*    q;      // 3 per row
    float*    part_rz;
    float*    part_pq;  // four per row block: one per product block of 64 rows
    BsrState* st;
    unsigned long long* words;  // of the one-launch form (GridSync: rz, pq, zx); cleared by the init
    uint32_t            n_words;
};

constexpr uint32_t kGridBsrRows = 2 * kGridWgs * 256;  // most rows of the one-launch form
constexpr uint32_t grid_words(uint32_t n) { return n <= kGridBsrRows ? 5u * ((n + kB - 1) / kB) + 3u * n : 0u; }

constexpr uint32_t align_up(uint32_t v) { return (v + kAlign - 1) / kAlign * kAlign; }

lcsx_status arg_error(const char* m)
{
    set_error(m);
    return LCSX_ERR_ARG;
}

// Floats of scratch a solve of n rows needs.
constexpr size_t work_floats(uint32_t n)
{
    return (size_t)align_up(9 * n) + 2 * (size_t)align_up(3 * n) + 2 * (size_t)align_up(4 * n) + align_up(3 * n) +
           align_up((n + kB - 1) / kB) + align_up(4 * ((n + kB - 1) / kB)) + align_up(sizeof(BsrState) / 4) +
           align_up(2 * grid_words(n));
}

BsrWork carve(float* base, uint32_t n)
{
    BsrWork w{};
    w.n             = n;
    w.nb            = (n + kB - 1) / kB;
    float* c        = base;
    auto   take     = [&](uint32_t k) {
        float* o = c;
        c += align_up(k);
        return o;
    };
    w.minv    = take(9 * n);
    w.r       = take(3 * n);
    w.z       = take(3 * n);
    w.p[0]    = take(4 * n);
    w.p[1]    = take(4 * n);
    w.q       = take(3 * n);
    w.part_rz = take(w.nb);
    w.part_pq = take(4 * w.nb);
    w.st      = reinterpret_cast<BsrState*>(take(sizeof(BsrState) / 4));
    w.n_words = grid_words(n);
    w.words   = reinterpret_cast<unsigned long long*>(take(2 * w.n_words));
    return w;
}

LCSX_D float bsum(float v, float* sh)
{
    v = wave_sum(v);
    if (lane_id() == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    float r = 0.0f;
    if (threadIdx.x == 0) r = ((sh[0] + sh[1]) + sh[2]) + sh[3];
    __syncthreads();
    return r;
}

// Sum of n partials in a fixed order, in every thread of the block.
LCSX_D float reduce_all(const float* __restrict__ part, uint32_t n, float* sh)
{
    __shared__ float bc;
    float            v = 0.0f;
    for (uint32_t i = threadIdx.x; i < n; i += kB) v = v + part[i];
    v = bsum(v, sh);
    if (threadIdx.x == 0) bc = v;
    __syncthreads();
    v = bc;
    __syncthreads();
    return v;
}

LCSX_D bool flag_set(const uint32_t* f)
{
    __shared__ uint32_t s;
    if (threadIdx.x == 0) s = *f;
    __syncthreads();
    const bool r = s != 0u;
    __syncthreads();
    return r;
}

LCSX_D m3 ld9(const float* __restrict__ a, size_t i)
{
    m3 m;
#pragma unroll
    for (int c = 0; c < 9; c++) m.m[c] = a[9 * i + c];
    return m;
}
LCSX_D f3 ldp(const float* p, uint32_t i)
{
    const float4 v = reinterpret_cast<const float4*>(p)[i];
    return mk(v.x, v.y, v.z);
}
LCSX_D void stp(float* p, uint32_t i, f3 v) { reinterpret_cast<float4*>(p)[i] = make_float4(v.x, v.y, v.z, 0.0f); }

// Minv = D^-1 by cofactors, r = b, z = Minv r, x = 0, p = 0, r.z partials; block 0 resets the state.
__global__ __launch_bounds__(kB) void k_bsr_init(BsrWork w, const float* __restrict__ diag, const float* __restrict__ b,
                                                 float* __restrict__ x)
{
    __shared__ float sh[4];
    const uint32_t   i   = blockIdx.x * kB + threadIdx.x;
    float            loc = 0.0f;
    for (uint32_t k = i; k < w.n_words; k += gridDim.x * kB) w.words[k] = 0ull;
    if (i < w.n)
    {
        const m3     D = ld9(diag, i);
        const float* m = D.m;
        float        c00 = m[4] * m[8] - m[5] * m[7];
        float        c01 = m[5] * m[6] - m[3] * m[8];
        float        c02 = m[3] * m[7] - m[4] * m[6];
        float        det = m[0] * c00 + m[1] * c01 + m[2] * c02;
        float        inv = 1.0f / det;
        float        Mi[9];
        Mi[0] = c00 * inv;
        Mi[1] = (m[2] * m[7] - m[1] * m[8]) * inv;
        Mi[2] = (m[1] * m[5] - m[2] * m[4]) * inv;
        Mi[3] = c01 * inv;
        Mi[4] = (m[0] * m[8] - m[2] * m[6]) * inv;
        Mi[5] = (m[2] * m[3] - m[0] * m[5]) * inv;
        Mi[6] = c02 * inv;
        Mi[7] = (m[1] * m[6] - m[0] * m[7]) * inv;
        Mi[8] = (m[0] * m[4] - m[1] * m[3]) * inv;
        m3 M;
#pragma unroll
        for (int c = 0; c < 9; c++)
        {
            w.minv[9 * (size_t)i + c] = Mi[c];
            M.m[c]                    = Mi[c];
        }
        const f3 r = ld3(b, i);
        st3(w.r, i, r);
        const f3 z = mul(M, r);
        st3(w.z, i, z);
        st3(x, i, mk(0.0f, 0.0f, 0.0f));
        stp(w.p[0], i, mk(0.0f, 0.0f, 0.0f));
        loc = dot(r, z);
    }
    const float s = bsum(loc, sh);
    if (threadIdx.x == 0)
    {
        w.part_rz[blockIdx.x] = s;
        if (blockIdx.x == 0)
        {
            w.st->rz[0] = w.st->rz[1] = w.st->rz0 = 0.0f;
            w.st->converged = w.st->iters = w.st->nan = w.st->bad_index = w.st->fail = 0u;
        }
    }
}

// Iteration k's r.z, convergence test and beta; p_new = z + beta p_old.
__global__ __launch_bounds__(kB) void k_bsr_dir(BsrWork w, uint32_t k, uint32_t check_every, float abs_tol, float rel2)
{
    __shared__ float sh[4];
    if (flag_set(&w.st->converged)) return;
    const float rz    = reduce_all(w.part_rz, w.nb, sh);
    const float rz0   = k == 0 ? rz : w.st->rz0;
    const bool  check = (k % check_every) == 0u;
    const bool  stop  = !(rz == rz) || (check && (rz < abs_tol || rz <= rel2 * rz0));
    const float rz_old = k == 0 ? 0.0f : w.st->rz[(k - 1u) & 1u];
    const float beta   = rz_old < 1e-10f ? 0.0f : rz / rz_old;
    if (blockIdx.x == 0 && threadIdx.x == 0)
    {
        w.st->rz[k & 1u] = rz;
        if (k == 0) w.st->rz0 = rz;
        if (stop)
        {
            w.st->iters     = k;
            w.st->nan       = (rz == rz) ? 0u : 1u;
            w.st->converged = 1u;
        }
    }
    if (stop) return;
    const uint32_t i = blockIdx.x * kB + threadIdx.x;
    if (i < w.n) stp(w.p[(k + 1u) & 1u], i, ld3(w.z, i) + beta * ldp(w.p[k & 1u], i));
}

// q = D p + sum_k A_k p_col(k) with 4 lanes per row (lane j takes the row's blocks j, j + 4, ...),
// p.q partial per block. A column outside [0, n) or a row range outside [0, nnz) is not read; it
// sets bad_index (reported as an argument error).
__global__ __launch_bounds__(kProdB) void k_bsr_spmv(BsrWork w, uint32_t k, const int32_t* __restrict__ row_ptr,
                                                     const int32_t* __restrict__ col, const float* __restrict__ blocks,
                                                     const float* __restrict__ diag, uint32_t nnz)
{
    __shared__ float sh[4];
    if (flag_set(&w.st->converged)) return;
    const float*   p    = w.p[(k + 1u) & 1u];
    const uint32_t lane = lane_id(), j = lane >> 4;
    const uint32_t i    = blockIdx.x * (kProdB / 4) + (threadIdx.x >> 6) * 16u + (lane & 15u);
    const bool     valid = i < w.n;
    f3             y = mk(0.0f, 0.0f, 0.0f), pi = mk(0.0f, 0.0f, 0.0f);
    if (valid)
    {
        if (j == 0u)
        {
            pi = ldp(p, i);
            y  = mul(ld9(diag, i), pi);
        }
        const int32_t b0 = row_ptr[i], b1 = row_ptr[i + 1];
        if (b0 < 0 || b1 > (int32_t)nnz || b1 < b0)
            w.st->bad_index = 1u;
        else
            for (int32_t kk = b0 + (int32_t)j; kk < b1; kk += 4)
            {
                const int32_t c = col[kk];
                if (c < 0 || c >= (int32_t)w.n)
                {
                    w.st->bad_index = 1u;
                    continue;
                }
                y = y + mul(ld9(blocks, (size_t)kk), ldp(p, (uint32_t)c));
            }
    }
    y = xor_add<32>(xor_add<16>(y));
    if (valid && j < 3u) w.q[3 * (size_t)i + j] = get(y, (int)j);
    const float s = bsum(valid && j == 0u ? dot(pi, y) : 0.0f, sh);
    if (threadIdx.x == 0) w.part_pq[blockIdx.x] = s;
}

// alpha = r.z / p.q; x += alpha p, r -= alpha q, z = Minv r, r.z partials.
__global__ __launch_bounds__(kB) void k_bsr_update(BsrWork w, uint32_t k, float* __restrict__ x)
{
    __shared__ float sh[4];
    if (flag_set(&w.st->converged)) return;
    const float    pq    = reduce_all(w.part_pq, 4 * w.nb, sh);
    const float    rz    = w.st->rz[k & 1u];
    const float    alpha = pq < 1e-10f ? 0.0f : rz / pq;
    const uint32_t i     = blockIdx.x * kB + threadIdx.x;
    float          loc   = 0.0f;
    if (i < w.n)
    {
        st3(x, i, ld3(x, i) + alpha * ldp(w.p[(k + 1u) & 1u], i));
        const f3 r = ld3(w.r, i) - alpha * ld3(w.q, i);
        st3(w.r, i, r);
        m3 M;
#pragma unroll
        for (int c = 0; c < 9; c++) M.m[c] = w.minv[9 * (size_t)i + c];
        const f3 z = mul(M, r);
        st3(w.z, i, z);
        loc = dot(r, z);
    }
    const float s = bsum(loc, sh);
    if (threadIdx.x == 0) w.part_rz[blockIdx.x] = s;
}

__global__ void k_zero_word(uint32_t* w)
{
    if (threadIdx.x == 0) *w = 0u;
}

// y = A x on a caller's block-CSR matrix (x, y: 3 floats per row), 4 lanes per row as k_bsr_spmv.
// An out-of-range column or row range is not read and sets *bad.
__global__ __launch_bounds__(kProdB) void k_bsr_apply(uint32_t n, const int32_t* __restrict__ row_ptr,
                                                      const int32_t* __restrict__ col, const float* __restrict__ blocks,
                                                      const float* __restrict__ diag, uint32_t nnz,
                                                      const float* __restrict__ x, float* __restrict__ y,
                                                      uint32_t* __restrict__ bad)
{
    const uint32_t lane = lane_id(), j = lane >> 4;
    const uint32_t i    = blockIdx.x * (kProdB / 4) + (threadIdx.x >> 6) * 16u + (lane & 15u);
    const bool     valid = i < n;
    f3             acc   = mk(0.0f, 0.0f, 0.0f);
    if (valid)
    {
        if (j == 0u) acc = mul(ld9(diag, i), ld3(x, i));
        const int32_t b0 = row_ptr[i], b1 = row_ptr[i + 1];
        if (b0 < 0 || b1 > (int32_t)nnz || b1 < b0)
            *bad = 1u;
        else
            for (int32_t kk = b0 + (int32_t)j; kk < b1; kk += 4)
            {
                const int32_t c = col[kk];
                if (c < 0 || c >= (int32_t)n)
                {
                    *bad = 1u;
                    continue;
                }
                acc = acc + mul(ld9(blocks, (size_t)kk), ld3(x, (uint32_t)c));
            }
    }
    acc = xor_add<32>(xor_add<16>(acc));
    if (valid && j < 3u) y[3 * (size_t)i + j] = get(acc, (int)j);
}

// ---------------------------------------------------------------- operator form
// The PCG around a caller's product function (lcsx_pcg_solve_op): the direction keeps p in 3-float
// rows (the function's input, updated in place: p = z + beta p), the function writes q, k_op_dot
// sums p.q per block, and the update is k_bsr_update's on those layouts. Each iteration is the
// direction, the caller's product, the dot and the update; the scalars come from the previous
// launch's per-block partials, as in the block-CSR form.
struct OpWork
{
    uint32_t  n, nb;
    float*    minv;  // 9 per row
    float*    r;     // 3 per row
    float*    z;     // 3 per row
    float*    p;     // 3 per row
    float*    q;     // 3 per row
    float*    part_rz;
    float*    part_pq;
    BsrState* st;
};
constexpr size_t op_work_floats(uint32_t n)
{
    return (size_t)align_up(9 * n) + 4 * (size_t)align_up(3 * n) + 2 * (size_t)align_up((n + kB - 1) / kB) +
           align_up(sizeof(BsrState) / 4);
}
OpWork op_carve(float* base, uint32_t n)
{
    OpWork w{};
    w.n      = n;
    w.nb     = (n + kB - 1) / kB;
    float* c = base;
    auto take = [&](uint32_t k) {
        float* o = c;
        c += align_up(k);
        return o;
    };
    w.minv    = take(9 * n);
    w.r       = take(3 * n);
    w.z       = take(3 * n);
    w.p       = take(3 * n);
    w.q       = take(3 * n);
    w.part_rz = take(w.nb);
    w.part_pq = take(w.nb);
    w.st      = reinterpret_cast<BsrState*>(take(sizeof(BsrState) / 4));
    return w;
}

__global__ __launch_bounds__(kB) void k_op_init(OpWork w, const float* __restrict__ diag, const float* __restrict__ b,
                                                float* __restrict__ x)
{
    __shared__ float sh[4];
    const uint32_t   i   = blockIdx.x * kB + threadIdx.x;
    float            loc = 0.0f;
    if (i < w.n)
    {
        const m3     D = ld9(diag, i);
        const float* m = D.m;
        float        c00 = m[4] * m[8] - m[5] * m[7];
        float        c01 = m[5] * m[6] - m[3] * m[8];
        float        c02 = m[3] * m[7] - m[4] * m[6];
        float        det = m[0] * c00 + m[1] * c01 + m[2] * c02;
        float        inv = 1.0f / det;
        m3           M;
        M.m[0] = c00 * inv;
        M.m[1] = (m[2] * m[7] - m[1] * m[8]) * inv;
        M.m[2] = (m[1] * m[5] - m[2] * m[4]) * inv;
        M.m[3] = c01 * inv;
        M.m[4] = (m[0] * m[8] - m[2] * m[6]) * inv;
        M.m[5] = (m[2] * m[3] - m[0] * m[5]) * inv;
        M.m[6] = c02 * inv;
        M.m[7] = (m[1] * m[6] - m[0] * m[7]) * inv;
        M.m[8] = (m[0] * m[4] - m[1] * m[3]) * inv;
#pragma unroll
        for (int c = 0; c < 9; c++) w.minv[9 * (size_t)i + c] = M.m[c];
        const f3 r = ld3(b, i);
        st3(w.r, i, r);
        const f3 z = mul(M, r);
        st3(w.z, i, z);
        st3(x, i, mk(0.0f, 0.0f, 0.0f));
        st3(w.p, i, mk(0.0f, 0.0f, 0.0f));
        loc = dot(r, z);
    }
    const float sum = bsum(loc, sh);
    if (threadIdx.x == 0)
    {
        w.part_rz[blockIdx.x] = sum;
        if (blockIdx.x == 0)
        {
            w.st->rz[0] = w.st->rz[1] = w.st->rz0 = 0.0f;
            w.st->converged = w.st->iters = w.st->nan = w.st->bad_index = w.st->fail = 0u;
        }
    }
}

__global__ __launch_bounds__(kB) void k_op_dir(OpWork w, uint32_t k, uint32_t check_every, float abs_tol, float rel2)
{
    __shared__ float sh[4];
    if (flag_set(&w.st->converged)) return;
    const float rz     = reduce_all(w.part_rz, w.nb, sh);
    const float rz0    = k == 0 ? rz : w.st->rz0;
    const bool  check  = (k % check_every) == 0u;
    const bool  stop   = !(rz == rz) || (check && (rz < abs_tol || rz <= rel2 * rz0));
    const float rz_old = k == 0 ? 0.0f : w.st->rz[(k - 1u) & 1u];
    const float beta   = rz_old < 1e-10f ? 0.0f : rz / rz_old;
    if (blockIdx.x == 0 && threadIdx.x == 0)
    {
        w.st->rz[k & 1u] = rz;
        if (k == 0) w.st->rz0 = rz;
        if (stop)
        {
            w.st->iters     = k;
            w.st->nan       = (rz == rz) ? 0u : 1u;
            w.st->converged = 1u;
        }
    }
    if (stop) return;
    const uint32_t i = blockIdx.x * kB + threadIdx.x;
    if (i < w.n) st3(w.p, i, ld3(w.z, i) + beta * ld3(w.p, i));
}

__global__ __launch_bounds__(kB) void k_op_dot(OpWork w)
{
    __shared__ float sh[4];
    if (flag_set(&w.st->converged)) return;
    const uint32_t i   = blockIdx.x * kB + threadIdx.x;
    const float    loc = i < w.n ? dot(ld3(w.p, i), ld3(w.q, i)) : 0.0f;
    const float    sum = bsum(loc, sh);
    if (threadIdx.x == 0) w.part_pq[blockIdx.x] = sum;
}

__global__ __launch_bounds__(kB) void k_op_update(OpWork w, uint32_t k, float* __restrict__ x)
{
    __shared__ float sh[4];
    if (flag_set(&w.st->converged)) return;
    const float    pq    = reduce_all(w.part_pq, w.nb, sh);
    const float    rz    = w.st->rz[k & 1u];
    const float    alpha = pq < 1e-10f ? 0.0f : rz / pq;
    const uint32_t i     = blockIdx.x * kB + threadIdx.x;
    float          loc   = 0.0f;
    if (i < w.n)
    {
        st3(x, i, ld3(x, i) + alpha * ld3(w.p, i));
        const f3 r = ld3(w.r, i) - alpha * ld3(w.q, i);
        st3(w.r, i, r);
        m3 M;
#pragma unroll
        for (int c = 0; c < 9; c++) M.m[c] = w.minv[9 * (size_t)i + c];
        const f3 z = mul(M, r);
        st3(w.z, i, z);
        loc = dot(r, z);
    }
    const float sum = bsum(loc, sh);
    if (threadIdx.x == 0) w.part_rz[blockIdx.x] = sum;
}

// The block-CSR matrix as k_pcg_grid reads it.
struct GridBsr
{
    const int32_t* row_ptr;
    const int32_t* cols;
    const float*   blocks;
    const float*   dg;
    BsrState*      st;
    uint32_t       nnz;
    struct Row
    {
        uint32_t b0, count;
        bool     ok;
    };
    using Raw = m3;
    LCSX_D Row row(uint32_t i) const
    {
        const int32_t r0 = row_ptr[i], r1 = row_ptr[i + 1];
        const bool    ok = r0 >= 0 && r1 <= (int32_t)nnz && r1 >= r0;
        if (!ok) bad_column();
        return Row{(uint32_t)r0, ok ? (uint32_t)(r1 - r0) : 0u, ok};
    }
    LCSX_D uint32_t col(const Row& r, uint32_t k) const { return (uint32_t)cols[r.b0 + k]; }
    LCSX_D m3       load(const Row& r, uint32_t k) const { return ld9(blocks, (size_t)r.b0 + k); }
    LCSX_D m3       get(const m3& w, uint32_t, uint32_t, bool) const { return w; }
    LCSX_D m3       diag(uint32_t i) const { return ld9(dg, i); }
    LCSX_D m3       minv(const float* P, uint32_t i) const { return ld9(P, i); }
    LCSX_D void     bad_column() const { st->bad_index = 1u; }
    template <int U, int K>
    LCSX_D void opaque(m3 (&)[U][K]) const
    {
    }
};

// The shape of the one-launch form. The widest row is not known here (the row pointers are on the device, and
// a count of them would cost every solve a wait): cloth-like matrices have rows of up to one and
// a half times the mean. A row with more blocks than the shape holds, or columns that name more rows, make the
// kernel give up before its first iteration, which costs such a solve 25-40 us (8 iterations of 1,089 rows:
// 176 us, 150 as launches at once, 65 where the rows fit; of 88,209 rows: 294, 260 and 137).
GridPlan bsr_plan(const lcsx_bsr* A, uint32_t nb, uint32_t wgs)
{
    const double mean = (double)A->nnz / A->n_rows;
    if (A->n_rows > (int)kGridBsrRows) return GridPlan{};
    return grid_plan(nb, nb, nb > wgs ? (mean <= 12.0 ? 12u : 64u) : (mean <= 12.0 ? 16u : (mean <= 24.0 ? 32u : 64u)),
                     wgs);
}
void launch_bsr_grid(const GridPlan& p, const lcsx_bsr* A, const BsrWork& w, const lcsx_pcg_options& o, float* x,
                     hipStream_t s)
{
    PcgArgs a{};
    a.n           = w.n;
    a.minv        = w.minv;
    a.x           = x;
    a.r           = w.r;
    a.z           = w.z;
    a.p_old       = w.p[0];
    a.p_new       = w.p[1];
    a.part_rz     = w.part_rz;
    a.seg.nscenes = 1u;
    a.seg.n_rb    = w.nb;
    a.s           = w.st;
    a.rel2        = o.rel_tol * o.rel_tol;
    a.abs_tol     = o.abs_tol;
    a.check_every = (uint32_t)o.check_every;
    const GridBsr  M{A->row_ptr, A->col, A->blocks, A->diag, w.st, (uint32_t)A->nnz};
    const GridSync g{w.words, w.words + w.nb, w.words + 5u * w.nb, nullptr, 2u};
    const unsigned wgs = (w.nb + p.row_blocks() - 1u) / p.row_blocks();
    auto go = [&](auto kern) { kern<<<wgs, kGridThreads, 0, s>>>(a, M, NoContacts{}, g, (uint32_t)o.max_iters); };
    if (p.U == 4) go(k_pcg_grid<GridBsr, 4, 3, false, NoContacts>);
    else if (p.K <= 4) go(k_pcg_grid<GridBsr, 2, 4, false, NoContacts>);
    else go(k_pcg_grid<GridBsr, 2, 8, false, NoContacts>);
    LCSX_HIP(hipGetLastError());
}

// The solve on scratch `base` (work_floats(n) floats, 256-byte aligned).
lcsx_status solve(const lcsx_bsr* A, const float* b, float* x, const lcsx_pcg_options& o, hipStream_t s, float* base,
                  lcsx_pcg_result* res)
{
    const BsrWork  w  = carve(base, (uint32_t)A->n_rows);
    const float    rel2 = o.rel_tol * o.rel_tol;
    GridPlan       gp;
    GridLease      lease;
    if (o.max_iters > 0)
    {
        int dev = 0;
        if (hipGetDevice(&dev) == hipSuccess) gp = bsr_plan(A, w.nb, grid_wgs(dev));
        if (gp.U && !lease.take(dev)) gp = GridPlan{};
    }
    k_bsr_init<<<w.nb, kB, 0, s>>>(w, A->diag, b, x);
    LCSX_HIP(hipGetLastError());
    BsrState h{};
    int      issued = 0;
    while (issued < o.max_iters)
    {
        const int chunk = gp.U ? o.max_iters : std::min(std::max(o.check_every, 8), o.max_iters - issued);
        if (gp.U) launch_bsr_grid(gp, A, w, o, x, s);
        for (int k = issued; !gp.U && k < issued + chunk; k++)
        {
            k_bsr_dir<<<w.nb, kB, 0, s>>>(w, (uint32_t)k, (uint32_t)o.check_every, o.abs_tol, rel2);
            k_bsr_spmv<<<4 * w.nb, kProdB, 0, s>>>(w, (uint32_t)k, A->row_ptr, A->col, A->blocks, A->diag, (uint32_t)A->nnz);
            k_bsr_update<<<w.nb, kB, 0, s>>>(w, (uint32_t)k, x);
        }
        LCSX_HIP(hipGetLastError());
        issued += chunk;
        LCSX_HIP(hipMemcpyAsync(&h, w.st, sizeof(BsrState), hipMemcpyDeviceToHost, s));
        LCSX_HIP(hipStreamSynchronize(s));
        if (h.bad_index) break;
        if (gp.U)
        {
            lease.outcome(h.fail);
            if (h.fail)
            {
                // From the start, as launches. What does not fit is found before the first update, so the vectors
                // are still the init's (unless a wait ran out: some workgroups may have ended before it).
                if (!(h.fail & kGridUnfit)) k_bsr_init<<<w.nb, kB, 0, s>>>(w, A->diag, b, x);
                gp     = GridPlan{};
                issued = 0;
                continue;
            }
        }
        if (h.converged) break;
    }
    if (h.bad_index) return arg_error("a block column or row range is outside the matrix");
    if (h.nan)
    {
        set_error("NaN/Inf in the PCG iteration");
        return LCSX_ERR_NAN;
    }
    if (res)
    {
        res->iters     = h.converged ? (int)h.iters : issued;
        res->converged = h.converged ? 1 : 0;
        res->rz0       = h.rz0;
        res->rz        = h.rz[(h.converged ? h.iters : (uint32_t)std::max(issued - 1, 0)) & 1u];
    }
    return LCSX_OK;
}

lcsx_status check_args(const lcsx_bsr* A, const float* b, float* x, const lcsx_pcg_options* o)
{
    if (!A || !b || !x || !o) return arg_error("invalid arguments");
    if (A->n_rows <= 0 || A->nnz < 0 || !A->row_ptr || !A->diag || (A->nnz > 0 && (!A->col || !A->blocks)))
        return arg_error("invalid block matrix");
    if (o->max_iters < 0 || o->check_every <= 0) return arg_error("invalid PCG options");
    return LCSX_OK;
}
}  // namespace
}  // namespace lcsx

// Scratch of lcsx_pcg_solve_bsr_noalloc: every GPU the library runs on holds one copy (about
// 17 MB, for up to kNoAllocRows rows) until the process ends. In host code `scratch` names a
// host-side stand-in, not the device array: its device address is taken per device with
// hipGetSymbolAddress and only that address is passed to kernels.
static __device__ __align__(256) float scratch[lcsx::work_floats(lcsx::kNoAllocRows)];

namespace lcsx
{
namespace
{
constexpr int kMaxDevices = 64;
std::mutex    g_scratch_mu;
float*        g_scratch[kMaxDevices] = {};

// The device address of `scratch` on the current device, looked up once per device.
lcsx_status scratch_of_current_device(float** out)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    {
        set_error("no current HIP device");
        return LCSX_ERR_HIP;
    }
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch[dev])
    {
        void*            p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
        {
            set_error(std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
            return LCSX_ERR_HIP;
        }
        g_scratch[dev] = static_cast<float*>(p);
    }
    *out = g_scratch[dev];
    return LCSX_OK;
}
}  // namespace
}  // namespace lcsx

using namespace lcsx;

extern "C" void lcsx_pcg_options_default(lcsx_pcg_options* o)
{
    if (!o) return;
    o->max_iters   = 100;
    o->check_every = 25;
    o->rel_tol     = 0.0f;
    o->abs_tol     = 1e-10f;
}

extern "C" lcsx_status lcsx_pcg_form_counts(int device, uint64_t counts[4])
{
    if (!counts || device < 0) return arg_error("invalid arguments");
    const GridCounts g = grid_counts(device);
    counts[0]          = g.one;
    counts[1]          = g.unfit;
    counts[2]          = g.waited;
    counts[3]          = g.refused;
    return LCSX_OK;
}

extern "C" lcsx_status lcsx_pcg_solve_bsr(const lcsx_bsr* A, const float* device_b, float* device_x,
                                          const lcsx_pcg_options* options, void* stream, lcsx_pcg_result* result)
{
    lcsx_pcg_options o;
    lcsx_pcg_options_default(&o);
    if (options) o = *options;
    if (lcsx_status e = check_args(A, device_b, device_x, &o)) return e;
    hipStream_t s    = (hipStream_t)stream;
    float*      base = nullptr;
    try
    {
        LCSX_HIP(hipMalloc((void**)&base, work_floats((uint32_t)A->n_rows) * sizeof(float)));
        lcsx_status st = solve(A, device_b, device_x, o, s, base, result);
        LCSX_HIP(hipStreamSynchronize(s));
        LCSX_HIP(hipFree(base));
        return st;
    }
    catch (const HipFailure&)
    {
        if (base) (void)hipFree(base);
        return LCSX_ERR_HIP;
    }
}

extern "C" lcsx_status lcsx_pcg_solve_bsr_noalloc(const lcsx_bsr* A, const float* device_b, float* device_x,
                                                  const lcsx_pcg_options* options, void* stream,
                                                  lcsx_pcg_result* result)
{
    lcsx_pcg_options o;
    lcsx_pcg_options_default(&o);
    if (options) o = *options;
    if (lcsx_status e = check_args(A, device_b, device_x, &o)) return e;
    if ((uint32_t)A->n_rows > kNoAllocRows)
        return arg_error("lcsx_pcg_solve_bsr_noalloc: more rows than its scratch holds (131072)");
    float* base = nullptr;
    if (lcsx_status e = scratch_of_current_device(&base)) return e;
    try
    {
        return solve(A, device_b, device_x, o, (hipStream_t)stream, base, result);
    }
    catch (const HipFailure&)
    {
        return LCSX_ERR_HIP;
    }
}

extern "C" lcsx_status lcsx_spmv_bsr(const lcsx_bsr* A, const float* device_x, float* device_y, void* stream)
{
    if (!A || !device_x || !device_y) return arg_error("invalid arguments");
    if (A->n_rows <= 0 || A->nnz < 0 || !A->row_ptr || !A->diag || (A->nnz > 0 && (!A->col || !A->blocks)))
        return arg_error("invalid block matrix");
    hipStream_t s   = (hipStream_t)stream;
    uint32_t*   bad = nullptr;
    try
    {
        LCSX_HIP(hipMalloc((void**)&bad, sizeof(uint32_t)));
        k_zero_word<<<1, 64, 0, s>>>(bad);
        const uint32_t n = (uint32_t)A->n_rows;
        k_bsr_apply<<<(n + kProdB / 4 - 1) / (kProdB / 4), kProdB, 0, s>>>(n, A->row_ptr, A->col, A->blocks, A->diag,
                                                                        (uint32_t)A->nnz, device_x, device_y, bad);
        LCSX_HIP(hipGetLastError());
        uint32_t h = 0;
        LCSX_HIP(hipMemcpyAsync(&h, bad, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
        LCSX_HIP(hipStreamSynchronize(s));
        LCSX_HIP(hipFree(bad));
        if (h) return arg_error("a block column or row range is outside the matrix");
        return LCSX_OK;
    }
    catch (const HipFailure&)
    {
        if (bad) (void)hipFree(bad);
        return LCSX_ERR_HIP;
    }
}

extern "C" lcsx_status lcsx_pcg_solve_op(int n_rows, const float* device_diag, lcsx_spmv_fn spmv, void* user,
                                         const float* device_b, float* device_x, const lcsx_pcg_options* options,
                                         void* stream, lcsx_pcg_result* result)
{
    lcsx_pcg_options o;
    lcsx_pcg_options_default(&o);
    if (options) o = *options;
    if (n_rows <= 0 || !device_diag || !spmv || !device_b || !device_x) return arg_error("invalid arguments");
    if (o.max_iters < 0 || o.check_every <= 0) return arg_error("invalid PCG options");
    hipStream_t s    = (hipStream_t)stream;
    float*      base = nullptr;
    try
    {
        const uint32_t n = (uint32_t)n_rows;
        LCSX_HIP(hipMalloc((void**)&base, op_work_floats(n) * sizeof(float)));
        const OpWork w    = op_carve(base, n);
        const float  rel2 = o.rel_tol * o.rel_tol;
        k_op_init<<<w.nb, kB, 0, s>>>(w, device_diag, device_b, device_x);
        LCSX_HIP(hipGetLastError());
        BsrState h{};
        int      issued = 0;
        while (issued < o.max_iters)
        {
            const int chunk = std::min(std::max(o.check_every, 8), o.max_iters - issued);
            for (int k = issued; k < issued + chunk; k++)
            {
                k_op_dir<<<w.nb, kB, 0, s>>>(w, (uint32_t)k, (uint32_t)o.check_every, o.abs_tol, rel2);
                spmv(user, w.p, w.q, s);
                k_op_dot<<<w.nb, kB, 0, s>>>(w);
                k_op_update<<<w.nb, kB, 0, s>>>(w, (uint32_t)k, device_x);
            }
            LCSX_HIP(hipGetLastError());
            issued += chunk;
            LCSX_HIP(hipMemcpyAsync(&h, w.st, sizeof(BsrState), hipMemcpyDeviceToHost, s));
            LCSX_HIP(hipStreamSynchronize(s));
            if (h.converged) break;
        }
        LCSX_HIP(hipFree(base));
        base = nullptr;
        if (h.nan)
        {
            set_error("NaN/Inf in the PCG iteration");
            return LCSX_ERR_NAN;
        }
        if (result)
        {
            result->iters     = h.converged ? (int)h.iters : issued;
            result->converged = h.converged ? 1 : 0;
            result->rz0       = h.rz0;
            result->rz        = h.rz[(h.converged ? h.iters : (uint32_t)std::max(issued - 1, 0)) & 1u];
        }
        return LCSX_OK;
    }
    catch (const HipFailure&)
    {
        if (base) (void)hipFree(base);
        return LCSX_ERR_HIP;
    }
}
