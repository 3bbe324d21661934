// The block-Jacobi PCG in one launch (device code): a whole run of iterations in one kernel whose
// workgroups keep their rows' blocks in registers and exchange vectors and partial sums through
// device memory.
//
// What bounds a launched iteration is not the matrix but the launches: three dependent kernels and
// the gaps between them. Here a workgroup owns one or two 256-row blocks. It reads their blocks,
// vectors and preconditioner once, finds the rows outside its own that its blocks' columns name (a
// hash table in LDS), and holds p of all of them in LDS, so the product reads registers and LDS only.
// A scene of a batch is solved by its own workgroups, which wait only for each other; a batch that needs
// more workgroups than CUs takes several launches. An iteration waits twice: for every 64-row chunk's p.q
// partial, and for every row block's r.z partial together with the z of the named rows. A partial is posted as one 8-byte word (value, epoch), and so
// is every entry of z: the word that carries a value also says that it is there, so nothing has to be
// ordered between the stores. Every workgroup adds the partials up itself.
//
// Bits: each sum is taken over the same partition and in the same order as by the launched kernels
// (k_pcg_dir, k_spmv_pcg, k_pcg_update; k_bsr_*): wavefront butterflies, four wavefronts per partial,
// partials strided over 256 threads. A solve therefore gives the same bits in either form, which is
// what lets the host choose per solve and start over with the launches when this kernel gives up.
//
// Memory: what workgroups exchange is stored and loaded with relaxed atomics of agent scope, which
// go to the coherent level behind the eight L2s. No fence writes back or invalidates an L2.
//
// What an iteration costs: two waits (2.5-3 us each over 180-256 workgroups, 1.2 us over 5) and about
// 1 us per row block of a workgroup. 100 iterations of the cloth tube's system (93,969 rows): 1.08 ms
// against 1.88 ms launched; of a 33 x 33 cloth's (1,089 rows, 28 iterations to its test): 157 us against
// 400 us, start-up and the host's wait included.
//
// Waiting: the launch has at most one workgroup per CU (its LDS fills most of one) and the host starts one
// such launch at a time per GPU in the process, so all workgroups become resident. Every wait is bounded
// all the same: past kPolls polls a workgroup poisons its words, sets the state's `fail` and returns, and
// so does every workgroup that reads a poisoned word.
#pragma once
#include "lcsx_common.h"
#include "lcsx_kernels.h"

namespace lcsx
{
namespace grid
{
constexpr uint32_t kPoison = 0xffffffffu;  // epoch of a word whose workgroup has given up
constexpr uint32_t kPolls  = 200000;       // polls of one wait (about 0.7 us each)
constexpr uint32_t kHash   = 8192;         // hash table entries (columns outside the own rows)
constexpr uint32_t kProbes = 256;
constexpr uint32_t kUnfit  = 2;  // Lds::bad before the loop
static_assert(kGridRows * sizeof(float4) >= kHash * 6u, "the hash table lies in the p rows' space");

struct Lds
{
    union
    {
        float4 p[kGridRows];  // p of the own rows, then of the gathered ones
        struct
        {
            uint32_t key[kHash];
            uint16_t slot[kHash];
        } h;
    };
    uint32_t halo[kGridRows];  // rows gathered from other workgroups
    float    z[3 * kGridRows];  // their z
    float    q[3 * kGridOwn];
    float    sh[4][8];
    float    red[2][4], cs[8];
    uint32_t nhalo, bad, bad_tc;  // bad: kUnfit, or 1 once a wait has failed
};
static_assert(sizeof(Lds) <= 160 * 1024, "LDS of one CU");

using Word = unsigned long long;  // value in the low half, epoch in the high half
LCSX_D void post(Word* slot, float v, uint32_t epoch)
{
    __hip_atomic_store(slot, ((Word)epoch << 32) | __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
LCSX_D Word     peek(const Word* slot) { return __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
LCSX_D uint32_t epoch_of(Word w) { return (uint32_t)(w >> 32); }
LCSX_D float    value_of(Word w) { return __uint_as_float((uint32_t)w); }
// This wavefront's earlier stores have reached the coherent level.
LCSX_D void stores_done() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); }
// 16-byte rows, stored before a word that announces them
LCSX_D void st_row(float* base, uint32_t i, f3 v)
{
    Word* d = reinterpret_cast<Word*>(base) + 2 * (size_t)i;
    __hip_atomic_store(d, ((Word)__float_as_uint(v.y) << 32) | __float_as_uint(v.x), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(d + 1, (Word)__float_as_uint(v.z), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
LCSX_D f3 ld_row(const float* base, uint32_t i)
{
    const Word* d = reinterpret_cast<const Word*>(base) + 2 * (size_t)i;
    const Word  a = peek(d), b = peek(d + 1);
    return mk(value_of(a), __uint_as_float(epoch_of(a)), value_of(b));
}
// z as words in three planes of n
LCSX_D void st_z(Word* zx, uint32_t n, uint32_t i, f3 v, uint32_t epoch)
{
    post(zx + i, v.x, epoch);
    post(zx + n + (size_t)i, v.y, epoch);
    post(zx + 2 * (size_t)n + i, v.z, epoch);
}
LCSX_D f3 wait_z(const Word* zx, uint32_t n, uint32_t i, uint32_t epoch, uint32_t& bad)
{
    for (uint32_t tries = 0;; tries++)
    {
        const Word x = peek(zx + i), y = peek(zx + n + (size_t)i), z = peek(zx + 2 * (size_t)n + i);
        if (epoch_of(x) == epoch && epoch_of(y) == epoch && epoch_of(z) == epoch)
            return mk(value_of(x), value_of(y), value_of(z));
        if (tries > kPolls || *(volatile uint32_t*)&bad != 0u)
        {
            bad = 1u;
            return mk(0.0f, 0.0f, 0.0f);
        }
    }
}

// Waits for words [0, n0) of s0, then [0, n1) of s1, of `epoch` and adds them up as the launched
// kernels do: strided over the first 256 threads, a butterfly per wavefront (the four wavefronts' sums
// go to red). Called by the first four wavefronts. L.bad is set when a word was poisoned or the wait ran
// out.
template <int kIn>  // words in flight per thread
LCSX_D void wait_sum(const Word* s0, uint32_t n0, const Word* s1, uint32_t n1, uint32_t epoch, Lds& L, float* red)
{
    const uint32_t n = n0 + n1;
    float          v = 0.0f;
    for (uint32_t i0 = threadIdx.x; i0 < n; i0 += 256u * kIn)
    {
        uint32_t tries = 0;
        while (true)
        {
            Word w[kIn];
#pragma unroll
            for (int u = 0; u < kIn; u++)
            {
                const uint32_t i = i0 + 256u * u;
                w[u]             = i < n ? peek(i < n0 ? s0 + i : s1 + (i - n0)) : (Word)epoch << 32;
            }
            bool ok = true, gone = ++tries > kPolls || *(volatile uint32_t*)&L.bad != 0u;
#pragma unroll
            for (int u = 0; u < kIn; u++)
            {
                ok   = ok && epoch_of(w[u]) == epoch;
                gone = gone || epoch_of(w[u]) == kPoison;
            }
            if (ok)
            {
#pragma unroll
                for (int u = 0; u < kIn; u++)
                    if (i0 + 256u * u < n) v = v + value_of(w[u]);
                break;
            }
            if (gone)
            {
                L.bad = 1u;
                break;
            }
        }
        if (*(volatile uint32_t*)&L.bad != 0u) break;
    }
    v = wave_sum(v);
    if (lane_id() == 0) red[threadIdx.x >> 6] = v;
    asm volatile("" ::: "memory");
}
LCSX_D float sum4(const float* r) { return ((r[0] + r[1]) + r[2]) + r[3]; }

LCSX_D uint32_t hash_of(uint32_t c) { return (c * 2654435761u) >> 19; }
static_assert(kHash == 1u << 13, "hash_of keeps 13 bits");
// false: no place within kProbes entries
LCSX_D bool hash_insert(Lds& L, uint32_t c)
{
    uint32_t h = hash_of(c);
    for (uint32_t k = 0; k < kProbes; k++)
    {
        const uint32_t old = atomicCAS(&L.h.key[h], kInvalid, c);
        if (old == kInvalid || old == c) return true;
        h = (h + 1u) & (kHash - 1u);
    }
    return false;
}
LCSX_D uint32_t hash_find(const Lds& L, uint32_t c)
{
    uint32_t h = hash_of(c);
    for (uint32_t k = 0; k < kProbes; k++)
    {
        if (L.h.key[h] == c) return L.h.slot[h];
        h = (h + 1u) & (kHash - 1u);
    }
    return 0u;
}
}  // namespace grid

// The kernel. Mat gives a row's blocks: Raw (a block as it is kept in registers), row(i) (where the
// row's blocks lie and how many, ok = false when they must not be read), col(r, k), load(r, k),
// get(raw, i, k, on), diag(i) and minv(i). U row groups of K blocks per thread: lane = 16 j + l of a
// wavefront holds blocks j, j + 4, ... of row l of its 16 rows, as in k_spmv_pcg.
template <class Mat, int U, int K, bool CT, class Contacts>
__global__ __launch_bounds__(kGridThreads) void k_pcg_grid(PcgArgs a, Mat A, Contacts ct, GridSync g, uint32_t len)
{
    using namespace grid;
    __shared__ Lds L;
    constexpr uint32_t T = kGridThreads, gpw = T / 256u;  // gpw: 64-row chunks of one row group
    constexpr uint32_t M = U * gpw, R = 64u * M;          // chunks and rows of a workgroup
    static_assert(M % 4u == 0u && M <= T / 64u && R <= kGridOwn, "whole row blocks, one wavefront per chunk");
    const uint32_t t = threadIdx.x, lane = lane_id(), wv = t >> 6, j = lane >> 4, n = a.n;
    // this workgroup's scene, its place in it, the scene's rows [.., end) and row blocks [rb0, rb0 + nrb)
    const bool     one   = g.tab == nullptr;
    const uint2    me    = one ? make_uint2(0u, blockIdx.x) : g.tab[blockIdx.x];
    const uint32_t scene = me.x, part = me.y;
    const uint32_t rb0 = one ? 0u : a.seg.sc_rb0[scene], nrb = (one ? a.seg.n_rb : a.seg.sc_rb0[scene + 1]) - rb0;
    const uint32_t own0 = (one ? 0u : a.seg.sc_v0[scene]) + part * R, end = one ? n : a.seg.sc_v0[scene + 1];
    const uint32_t b0 = rb0 + part * (M / 4u), nb = min(M / 4u, rb0 + nrb - b0), nc = 4u * nb;
    const uint32_t parts = (nrb + M / 4u - 1u) / (M / 4u);
    PcgState*      st = a.s + scene;
    if (st->converged) return;  // set by an earlier launch: every workgroup of the scene reads the same
    Word* const S_pq = g.pq + 4u * rb0;  // the scene's words
    Word* const S_rz = g.rz + rb0;
    Word* const S_ch = g.pq + 4u * a.seg.n_rb;
    const float* const rz_part = a.part_rz + rb0;
    // ---- this thread's blocks, and the rows outside its own that they name
    typename Mat::Raw W[U][K];
    uint32_t          ci[U][K];
    for (uint32_t h = t; h < kHash; h += T) L.h.key[h] = kInvalid;
    if (t == 0)
    {
        L.nhalo = 0u;
        L.bad = L.bad_tc = 0u;
    }
    __syncthreads();
    bool good = true;
#pragma unroll
    for (int u = 0; u < U; u++)
    {
        const uint32_t lc = (uint32_t)u * gpw + (wv >> 2);
        const uint32_t i  = own0 + 64u * lc + 16u * (wv & 3u) + (lane & 15u);
        const bool     in = lc < nc && i < end;
        typename Mat::Row r{};
        if (in)
        {
            r    = A.row(i);
            good = good && r.ok && r.count <= 4u * K;
        }
#pragma unroll
        for (int k = 0; k < K; k++)
        {
            ci[u][k] = kInvalid;
            W[u][k]  = typename Mat::Raw{};
            const uint32_t kk = j + 4u * (uint32_t)k;
            if (in && r.ok && kk < r.count)
            {
                const uint32_t cl = A.col(r, kk);
                if (cl < n)
                {
                    ci[u][k] = cl;
                    W[u][k]  = A.load(r, kk);
                    if (cl - own0 >= R) good = hash_insert(L, cl) && good;
                }
                else
                {
                    good = false;
                    A.bad_column();
                }
            }
        }
    }
    if (!good) L.bad = kUnfit;
    __syncthreads();
    for (uint32_t h = t; h < kHash; h += T)
        if (L.h.key[h] != kInvalid)
        {
            const uint32_t s = atomicAdd(&L.nhalo, 1u);
            if (R + s < kGridRows)
            {
                L.halo[s]   = L.h.key[h];
                L.h.slot[h] = (uint16_t)(R + s);
            }
        }
    __syncthreads();
    // more named rows than there is room for: halo holds the first ones only, and none is read
    bool           ok    = L.bad == 0u && L.nhalo <= kGridRows - R;
    const uint32_t nhalo = ok ? L.nhalo : 0u;
    if (ok)
    {
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int k = 0; k < K; k++)
                if (ci[u][k] != kInvalid)
                    ci[u][k] = ci[u][k] - own0 < R ? ci[u][k] - own0 : hash_find(L, ci[u][k]);
    }
    __syncthreads();
    // ---- this thread's row (the first nc wavefronts: one chunk each) and p of all named rows
    const uint32_t row = own0 + t;
    const bool     rv  = wv < nc && row < end;
    m3             D{}, Mi{};
    f3             xr{}, r{}, z{}, p{};
    if (rv && ok)
    {
        D  = A.diag(row);
        Mi = A.minv(a.minv, row);
        xr = ld3(a.x, row);
        r  = ld3(a.r, row);
        z  = ld3(a.z, row);
        const float4 pv = reinterpret_cast<const float4*>(a.p_old)[row];
        p  = mk(pv.x, pv.y, pv.z);
    }
    if (ok)
        for (uint32_t e = t; e < nhalo; e += T) L.p[R + e] = reinterpret_cast<const float4*>(a.p_old)[L.halo[e]];
    // r.z of the first iteration from the previous launch's row-block partials
    if (t < 256u)
    {
        float v = 0.0f;
        for (uint32_t b = t; b < nrb; b += 256u) v = v + rz_part[b];
        v = wave_sum(v);
        if (lane == 0) L.red[0][wv] = v;
    }
    __syncthreads();
    float    rz     = sum4(L.red[0]);
    uint32_t k      = a.k;
    float    rz0    = k == 0u ? rz : st->rz0;
    float    rz_old = k == 0u ? 0.0f : st->rz[(k - 1u) & 1u];
    float*   p_cur = a.p_old;
    float*   p_nxt = a.p_new;
    bool     stop  = false;
    ct.begin(a, scene, part, parts);
    for (uint32_t e = t; e < nhalo; e += T)
    {
        const f3 ze = ld3(a.z, L.halo[e]);
        st3(L.z, e, ze);
    }
    for (uint32_t it = 0; ok && it < len; it++, k++)
    {
        const uint32_t ep    = g.epoch + it;
        const bool     check = (k % a.check_every) == 0u;
        stop                 = !(rz == rz) || (check && (rz < a.abs_tol || rz <= a.rel2 * rz0));
        if (part == 0u && t == 0)
        {
            st->rz[k & 1u] = rz;
            if (k == 0u) st->rz0 = rz;
            if (stop)
            {
                st->iters     = k;
                st->nan       = (rz == rz) ? 0u : 1u;
                st->converged = 1u;
            }
        }
        if (stop) break;
        const float beta = rz_old < 1e-10f ? 0.0f : rz / rz_old;
        // ---- direction: own rows (and D p, the first term of the product), named rows
        if (rv)
        {
            p      = z + beta * p;
            L.p[t] = make_float4(p.x, p.y, p.z, 0.0f);
            st3(L.q, t, mul(D, p));
            if (CT) st_row(p_nxt, row, p);
        }
        for (uint32_t e = t; e < nhalo; e += T)
        {
            const float4 pe = L.p[R + e];
            const f3     pn = ld3(L.z, e) + beta * mk(pe.x, pe.y, pe.z);
            L.p[R + e]      = make_float4(pn.x, pn.y, pn.z, 0.0f);
        }
        __syncthreads();
        // ---- product
        A.opaque(W);
#pragma unroll
        for (int u = 0; u < U; u++)
        {
            const uint32_t lc = (uint32_t)u * gpw + (wv >> 2);
            const uint32_t lr = 64u * lc + 16u * (wv & 3u) + (lane & 15u);
            const bool     in = lc < nc && own0 + lr < end;
            f3             y  = mk(0.0f, 0.0f, 0.0f);
            if (in && j == 0u) y = ld3(L.q, lr);
#pragma unroll
            for (int kk = 0; kk < K; kk++)
            {
                const bool   on = ci[u][kk] != kInvalid;
                const float4 pc = L.p[on ? ci[u][kk] : 0u];
                const f3     yy = y + mul(A.get(W[u][kk], own0 + lr, j + 4u * (uint32_t)kk, on), mk(pc.x, pc.y, pc.z));
                y.x             = on ? yy.x : y.x;
                y.y             = on ? yy.y : y.y;
                y.z             = on ? yy.z : y.z;
            }
            y = xor_add<16>(y);
            y = xor_add<32>(y);
            float loc = 0.0f;
            if (in && j == 0u)
            {
                const float4 pi = L.p[lr];
                loc             = dot(mk(pi.x, pi.y, pi.z), y);
            }
            if (in && j < 3u) L.q[3 * lr + j] = get(y, (int)j);
            loc = wave_sum(loc);
            if (lane == 0) L.sh[u][wv] = loc;
        }
        __syncthreads();
        if (t < nc) post(S_pq + 4u * (b0 - rb0) + t, sum4(&L.sh[t / gpw][4u * (t % gpw)]), ep);
        if (CT)
        {
            ct.slots(a, g.zx, it == 0u, ep - 1u, p_cur, beta, S_ch, ep, L.cs, L.bad_tc);
            __syncthreads();
        }
        if (t < 256u) wait_sum<4 * U / 2>(S_pq, 4u * nrb, S_ch + ct.first(), ct.chunks(), ep, L, L.red[1]);
        __syncthreads();
        ok = (L.bad | L.bad_tc) == 0u;
        if (!ok) break;
        const float pq    = sum4(L.red[1]);
        const float alpha = pq < 1e-10f ? 0.0f : rz / pq;
        // ---- update
        float loc = 0.0f;
        if (rv)
        {
            f3 q = ld3(L.q, t);
            if (CT) q = ct.fold(q, row);
            if (CT) stores_done();  // this row's p, before the word below lets others read it
            xr  = xr + alpha * p;
            r   = r - alpha * q;
            z   = mul(Mi, r);
            st_z(g.zx, n, row, z, ep);
            loc = dot(r, z);
        }
        loc = wave_sum(loc);
        if (lane == 0) L.cs[wv] = loc;
        __syncthreads();
        if (t < nb) post(S_rz + (b0 - rb0) + t, sum4(&L.cs[4u * t]), ep);
        // ---- r.z of all row blocks, and the named rows' z, waited for by the other wavefronts meanwhile
        if (t < 256u) wait_sum<U / 2>(S_rz, nrb, nullptr, 0u, ep, L, L.red[0]);
        for (uint32_t e = (t + 256u) % T; e < nhalo; e += T) st3(L.z, e, wait_z(g.zx, n, L.halo[e], ep, L.bad));
        __syncthreads();
        ok = L.bad == 0u;
        if (!ok) break;
        rz_old = rz;
        rz     = sum4(L.red[0]);
        float* const sw = p_cur;
        p_cur           = p_nxt;
        p_nxt           = sw;
    }
    if (!ok)
    {
        // no workgroup may wait for this one any longer
        if (t < nc) post(S_pq + 4u * (b0 - rb0) + t, 0.0f, kPoison);
        if (t < nb) post(S_rz + (b0 - rb0) + t, 0.0f, kPoison);
        if (t == 0)
        {
            ct.poison(S_ch);
            // (unfit: known before the loop, so the LDS words are still what they were there)
            const bool unfit = L.bad == kUnfit || L.nhalo > kGridRows - R;
            __hip_atomic_fetch_or(&st->fail, unfit ? kGridUnfit : kGridWaited, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        return;
    }
    if (rv)
    {
        st3(a.x, row, xr);
        st3(a.r, row, r);
        st3(a.z, row, z);
        reinterpret_cast<float4*>(p_cur)[row] = make_float4(p.x, p.y, p.z, 0.0f);
    }
    if (!stop && len > 0u && t < nb) a.part_rz[b0 + t] = sum4(&L.cs[4u * t]);
}

// Solves without contacts.
struct NoContacts
{
    LCSX_D void     begin(const PcgArgs&, uint32_t, uint32_t, uint32_t) {}
    LCSX_D uint32_t first() const { return 0u; }
    LCSX_D uint32_t chunks() const { return 0u; }
    LCSX_D void     slots(const PcgArgs&, const grid::Word*, bool, uint32_t, const float*, float, grid::Word*, uint32_t,
                          float*, uint32_t&) const
    {
    }
    LCSX_D void poison(grid::Word*) const {}
    LCSX_D f3       fold(f3 q, uint32_t) const { return q; }
};
}  // namespace lcsx
