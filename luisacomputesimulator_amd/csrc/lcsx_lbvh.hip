// Linear BVH on gfx950: global AABB, Morton codes, stable LSD radix sort, Karras build,
// bottom-up refit and stack traversal with wave-aggregated pair emission.
//
// Semantics follow reference Solver/CollisionDetector/lbvh.cpp (file:line per kernel below);
// the data path is MI355X-first: the sort runs on the device (the reference sorts on the host
// and copies keys twice per tree and frame), the refit climbs subtrees of up to 1024 leaves in LDS
// instead of the whole tree with a float-flag spin protocol, and pair lists are appended with one
// atomic per staged batch.
#include <algorithm>
#include "lcsx_internal.h"
#include "lcsx_physics.h"

namespace lcsx
{

namespace
{
constexpr int kBlock     = 256;
constexpr int kSortItems = 16;  // most keys per thread and sort pass
constexpr uint32_t kTreeletLeaves = 1024;    // most leaves of a treelet
// Largest single tree whose top is not counted on the host: with the cloth meshes' 1.5 top nodes per 1024 leaves
// it has 293, a third of what k_refit_top keeps in LDS, so a tree three times as uneven still fits (a larger top
// is right all the same, one level of it at a time by one workgroup).
constexpr uint32_t kUncounted     = 200000;

LCSX_HD uint32_t expand_bits(uint32_t b)
{
    b = (b | (b << 16)) & 0x030000FFu;
    b = (b | (b << 8)) & 0x0300F00Fu;
    b = (b | (b << 4)) & 0x030C30C3u;
    return (b | (b << 2)) & 0x09249249u;
}
// lbvh.cpp:108-121
LCSX_HD uint32_t morton32(f3 p)
{
    float x = clampf(p.x * 1024.0f, 0.0f, 1023.0f);
    float y = clampf(p.y * 1024.0f, 0.0f, 1023.0f);
    float z = clampf(p.z * 1024.0f, 0.0f, 1023.0f);
    return (expand_bits((uint32_t)x) << 2) | (expand_bits((uint32_t)y) << 1) | expand_bits((uint32_t)z);
}

// Leaf centres (lbvh.cpp:449-491) and each segment's global box over its first cover leaves: the
// reference's second reduction pass is dispatched over ceil(n_verts / 256) blocks of leaves
// (lbvh.cpp:958, 968). seg_tab holds (first leaf, leaves, first inner node, cover) per segment.
// A block whose leaves share one segment reduces in LDS and issues one atomic per bound; a
// mixed block falls back to one atomic per wavefront, or per lane.
LCSX_D void box_atomics(uint32_t* gbox, uint32_t g, const float v[6])
{
    for (int k = 0; k < 3; k++) atomicMin(&gbox[6 * g + k], f2ord(v[k]));
    for (int k = 3; k < 6; k++) atomicMax(&gbox[6 * g + k], f2ord(v[k]));
}

__global__ __launch_bounds__(kBlock) void k_leaf_centers(uint32_t n, int arity, const uint32_t* __restrict__ prims,
                                                          const float* __restrict__ x, const uint32_t* __restrict__ seg_of_leaf,
                                                          const uint32_t* __restrict__ seg_tab, float4* __restrict__ center,
                                                          uint32_t* __restrict__ gbox)
{
    __shared__ uint32_t g_first;
    uint32_t l   = blockIdx.x * kBlock + threadIdx.x;
    f3       lo  = mk(3.0e38f, 3.0e38f, 3.0e38f), hi = mk(-3.0e38f, -3.0e38f, -3.0e38f);
    uint32_t g   = 0;
    bool     in  = false;
    if (threadIdx.x == 0) g_first = seg_of_leaf[blockIdx.x * kBlock];
    if (l < n)
    {
        g = seg_of_leaf[l];
        f3 c, blo, bhi;
        if (arity == 3)
        {
            f3 p0 = ld3(x, prims[3 * l]), p1 = ld3(x, prims[3 * l + 1]), p2 = ld3(x, prims[3 * l + 2]);
            c   = 0.333333f * ((p0 + p1) + p2);
            blo = vmin(p0, vmin(p1, p2));
            bhi = vmax(p0, vmax(p1, p2));
        }
        else
        {
            f3 p0 = ld3(x, prims[2 * l]), p1 = ld3(x, prims[2 * l + 1]);
            c   = 0.5f * (p0 + p1);
            blo = vmin(p0, p1);
            bhi = vmax(p0, p1);
        }
        center[l] = make_float4(c.x, c.y, c.z, 0.0f);
        if (l - seg_tab[4 * g] < seg_tab[4 * g + 3])
        {
            lo = blo;
            hi = bhi;
            in = true;
        }
    }
    __syncthreads();
    const uint32_t g0      = g_first;
    const bool     uniform = __syncthreads_and(l >= n || g == g0) != 0;
    float v[6] = {lo.x, lo.y, lo.z, hi.x, hi.y, hi.z};
    if (uniform)
    {
        for (int k = 0; k < 3; k++) v[k] = wave_min(v[k]);
        for (int k = 3; k < 6; k++) v[k] = wave_max(v[k]);
        __shared__ float sb[4][6];
        int              w = threadIdx.x >> 6;
        if (lane_id() == 0)
            for (int k = 0; k < 6; k++) sb[w][k] = v[k];
        __syncthreads();
        if (threadIdx.x < 6)
        {
            int   k = threadIdx.x;
            float r = sb[0][k];
            for (int ww = 1; ww < 4; ww++) r = k < 3 ? smin(r, sb[ww][k]) : smax(r, sb[ww][k]);
            if (blockIdx.x * kBlock - seg_tab[4 * g0] < seg_tab[4 * g0 + 3])
            {
                if (k < 3) atomicMin(&gbox[6 * g0 + k], f2ord(r));
                else atomicMax(&gbox[6 * g0 + k], f2ord(r));
            }
        }
        return;
    }
    // mixed block: wavefronts of one segment reduce first
    uint32_t gw    = __shfl(g, 0);
    bool     wuni  = __ballot(l < n && g != gw) == 0ull;
    if (wuni)
    {
        for (int k = 0; k < 3; k++) v[k] = wave_min(v[k]);
        for (int k = 3; k < 6; k++) v[k] = wave_max(v[k]);
        const bool any_in = __ballot(in) != 0ull;
        if (lane_id() == 0 && any_in) box_atomics(gbox, gw, v);
    }
    else if (in)
        box_atomics(gbox, g, v);
}

__global__ void k_init_gbox(uint32_t* gbox, uint32_t nseg)
{
    uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= 6 * nseg) return;
    gbox[i] = (i % 6) < 3 ? 0xffffffffu : 0u;
}

// fn_compute_mortons, lbvh.cpp:507-523: key = morton32 of the normalised centre, value = leaf id.
__global__ __launch_bounds__(kBlock) void k_morton(uint32_t n, const float4* __restrict__ center,
                                                    const uint32_t* __restrict__ seg_of_leaf,
                                                    const uint32_t* __restrict__ gbox, uint32_t* __restrict__ keys,
                                                    uint32_t* __restrict__ vals)
{
    uint32_t l = blockIdx.x * kBlock + threadIdx.x;
    if (l >= n) return;
    const uint32_t* G = gbox + 6 * (size_t)seg_of_leaf[l];
    f3     lo  = mk(ord2f(G[0]), ord2f(G[1]), ord2f(G[2]));
    f3     hi  = mk(ord2f(G[3]), ord2f(G[4]), ord2f(G[5]));
    f3     ext = vmax(hi - lo, mk(1e-6f, 1e-6f, 1e-6f));
    f3     inv = mk(1.0f / ext.x, 1.0f / ext.y, 1.0f / ext.z);
    float4 c4  = center[l];
    f3     c   = mk(c4.x, c4.y, c4.z) - lo;
    keys[l]    = morton32(mk(c.x * inv.x, c.y * inv.y, c.z * inv.z));
    vals[l]    = l;
}

// Everything up to the sorted leaves in one workgroup, for one tree of at most kSmallLeaves leaves:
// the centres, the global box over the first `cover` leaves, the Morton keys, four radix passes in LDS
// and the leaf records, the values of k_leaf_centers, k_morton, the sort and k_leaves. The launches
// this replaces (24, of 2-13 us each with as much again in gaps) are what a small tree's construction
// consists of: 23 us for 3,136 edges. Twice as many leaves per thread as the 8 here spill registers and
// take 175 us for 14,000 leaves, no less than the launches.
// A wavefront owns a contiguous stretch of `per` times 64 leaves, so ranking its batches of 64 in
// order against its own running digit counts keeps the sort stable without a barrier per batch.
constexpr uint32_t kSmallLeaves = 8192;
template <int kPer>
__global__ __launch_bounds__(1024) void k_build_small(uint32_t n, uint32_t ni, int arity, const uint32_t* __restrict__ prims,
                                                       const float* __restrict__ x, uint32_t cover,
                                                       uint32_t* __restrict__ gbox, uint64_t* __restrict__ morton_sorted,
                                                       uint32_t* __restrict__ sorted, uint2* __restrict__ children,
                                                       uint32_t* __restrict__ object_idx, uint32_t* __restrict__ parent,
                                                       uint32_t* __restrict__ tcount, uint32_t* __restrict__ leaf_of)
{
    constexpr uint32_t kN = 1024u * kPer;
    __shared__ uint32_t skey[kN];
    __shared__ uint16_t sval[kN];
    __shared__ uint32_t cnt[16][256];
    __shared__ uint32_t wsum[16];
    __shared__ float    sb[16][6];
    const uint32_t t = threadIdx.x, w = t >> 6, lane = lane_id();
    const uint32_t per = (n + 1023u) / 1024u, base = w * 64u * per;  // this wavefront's leaves
    uint32_t       key[kPer];
    uint16_t       val[kPer];
    float          v[6] = {3.0e38f, 3.0e38f, 3.0e38f, -3.0e38f, -3.0e38f, -3.0e38f};
    if (t < 2u) tcount[t] = 0u;
    for (uint32_t i = 0; i < per; i++)
    {
        const uint32_t l = base + 64u * i + lane;
        if (l >= min(n, cover)) continue;
        f3 p0 = ld3(x, prims[(uint32_t)arity * l]), p1 = ld3(x, prims[(uint32_t)arity * l + 1]);
        f3 blo = vmin(p0, p1), bhi = vmax(p0, p1);
        if (arity == 3)
        {
            f3 p2 = ld3(x, prims[3 * l + 2]);
            blo   = vmin(p0, vmin(p1, p2));
            bhi   = vmax(p0, vmax(p1, p2));
        }
        v[0] = fminf(v[0], blo.x);
        v[1] = fminf(v[1], blo.y);
        v[2] = fminf(v[2], blo.z);
        v[3] = fmaxf(v[3], bhi.x);
        v[4] = fmaxf(v[4], bhi.y);
        v[5] = fmaxf(v[5], bhi.z);
    }
    for (int k = 0; k < 3; k++) v[k] = wave_min(v[k]);
    for (int k = 3; k < 6; k++) v[k] = wave_max(v[k]);
    if (lane == 0)
        for (int k = 0; k < 6; k++) sb[w][k] = v[k];
    __syncthreads();
    for (int ww = 0; ww < 16; ww++)
        for (int k = 0; k < 6; k++) v[k] = k < 3 ? smin(v[k], sb[ww][k]) : smax(v[k], sb[ww][k]);
    if (t < 6u)
    {
        float r = sb[0][t];
        for (int ww = 1; ww < 16; ww++) r = t < 3u ? smin(r, sb[ww][t]) : smax(r, sb[ww][t]);
        gbox[t] = f2ord(r);
    }
    const f3 lo = mk(v[0], v[1], v[2]), ext = vmax(mk(v[3], v[4], v[5]) - lo, mk(1e-6f, 1e-6f, 1e-6f));
    const f3 inv = mk(1.0f / ext.x, 1.0f / ext.y, 1.0f / ext.z);
#pragma unroll
    for (int i = 0; i < kPer; i++)
    {
        const uint32_t l = base + 64u * (uint32_t)i + lane;
        key[i]           = 0u;
        val[i]           = (uint16_t)l;
        if ((uint32_t)i < per && l < n)
        {
            f3 p0 = ld3(x, prims[(uint32_t)arity * l]), p1 = ld3(x, prims[(uint32_t)arity * l + 1]), cen = 0.5f * (p0 + p1);
            if (arity == 3) cen = 0.333333f * ((p0 + p1) + ld3(x, prims[3 * l + 2]));
            const f3 c = cen - lo;
            key[i]     = morton32(mk(c.x * inv.x, c.y * inv.y, c.z * inv.z));
        }
    }
    for (int shift = 0; shift < 32; shift += 8)
    {
        for (uint32_t d = lane; d < 256u; d += 64u) cnt[w][d] = 0u;
        uint32_t off[kPer];
#pragma unroll
        for (int i = 0; i < kPer; i++)
        {
            off[i] = 0u;
            if ((uint32_t)i >= per) continue;  // the same for the whole workgroup
            const bool     valid = base + 64u * (uint32_t)i + lane < n;
            const uint32_t d     = (key[i] >> shift) & 255u;
            uint64_t       peers = __ballot(valid);
            for (int b = 0; b < 8; b++)
            {
                const bool     bit = (d >> b) & 1u;
                const uint64_t bal = __ballot(bit);
                peers &= bit ? bal : ~bal;
            }
            const uint32_t rank = (uint32_t)__popcll(peers & lanemask_lt());
            if (valid)
            {
                const uint32_t c = cnt[w][d];
                off[i]           = c + rank;
                __builtin_amdgcn_wave_barrier();
                if (rank == 0u) cnt[w][d] = c + (uint32_t)__popcll(peers);
            }
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();
        // exclusive scan of the counts, digit by digit and wavefront by wavefront: four per thread
        const uint32_t d = t >> 2, q = (t & 3u) * 4u;
        uint32_t       c4[4], s = 0u;
        for (int k = 0; k < 4; k++)
        {
            c4[k] = cnt[q + k][d];
            s += c4[k];
        }
        uint32_t inc = s;
        for (int o = 1; o < 64; o <<= 1)
        {
            const uint32_t u = __shfl_up(inc, o);
            if ((int)lane >= o) inc += u;
        }
        if (lane == 63u) wsum[w] = inc;
        __syncthreads();
        uint32_t run = inc - s;
        for (uint32_t ww = 0; ww < w; ww++) run += wsum[ww];
        for (int k = 0; k < 4; k++)
        {
            cnt[q + k][d] = run;
            run += c4[k];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kPer; i++)
            if ((uint32_t)i < per && base + 64u * (uint32_t)i + lane < n)
            {
                const uint32_t pos = cnt[w][(key[i] >> shift) & 255u] + off[i];
                skey[pos]          = key[i];
                sval[pos]          = val[i];
            }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kPer; i++)
        {
            const uint32_t l = base + 64u * (uint32_t)i + lane;
            if ((uint32_t)i < per && l < n)
            {
                key[i] = skey[l];
                val[i] = sval[l];
            }
        }
    }
#pragma unroll
    for (int i = 0; i < kPer; i++)
    {
        const uint32_t l = base + 64u * (uint32_t)i + lane;
        if ((uint32_t)i < per && l < n)
        {
            const uint32_t o   = val[i];
            sorted[l]          = o;
            morton_sorted[l]   = ((uint64_t)key[i] << 32) | (uint64_t)o;
            children[ni + l]   = make_uint2(o, o);
            object_idx[ni + l] = o;
            leaf_of[o]         = l;
            if (n == 1u) parent[ni + l] = kInvalid;
        }
    }
}

// ---------------------------------------------------------------- stable LSD radix sort
// Keys per thread of a pass over n keys: a tile's rounds are serial, so few keys want small tiles
// (187,088 leaves: 17 us a scatter with 16 keys per thread in 46 workgroups, 10 us with 8 in 92), as
// long as one workgroup can still scan the tiles' counts.
constexpr uint32_t kSort4 = 65536, kSort8 = 294912;  // most keys with 4 and with 8 per thread
int sort_items(uint32_t n) { return n <= kSort4 ? 4 : (n <= kSort8 ? 8 : kSortItems); }

// Histogram of the digit (dig >> shift) & 255 per tile.
template <int kItems>
__global__ __launch_bounds__(kBlock) void k_radix_hist(const uint32_t* __restrict__ keys, uint32_t n, int shift,
                                                        uint32_t* __restrict__ hist, uint32_t nblocks)
{
    __shared__ uint32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    uint32_t base = blockIdx.x * (kBlock * kItems);
#pragma unroll
    for (int i = 0; i < kItems; i++)
    {
        uint32_t idx = base + i * kBlock + threadIdx.x;
        if (idx < n) atomicAdd(&h[(keys[idx] >> shift) & 255u], 1u);
    }
    __syncthreads();
    hist[threadIdx.x * nblocks + blockIdx.x] = h[threadIdx.x];
}

// Stable scatter by the digit of dig (kin, or the segment keys hin): kin, vin and, when present,
// hin move together.
template <int kItems>
__global__ __launch_bounds__(kBlock) void k_radix_scatter(const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
                                                           uint32_t* __restrict__ kout, uint32_t* __restrict__ vout,
                                                           const uint32_t* __restrict__ hin, uint32_t* __restrict__ hout,
                                                           const uint32_t* __restrict__ dig,
                                                           uint32_t n, int shift, const uint32_t* __restrict__ hist,
                                                           uint32_t nblocks)
{
    __shared__ uint32_t s_base[256];
    __shared__ uint32_t s_cnt[4][256];
    const uint32_t      t = threadIdx.x, w = t >> 6, lane = t & 63;
    s_base[t]              = hist[t * nblocks + blockIdx.x];
    const uint32_t base    = blockIdx.x * (kBlock * kItems);
    uint32_t       key[kItems], dg[kItems];
#pragma unroll
    for (int i = 0; i < kItems; i++)
    {
        const uint32_t idx = base + i * kBlock + t;
        key[i]             = idx < n ? kin[idx] : 0u;
        dg[i]              = idx < n ? dig[idx] : 0u;
    }
#pragma unroll
    for (int i = 0; i < kItems; i++)
    {
        for (int k = 0; k < 4; k++) s_cnt[w][lane + 64 * k] = 0;
        __syncthreads();
        uint32_t idx   = base + i * kBlock + t;
        bool     valid = idx < n;
        uint32_t d     = (dg[i] >> shift) & 255u;
        uint64_t peers = __ballot(valid);
        for (int b = 0; b < 8; b++)
        {
            bool     bit = (d >> b) & 1u;
            uint64_t bal = __ballot(bit);
            peers &= bit ? bal : ~bal;
        }
        uint32_t rank = (uint32_t)__popcll(peers & lanemask_lt());
        if (valid && rank == 0) s_cnt[w][d] = (uint32_t)__popcll(peers);
        __syncthreads();
        if (valid)
        {
            uint32_t off = s_base[d] + rank;
            for (uint32_t ww = 0; ww < w; ww++) off += s_cnt[ww][d];
            kout[off] = key[i];
            vout[off] = vin[idx];
            if (hin) hout[off] = hin[idx];
        }
        __syncthreads();
        s_base[t] += s_cnt[0][t] + s_cnt[1][t] + s_cnt[2][t] + s_cnt[3][t];
        __syncthreads();
    }
}

// One pass: the tiles' digit counts, their scan, the scatter.
void sort_pass(uint32_t n, int shift, const uint32_t* dig, const uint32_t* kin, const uint32_t* vin, uint32_t* kout,
               uint32_t* vout, const uint32_t* hin, uint32_t* hout, uint32_t* hist, uint32_t* tmp, hipStream_t s)
{
    const int      items = sort_items(n);
    const uint32_t nb    = (n + kBlock * items - 1) / (kBlock * items);
    auto           go    = [&](auto hk, auto sk) {
        hk<<<nb, kBlock, 0, s>>>(dig, n, shift, hist, nb);
        launch_scan_excl_u32(hist, hist, 256 * nb, tmp, s);
        sk<<<nb, kBlock, 0, s>>>(kin, vin, kout, vout, hin, hout, dig, n, shift, hist, nb);
    };
    if (items == 4) go(k_radix_hist<4>, k_radix_scatter<4>);
    else if (items == 8) go(k_radix_hist<8>, k_radix_scatter<8>);
    else go(k_radix_hist<kSortItems>, k_radix_scatter<kSortItems>);
}

// fn_apply_sorted, lbvh.cpp:525-539 (+ the 64-bit keys the build reads: Morton key and the leaf's
// index within its segment, as in a tree built over that segment alone)
__global__ __launch_bounds__(kBlock) void k_leaves(uint32_t n, uint32_t ni, const uint32_t* __restrict__ skeys,
                                                    const uint32_t* __restrict__ svals,
                                                    const uint32_t* __restrict__ seg_of_leaf,
                                                    const uint32_t* __restrict__ seg_tab, uint64_t* __restrict__ morton_sorted,
                                                    uint2* __restrict__ children, uint32_t* __restrict__ object_idx,
                                                    uint32_t* __restrict__ parent, uint32_t* __restrict__ leaf_of)
{
    uint32_t l = blockIdx.x * kBlock + threadIdx.x;
    if (l >= n) return;
    uint32_t o       = svals[l];
    uint32_t g       = seg_of_leaf[o];
    morton_sorted[l] = ((uint64_t)skeys[l] << 32) | (uint64_t)(o - seg_tab[4 * g]);
    children[ni + l] = make_uint2(o, o);
    object_idx[ni + l] = o;
    leaf_of[o]         = l;
    if (seg_tab[4 * g + 1] == 1u) parent[ni + l] = kInvalid;  // a one-leaf segment: the leaf is its root
}

__global__ __launch_bounds__(kBlock) void k_seg_keys(uint32_t n, const uint32_t* __restrict__ vals,
                                                      const uint32_t* __restrict__ seg_of_leaf, uint32_t* __restrict__ khi)
{
    uint32_t l = blockIdx.x * kBlock + threadIdx.x;
    if (l < n) khi[l] = seg_of_leaf[vals[l]];
}

LCSX_D int clz64(uint64_t v) { return v == 0 ? 64 : __clzll((long long)v); }

// fn_build_inner_nodes with determineRange / findSplit, lbvh.cpp:204-291, 541-596, on the keys
// of the inner node's segment: local leaf j is sorted position L + j (node ni + L + j), local
// inner node j is node ib + j, and the segment's local node 0 is its root.
__global__ __launch_bounds__(kBlock) void k_karras(uint32_t ni_, const uint64_t* __restrict__ mg,
                                                    const uint32_t* __restrict__ inner_seg,
                                                    const uint32_t* __restrict__ seg_tab, uint32_t* __restrict__ parent,
                                                    uint2* __restrict__ children, uint32_t* __restrict__ object_idx,
                                                    uint32_t* __restrict__ tsize, uint32_t* __restrict__ tfirst,
                                                    uint32_t* __restrict__ tleaf)
{
    int gid = blockIdx.x * kBlock + threadIdx.x;
    if (gid >= (int)ni_) return;
    const uint32_t  g   = inner_seg[gid];
    const int       L   = (int)seg_tab[4 * g], N = (int)seg_tab[4 * g + 1], ib = (int)seg_tab[4 * g + 2];
    const int       GI  = (int)ni_;
    const uint64_t* m   = mg + L;
    const int       nid = gid - ib;
    const int       ni  = N - 1;
    auto cp = [&](uint64_t mi, int j) -> int { return (j >= 0 && j < N) ? clz64(mi ^ m[j]) : -1; };
    int  i = 0, j = ni;
    if (nid != 0)
    {
        i            = nid;
        uint64_t mi  = m[i];
        int      cl  = clz64(mi ^ m[i - 1]);
        int      cr  = clz64(mi ^ m[i + 1]);
        int      d   = cl < cr ? 1 : -1;
        int      cpm = cl < cr ? cl : cr;
        int      lmax = 2;
        while (cp(mi, i + lmax * d) > cpm) lmax <<= 1;
        int l = 0;
        for (int t = lmax >> 1; t >= 1; t >>= 1)
            if (cp(mi, i + (l + t) * d) > cpm) l += t;
        j = i + l * d;
    }
    int      a = i < j ? i : j, b = i < j ? j : i;
    uint64_t ma = m[a], mb = m[b];
    int      split;
    if (ma == mb)
        split = (a + b) >> 1;
    else
    {
        int cpn = clz64(ma ^ mb);
        int t   = b - a;
        split   = a;
        while (true)
        {
            t      = (t + 1) >> 1;
            int ns = split + t;
            if (ns < b && clz64(ma ^ m[ns]) > cpn) split = ns;
            if (!(t > 1)) break;
        }
    }
    int cl_ = (a == split) ? GI + L + split : ib + split;
    int cr_ = (b == split + 1) ? GI + L + split + 1 : ib + split + 1;
    if (cr_ >= GI)  // a leaf child comes first (lbvh.cpp:579-584)
    {
        int tmp = cl_;
        cl_     = cr_;
        cr_     = tmp;
    }
    parent[cl_]     = (uint32_t)gid;
    parent[cr_]     = (uint32_t)gid;
    children[gid]   = make_uint2((uint32_t)cl_, (uint32_t)cr_);
    object_idx[gid] = kInvalid;
    if (nid == 0) parent[gid] = kInvalid;
    // the subtree over leaves [a, b] holds the inner nodes [a, b - 1] when this node is its left
    // end (i = a), else [a + 1, b]
    tsize[gid]  = (uint32_t)(b - a + 1);
    tfirst[gid] = (uint32_t)(ib + (i == a ? a : a + 1));
    tleaf[gid]  = (uint32_t)(L + a);  // its first leaf in sorted order
}

// Treelet roots: inner nodes of at most `limit` leaves whose parent has more (or is none), and the
// inner nodes above them ("top"), both listed in any order, one atomic per wavefront. count[0]:
// treelet roots, count[1]: top nodes (zero before the launch).
__global__ __launch_bounds__(kBlock) void k_treelet_mark(uint32_t ni, const uint32_t* __restrict__ parent,
                                                          const uint32_t* __restrict__ tsize, uint32_t limit,
                                                          uint32_t* count, uint32_t* __restrict__ troots,
                                                          uint32_t* __restrict__ top)
{
    const uint32_t i      = blockIdx.x * kBlock + threadIdx.x;
    bool           is_top = false, is_root = false;
    if (i < ni)
    {
        is_top = tsize[i] > limit;
        if (!is_top)
        {
            const uint32_t p = parent[i];
            is_root          = p == kInvalid || tsize[p] > limit;
        }
    }
    const uint32_t a = wave_append(count, is_root), b = wave_append(count + 1, is_top);
    if (is_root) troots[a] = i;
    if (is_top) top[b] = i;
}

// The top nodes sorted by depth (their ancestors are top nodes; order within a level is free) with
// the levels' offsets and every top node's place (top_idx), one workgroup. A depth is below 64: a
// node's common prefix of the distinct 64-bit keys is longer than its parent's.
constexpr uint32_t kMaxLevels = 64;
__global__ __launch_bounds__(1024) void k_top_sort(const uint32_t* __restrict__ count, const uint32_t* __restrict__ parent,
                                                    const uint32_t* __restrict__ top, uint32_t* __restrict__ depth,
                                                    uint32_t* __restrict__ top_order, uint32_t* __restrict__ top_idx,
                                                    uint32_t* __restrict__ level_ptr)
{
    __shared__ uint32_t cnt[kMaxLevels], at[kMaxLevels];
    const uint32_t      T = count[1];
    if (threadIdx.x < kMaxLevels) cnt[threadIdx.x] = 0u;
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < T; k += 1024u)
    {
        uint32_t d = 0u;
        for (uint32_t q = parent[top[k]]; q != kInvalid && d < kMaxLevels - 1u; q = parent[q]) d++;
        depth[k] = d;
        atomicAdd(&cnt[d], 1u);
    }
    __syncthreads();
    if (threadIdx.x == 0)
    {
        uint32_t run = 0u;
        for (uint32_t h = 0; h < kMaxLevels; h++)
        {
            level_ptr[h] = at[h] = run;
            run += cnt[h];
        }
        level_ptr[kMaxLevels] = run;
    }
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < T; k += 1024u)
    {
        const uint32_t pos = atomicAdd(&at[depth[k]], 1u), p = top[k];
        top_order[pos] = p;
        top_idx[p]     = pos;
    }
}

__global__ void k_fill_u32(uint32_t* a, uint32_t n, uint32_t v)
{
    uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) a[i] = v;
}

// ---------------------------------------------------------------- refit
// Cross-workgroup hand-off inside one kernel needs device-scope fences, which on a multi-XCD part
// write back and invalidate L2. The refit therefore runs in steps ordered by kernel boundaries: the
// leaf boxes, the treelets (one workgroup each, climbing in LDS) and the nodes above them.

// per top node: its children, and which of them are top nodes at which place
__global__ __launch_bounds__(kBlock) void k_top_children(uint32_t ni, const uint32_t* __restrict__ top_order,
                                                          const uint32_t* __restrict__ top_count,
                                                          const uint2* __restrict__ children,
                                                          const uint32_t* __restrict__ tsize, uint32_t limit,
                                                          const uint32_t* __restrict__ top_idx, uint4* __restrict__ top_child)
{
    const uint32_t T = *top_count;
    for (uint32_t k = blockIdx.x * kBlock + threadIdx.x; k < T; k += gridDim.x * kBlock)
    {
        const uint2 c  = children[top_order[k]];
        const bool  ta = c.x < ni && tsize[c.x] > limit, tb = c.y < ni && tsize[c.y] > limit;
        top_child[k]   = make_uint4(c.x | (ta ? 0x80000000u : 0u), c.y | (tb ? 0x80000000u : 0u), ta ? top_idx[c.x] : 0u,
                                    tb ? top_idx[c.y] : 0u);
    }
}

// update_*_leave_aabb, lbvh.cpp:636-683: leaf box = AABB(x0 and x1 of the element) +- pad[v0]
LCSX_D NodeBox leaf_box(uint32_t l, int arity, const uint32_t* __restrict__ prims, const uint32_t* __restrict__ sorted_to_orig,
                        const float* __restrict__ x0, const float* __restrict__ x1, const float* __restrict__ pad)
{
    uint32_t o = sorted_to_orig[l];
    f3       lo, hi;
    float    th;
    if (arity == 3)
    {
        uint32_t a = prims[3 * o], b = prims[3 * o + 1], c = prims[3 * o + 2];
        f3       s0 = ld3(x0, a), s1 = ld3(x0, b), s2 = ld3(x0, c);
        f3       e0 = ld3(x1, a), e1 = ld3(x1, b), e2 = ld3(x1, c);
        lo = vmin(vmin(s0, vmin(s1, s2)), vmin(e0, vmin(e1, e2)));
        hi = vmax(vmax(s0, vmax(s1, s2)), vmax(e0, vmax(e1, e2)));
        th = pad[a];
    }
    else
    {
        uint32_t a = prims[2 * o], b = prims[2 * o + 1];
        f3       s0 = ld3(x0, a), s1 = ld3(x0, b), e0 = ld3(x1, a), e1 = ld3(x1, b);
        lo = vmin(vmin(s0, s1), vmin(e0, e1));
        hi = vmax(vmax(s0, s1), vmax(e0, e1));
        th = pad[a];
    }
    lo = lo - mk(th, th, th);
    hi = hi + mk(th, th, th);
    return NodeBox{make_float4(lo.x, lo.y, lo.z, 0.0f), make_float4(hi.x, hi.y, hi.z, 0.0f)};
}

// fn_refit_tree_aabb, lbvh.cpp:702-754, for inner node p whose children are final: its box, and
// its packed record (child boxes, child codes, and under each child the largest element id, or
// with sorted_keys the largest sorted leaf index, i.e. the end of its leaf range).
// An unused slot of a 4-wide record: a box that overlaps nothing, a leaf code, key 0.
LCSX_D void empty_slot(float4* Q)
{
    const float inf = __int_as_float(0x7f800000);
    Q[0]            = make_float4(inf, inf, inf, __uint_as_float(0x80000000u));
    Q[1]            = make_float4(-inf, -inf, -inf, 0.0f);
}

// ... and, in packed4, the 4-wide record of p: the slots of its two children's records (a leaf
// child: the leaf and an empty slot), so a traversal step tests p's grandchildren with one 128 B
// load. A grandchild box lies inside its parent's box, so every grandchild that overlaps a query
// sits under a child that overlaps it: the leaves found are those of the binary traversal.
LCSX_D void inner_box(uint32_t p, uint32_t ni, const uint2* __restrict__ children, NodeBox* nodes, float4* packed,
                      float4* packed4, int sorted_keys)
{
    uint2   c = children[p];
    NodeBox A = nodes[c.x], B = nodes[c.y];
    NodeBox U;
    U.lo     = make_float4(smin(A.lo.x, B.lo.x), smin(A.lo.y, B.lo.y), smin(A.lo.z, B.lo.z), 0.0f);
    U.hi     = make_float4(smax(A.hi.x, B.hi.x), smax(A.hi.y, B.hi.y), smax(A.hi.z, B.hi.z), 0.0f);
    nodes[p] = U;
    uint32_t ca, cb, ma, mb;
    if (c.x >= ni)
    {
        ma = children[c.x].x;
        ca = 0x80000000u | ma;
        if (sorted_keys) ma = c.x - ni;
    }
    else
    {
        ca              = c.x;
        const float4* C = packed + 4 * (size_t)c.x;
        ma              = max(__float_as_uint(C[1].w), __float_as_uint(C[3].w));
    }
    if (c.y >= ni)
    {
        mb = children[c.y].x;
        cb = 0x80000000u | mb;
        if (sorted_keys) mb = c.y - ni;
    }
    else
    {
        cb              = c.y;
        const float4* C = packed + 4 * (size_t)c.y;
        mb              = max(__float_as_uint(C[1].w), __float_as_uint(C[3].w));
    }
    float4* P = packed + 4 * (size_t)p;
    const float4 pa0 = make_float4(A.lo.x, A.lo.y, A.lo.z, __uint_as_float(ca));
    const float4 pa1 = make_float4(A.hi.x, A.hi.y, A.hi.z, __uint_as_float(ma));
    const float4 pb0 = make_float4(B.lo.x, B.lo.y, B.lo.z, __uint_as_float(cb));
    const float4 pb1 = make_float4(B.hi.x, B.hi.y, B.hi.z, __uint_as_float(mb));
    P[0]      = pa0;
    P[1]      = pa1;
    P[2]      = pb0;
    P[3]      = pb1;
    if (!packed4) return;
    float4* Q = packed4 + 8 * (size_t)p;
    if (c.x < ni)
    {
        const float4* C = packed + 4 * (size_t)c.x;
        Q[0] = C[0];
        Q[1] = C[1];
        Q[2] = C[2];
        Q[3] = C[3];
    }
    else
    {
        Q[0] = pa0;
        Q[1] = pa1;
        empty_slot(Q + 2);
    }
    if (c.y < ni)
    {
        const float4* C = packed + 4 * (size_t)c.y;
        Q[4] = C[0];
        Q[5] = C[1];
        Q[6] = C[2];
        Q[7] = C[3];
    }
    else
    {
        Q[4] = pb0;
        Q[5] = pb1;
        empty_slot(Q + 6);
    }
}

__global__ __launch_bounds__(kBlock) void k_refit_leaves(uint32_t n, uint32_t ni, int arity, const uint32_t* __restrict__ prims,
                                                          const uint32_t* __restrict__ sorted_to_orig,
                                                          const float* __restrict__ x0, const float* __restrict__ x1,
                                                          const float* __restrict__ pad, NodeBox* __restrict__ nodes)
{
    uint32_t l = blockIdx.x * kBlock + threadIdx.x;
    if (l >= n) return;
    nodes[ni + l] = leaf_box(l, arity, prims, sorted_to_orig, x0, x1, pad);
}


// The top nodes of one level, one thread each (forests with more top nodes than k_refit_top's
// LDS table: one launch per level, deepest first).
__global__ __launch_bounds__(kBlock) void k_refit_range(const uint32_t* __restrict__ order, uint32_t cnt, uint32_t ni,
                                                         const uint2* __restrict__ children, NodeBox* nodes,
                                                         float4* packed, float4* packed4, int sorted_keys)
{
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k < cnt) inner_box(order[k], ni, children, nodes, packed, packed4, sorted_keys);
}

// The top nodes with their children's slots held in LDS (one thread per top node): the slots of
// children outside the top (treelet roots and leaves, final after the treelet kernel) are read
// once, each level reads its top children's slots from LDS, and the node boxes and the binary and
// four-wide records are written at the end; the same records as inner_box, level by level. More
// top nodes than kTopLds: inner_box level by level over global memory.
constexpr uint32_t kTopLds = 896;
__global__ __launch_bounds__(1024) void k_refit_top(const uint32_t* __restrict__ order,
                                                     const uint32_t* __restrict__ level_ptr, uint32_t h1, uint32_t ni,
                                                     const uint4* __restrict__ top_child,
                                                     const uint2* __restrict__ children, NodeBox* nodes,
                                                     float4* packed, float4* packed4, int sorted_keys)
{
    __shared__ float4   sl[kTopLds][4];  // per top node: (lo, code) and (hi, key) of each child
    __shared__ uint32_t lvp[kMaxLevels + 2];
    const uint32_t      T = level_ptr[h1 + 1];
    if (T == 0u) return;
    if (T > kTopLds)
    {
        for (int h = (int)h1; h >= 0; h--)
        {
            for (uint32_t k = level_ptr[h] + threadIdx.x; k < level_ptr[h + 1]; k += 1024u)
                inner_box(order[k], ni, children, nodes, packed, packed4, sorted_keys);
            __threadfence_block();
            __syncthreads();
        }
        return;
    }
    for (uint32_t h = threadIdx.x; h <= h1 + 1u; h += 1024u) lvp[h] = level_ptr[h];
    const uint32_t k  = threadIdx.x;
    const bool     on = k < T;
    uint32_t       p  = 0u;
    uint4          tc = make_uint4(0u, 0u, 0u, 0u);
    if (on)
    {
        p  = order[k];
        tc = top_child[k];
        // top nodes below these levels (a larger top): refit before, read as what lies outside
        if (tc.z >= T) tc.x &= 0x7fffffffu;
        if (tc.w >= T) tc.y &= 0x7fffffffu;
        // the slot of a child outside the top
        auto outside = [&](uint32_t c, int side) {
            const NodeBox B = nodes[c];
            uint32_t      code, key;
            if (c < ni)
            {
                const float4* C = packed + 4 * (size_t)c;
                code            = c;
                key             = max(__float_as_uint(C[1].w), __float_as_uint(C[3].w));
            }
            else
            {
                const uint32_t el = children[c].x;
                code              = 0x80000000u | el;
                key               = sorted_keys ? c - ni : el;
            }
            sl[k][2 * side]     = make_float4(B.lo.x, B.lo.y, B.lo.z, __uint_as_float(code));
            sl[k][2 * side + 1] = make_float4(B.hi.x, B.hi.y, B.hi.z, __uint_as_float(key));
        };
        if (!(tc.x & 0x80000000u)) outside(tc.x, 0);
        if (!(tc.y & 0x80000000u)) outside(tc.y, 1);
    }
    __syncthreads();
    // this node's level: lvp[h] <= k < lvp[h + 1]; the deepest level holding a top node starts the loop
    int my_h = -1;
    if (on)
    {
        int a = 0, b = (int)h1;  // largest h with lvp[h] <= k
        while (a < b)
        {
            const int m = (a + b + 1) / 2;
            if (lvp[m] <= k) a = m;
            else b = m - 1;
        }
        my_h = a;
    }
    int deepest = 0;
    {
        // the last top node is on the deepest top level
        int a = 0, b = (int)h1;
        while (a < b)
        {
            const int m = (a + b + 1) / 2;
            if (lvp[m] <= T - 1u) a = m;
            else b = m - 1;
        }
        deepest = a;
    }
    for (int h = deepest; h >= 0; h--)
    {
        if (my_h == h)
        {
            // a top child's slot: the union of its own two slots, its node id, its largest key
            auto inside = [&](uint32_t c, uint32_t kc, int side) {
                const float4 a0 = sl[kc][0], a1 = sl[kc][1], b0 = sl[kc][2], b1 = sl[kc][3];
                const uint32_t key = max(__float_as_uint(a1.w), __float_as_uint(b1.w));
                sl[k][2 * side] = make_float4(smin(a0.x, b0.x), smin(a0.y, b0.y), smin(a0.z, b0.z), __uint_as_float(c));
                sl[k][2 * side + 1] =
                    make_float4(smax(a1.x, b1.x), smax(a1.y, b1.y), smax(a1.z, b1.z), __uint_as_float(key));
            };
            if (tc.x & 0x80000000u) inside(tc.x & 0x7fffffffu, tc.z, 0);
            if (tc.y & 0x80000000u) inside(tc.y & 0x7fffffffu, tc.w, 1);
        }
        __syncthreads();
    }
    if (!on) return;
    const float4 pa0 = sl[k][0], pa1 = sl[k][1], pb0 = sl[k][2], pb1 = sl[k][3];
    nodes[p] = NodeBox{make_float4(smin(pa0.x, pb0.x), smin(pa0.y, pb0.y), smin(pa0.z, pb0.z), 0.0f),
                       make_float4(smax(pa1.x, pb1.x), smax(pa1.y, pb1.y), smax(pa1.z, pb1.z), 0.0f)};
    float4* P = packed + 4 * (size_t)p;
    P[0]      = pa0;
    P[1]      = pa1;
    P[2]      = pb0;
    P[3]      = pb1;
    if (!packed4) return;
    float4* Q = packed4 + 8 * (size_t)p;
    const uint32_t cs[2] = {tc.x, tc.y}, ks[2] = {tc.z, tc.w};
    for (int side = 0; side < 2; side++)
    {
        const uint32_t c  = cs[side];
        float4*        QS = Q + 4 * side;
        if (c & 0x80000000u)
        {
            for (int t = 0; t < 4; t++) QS[t] = sl[ks[side]][t];
        }
        else if (c < ni)
        {
            const float4* C = packed + 4 * (size_t)c;
            for (int t = 0; t < 4; t++) QS[t] = C[t];
        }
        else
        {
            QS[0] = sl[k][2 * side];
            QS[1] = sl[k][2 * side + 1];
            empty_slot(QS + 2);
        }
    }
}

// One treelet per workgroup: its inner nodes, a contiguous index range of at most kTreeletLeaves - 1
// nodes, whose children lie in the treelet or are leaves of its leaf range. One thread per leaf
// climbs: of a node's two children the one that arrives last (a ticket in LDS) forms its box and
// goes on, so there is no barrier between levels, and everything the climb reads was put into LDS
// before it. The node boxes and records are written after the climb, all nodes at once. The results
// are the ones inner_box writes. (Level by level with the records written inside a level, every
// level's barrier waited for stores: 57 us on average on the cloth tube's 385 and 688 treelets, now 29.)
constexpr int kTreeletBlock = 1024;
__global__ __launch_bounds__(kTreeletBlock) void k_refit_treelets(const uint32_t* __restrict__ count,
                                                                   const uint32_t* __restrict__ troots,
                                                                   const uint32_t* __restrict__ tsize,
                                                                   const uint32_t* __restrict__ tfirst,
                                                                   const uint32_t* __restrict__ tleaf,
                                                                   const uint32_t* __restrict__ parent, uint32_t ni,
                                                                   const uint2* __restrict__ children, NodeBox* nodes,
                                                                   float4* packed, float4* packed4, int sorted_keys)
{
    static_assert(kTreeletLeaves == kTreeletBlock, "one thread per leaf and per inner node");
    constexpr uint32_t kN = kTreeletLeaves;
    __shared__ float    lb[6][kN], ib[6][kN];  // leaf and inner boxes (lo.xyz, hi.xyz)
    __shared__ uint32_t lcode[kN], lkey[kN], ikey[kN], ich[2][kN], ticket[kN];
    __shared__ uint16_t up[kN];  // a node's parent in the treelet
    const uint32_t      k = threadIdx.x, T = count[0];
    for (uint32_t b = blockIdx.x; b < T; b += gridDim.x)
    {
        const uint32_t r = troots[b], first = tfirst[r], cnt = tsize[r] - 1u, leaf0 = tleaf[r], nl = cnt + 1u;
        uint32_t       node = kN;  // the leaf's parent in the treelet
        if (k < nl)
        {
            const NodeBox  B  = nodes[ni + leaf0 + k];
            const uint32_t el = children[ni + leaf0 + k].x;  // a leaf keeps (element, element)
            node              = parent[ni + leaf0 + k] - first;
            lb[0][k]          = B.lo.x;
            lb[1][k]          = B.lo.y;
            lb[2][k]          = B.lo.z;
            lb[3][k]          = B.hi.x;
            lb[4][k]          = B.hi.y;
            lb[5][k]          = B.hi.z;
            lcode[k]          = 0x80000000u | el;
            lkey[k]           = sorted_keys ? leaf0 + k : el;
        }
        if (k < cnt)
        {
            const uint2 c = children[first + k];
            ich[0][k]     = c.x;
            ich[1][k]     = c.y;
            up[k]         = (uint16_t)(first + k == r ? kN : parent[first + k] - first);
            ticket[k]     = 0u;
        }
        __syncthreads();
        // a child's box and key from LDS (c: node id, a leaf of the range or an inner node)
        auto child = [&](uint32_t c, float* bx, uint32_t& key) {
            const bool     leaf = c >= ni;
            const uint32_t l    = leaf ? c - ni - leaf0 : c - first;
#pragma unroll
            for (int t = 0; t < 6; t++) bx[t] = leaf ? lb[t][l] : ib[t][l];
            key = leaf ? lkey[l] : ikey[l];
        };
        // a treelet of cnt nodes is climbed in at most cnt steps
        for (uint32_t step = 0; node < kN && step < cnt; step++)
        {
            if (atomicAdd(&ticket[node], 1u) == 0u) break;  // the sibling comes later
            __threadfence_block();
            float    A[6], B[6];
            uint32_t ma, mb;
            child(ich[0][node], A, ma);
            child(ich[1][node], B, mb);
#pragma unroll
            for (int t = 0; t < 3; t++)
            {
                ib[t][node]     = smin(A[t], B[t]);
                ib[t + 3][node] = smax(A[t + 3], B[t + 3]);
            }
            ikey[node] = max(ma, mb);
            __threadfence_block();
            node = up[node];
        }
        __syncthreads();
        // the records: lane by lane along memory (eight lanes per four-wide record, four per binary
        // one, two per box), so a wavefront's store is one contiguous kilobyte; a thread per node
        // wrote 14 times 64 separate lines
        auto part = [&](uint32_t c, bool hi) {
            const bool     leaf = c >= ni;
            const uint32_t l    = leaf ? c - ni - leaf0 : c - first, t = hi ? 3u : 0u;
            if (leaf) return make_float4(lb[t][l], lb[t + 1][l], lb[t + 2][l], __uint_as_float(hi ? lkey[l] : lcode[l]));
            return make_float4(ib[t][l], ib[t + 1][l], ib[t + 2][l], __uint_as_float(hi ? ikey[l] : c));
        };
        float4* const Q = packed4 + 8 * (size_t)first;
        for (uint32_t i = k; packed4 && i < 8u * cnt; i += kN)
        {
            const uint32_t c = ich[(i >> 2) & 1u][i >> 3], sub = (i >> 1) & 1u;
            const bool     hi = (i & 1u) != 0u;
            float4         v;
            if (c < ni) v = part(ich[sub][c - first], hi);
            else if (sub == 0u) v = part(c, hi);
            else
            {
                // a leaf child: itself and an empty slot
                const float inf = __int_as_float(hi ? 0xff800000 : 0x7f800000);
                v               = make_float4(inf, inf, inf, __uint_as_float(hi ? 0u : 0x80000000u));
            }
            Q[i] = v;
        }
        float4* const P = packed + 4 * (size_t)first;
        for (uint32_t i = k; i < 4u * cnt; i += kN) P[i] = part(ich[(i >> 1) & 1u][i >> 2], (i & 1u) != 0u);
        float4* const N = &nodes[first].lo;
        for (uint32_t i = k; i < 2u * cnt; i += kN)
        {
            const uint32_t t = 3u * (i & 1u);
            N[i]             = make_float4(ib[t][i >> 1], ib[t + 1][i >> 1], ib[t + 2][i >> 1], 0.0f);
        }
        __syncthreads();  // the next treelet's LDS
    }
}

// ---------------------------------------------------------------- traversal
constexpr int kQueryBlock = 128;
constexpr int kStack      = 32;  // traversal stack entries per query (lbvh.cpp:300)

// lbvh.cpp:293-360 / aabb.h:96-100: strict overlap of a node box (lo4, hi4) with the query box
LCSX_D bool overlap4(float4 lo4, float4 hi4, f3 lo, f3 hi)
{
    return (lo4.x < hi.x && lo4.y < hi.y && lo4.z < hi.z) && (hi4.x > lo.x && hi4.y > lo.y && hi4.z > lo.z);
}

// Query variants: stack entries held in LDS (the rest of the 32 go to a per-thread global spill
// area) and pairs staged per wavefront before one global reservation (a reservation is made once
// more than kBuf - 128 are staged). Fewer LDS stack entries leave room for a larger staging
// buffer (fewer atomics on the shared pair counter) or more resident wavefronts; the pairs found
// are the same in every variant.
struct QueryShape
{
    int wide;       // nodes tested per step: 2 (binary records) or 4 (grandchildren)
    int lds_stack;  // stack entries in LDS (per query)
    int buf;        // pairs staged per wavefront
    int lanes;      // lanes per query: 1, 2 or 4 (lane j tests 4 / lanes of the record's slots)
};
constexpr QueryShape kQueryShapes[kQueryVariants] = {{2, 32, 256, 1}, {2, 16, 512, 1}, {2, 16, 1024, 1},
                                                     {2, 8, 1024, 1},  {4, 16, 512, 1}, {4, 8, 1024, 1},
                                                     {4, 32, 512, 1},  {4, 16, 512, 4}, {4, 32, 512, 4},
                                                     {4, 16, 512, 2}};

// Copies a wavefront's staged pairs to the global list: one atomic reserves the range, lanes
// copy in strides of 64. Called by all 64 lanes.
LCSX_D void flush_pairs(const uint2* buf, uint32_t nbuf, uint32_t* count, uint32_t capacity, uint32_t* pairs)
{
    __builtin_amdgcn_wave_barrier();
    uint32_t base = 0;
    if (lane_id() == 0) base = count_reserve(count, nbuf);
    base = __shfl(base, 0);
    for (uint32_t k = lane_id(); k < nbuf; k += 64u)
        if (base + k < capacity)
        {
            const uint2 v = buf[k];
            pairs[2 * (size_t)(base + k)]     = v.x;
            pairs[2 * (size_t)(base + k) + 1] = v.y;
        }
    __builtin_amdgcn_wave_barrier();
}

// query_template2, lbvh.cpp:293-360: depth-first with a stack of kSt entries (the first kS in LDS,
// the rest in the spill area); a full stack ends the query (the reference's silent truncation),
// reported through *overflow. kW = 2: each step loads one binary record (both child boxes and
// codes, 64 B), tests the children and pushes inner hits in the reference's order, with the
// reference's 32 entries. kW = 4: each step loads a 4-wide record (the grandchildren, 128 B), so
// the traversal takes about half the dependent steps and finds the same leaves; up to three
// entries per step stay on the stack, so it holds 64. The wavefront loops until all its lanes are
// done, so hits are staged in LDS and written with one atomic per kBuf - 64 kW or more pairs.
template <int kW, int kS, int kBuf>
__global__ __launch_bounds__(kQueryBlock) void k_query(QueryArgs a, const float4* __restrict__ packed, uint32_t n_inner,
                                                        const uint32_t* __restrict__ roots, const NodeBox* __restrict__ nodes,
                                                        const uint2* __restrict__ children, uint32_t* __restrict__ spill)
{
    constexpr int kSt = kW == 2 ? kStack : 2 * kStack;
    static_assert((kW == 2 || kW == 4) && kS > 0 && kS <= kSt && kBuf >= 128 + 64 * kW, "query shape");
    __shared__ uint32_t stack[kS][kQueryBlock];
    __shared__ uint2    buf[kQueryBlock / 64][kBuf];
    const uint32_t      tid = threadIdx.x, wv = tid >> 6;
    // spill slot j of this thread: spill[j * threads + gt] (lanes of a wavefront are adjacent)
    const size_t        gt = (size_t)blockIdx.x * kQueryBlock + tid, threads = (size_t)gridDim.x * kQueryBlock;
    auto push = [&](int& sp, uint32_t v) {
        if (sp < kS) stack[sp][tid] = v;
        else spill[(size_t)(sp - kS) * threads + gt] = v;
        sp++;
    };
    auto pop = [&](int& sp) -> uint32_t {
        --sp;
        // an LDS read, and the spill read (a relaxed atomic load, which the compiler does not
        // merge with the LDS one into a flat load) only past the LDS part
        uint32_t v = stack[sp < kS ? sp : kS - 1][tid];
        if (sp >= kS)
            v = __hip_atomic_load(spill + (size_t)(sp - kS) * threads + gt, __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_WAVEFRONT);
        return v;
    };
    // consecutive queries (spatially close, so they visit the same subtrees) on one XCD
    const uint32_t      qi  = xcd_block(blockIdx.x, gridDim.x) * kQueryBlock + tid;
    bool                active = qi < a.n_queries;
    // sorted self-query (edges against their own tree, packed keys = sorted leaf indices): thread
    // qi queries the edge at sorted leaf qi and keeps leaves after it in sorted order
    const bool          self = a.mode == QueryEdges && a.sorted_self;
    const uint32_t      q    = (self && active) ? a.order[qi] : qi;
    const uint32_t      fk   = self ? qi : q;  // filter key, compared with the packed keys
    f3                  lo = mk(0.0f, 0.0f, 0.0f), hi = mk(0.0f, 0.0f, 0.0f);
    bool                filt = false;
    if (active)
    {
        if (a.mode == QueryVerts)
        {
            f3    p0 = ld3(a.x0, q), p1 = ld3(a.x1, q);
            float t  = a.offset[q] + a.dhat[q];
            lo       = vmin(p0, p1) - mk(t, t, t);
            hi       = vmax(p0, p1) + mk(t, t, t);
        }
        else if (a.mode == QueryEdges)
        {
            uint32_t e0 = a.edges[2 * q], e1 = a.edges[2 * q + 1];
            f3       s0 = ld3(a.x0, e0), s1 = ld3(a.x0, e1), t0 = ld3(a.x1, e0), t1 = ld3(a.x1, e1);
            float    t  = a.offset[e0] + a.dhat[e0];
            lo          = vmin(vmin(s0, s1), vmin(t0, t1)) - mk(t, t, t);
            hi          = vmax(vmax(s0, s1), vmax(t0, t1)) + mk(t, t, t);
            filt        = true;
        }
        else
        {
            lo   = ld3(a.boxes, 2 * q);
            hi   = ld3(a.boxes, 2 * q + 1);
            filt = a.edge_filter != 0;
        }
    }
    uint32_t root = kInvalid;
    if (active)
    {
        uint32_t g = 0;
        if (a.vert_scene && a.mode != QueryBoxes) g = a.vert_scene[a.mode == QueryVerts ? q : a.edges[2 * q]];
        root = roots[g];
        if (root == kInvalid || (a.active && a.active[g] == 0)) active = false;
        if (a.mode == QueryVerts && a.row_kind && a.row_kind[q] >= 2u) active = false;
    }
    int sp = 0;
    if (active) push(sp, root);
    // each inner node is expanded at most once per query in a well-formed tree; the cap (as the
    // reference's 100000-iteration guard) only bounds a corrupted one
    uint32_t visits = 0;
    uint32_t nbuf   = 0;  // staged pairs of this wavefront (uniform across its lanes)
    while (__ballot(active && sp > 0) != 0ull)
    {
        bool     e[kW];
        uint32_t o[kW];
#pragma unroll
        for (int c = 0; c < kW; c++)
        {
            e[c] = false;
            o[c] = 0u;
        }
        if (active && sp > 0)
        {
            if (++visits > n_inner + 1u)
            {
                if (a.overflow) atomicOr(a.overflow, 2u);
                active = false;
            }
            else
            {
                const uint32_t nd = pop(sp);
                float4         r[2 * kW];
                if (nd < n_inner)
                {
                    const float4* P = packed + 2 * kW * (size_t)nd;
#pragma unroll
                    for (int c = 0; c < 2 * kW; c++) r[c] = P[c];
                }
                else
                {
                    // a one-leaf segment's root: the leaf alone, as slot 0 (the other slots never hit)
                    NodeBox  B = nodes[nd];
                    uint32_t o0 = children[nd].x;
                    r[0] = make_float4(B.lo.x, B.lo.y, B.lo.z, __uint_as_float(0x80000000u | o0));
                    r[1] = make_float4(B.hi.x, B.hi.y, B.hi.z, __uint_as_float(self ? nd - n_inner : o0));
                    const float inf = __int_as_float(0x7f800000);
#pragma unroll
                    for (int c = 1; c < kW; c++)
                    {
                        r[2 * c]     = make_float4(inf, inf, inf, __uint_as_float(0x80000000u));
                        r[2 * c + 1] = make_float4(-inf, -inf, -inf, 0.0f);
                    }
                }
                bool brk = false;
#pragma unroll
                for (int c = 0; c < kW; c++)
                {
                    const uint32_t code = __float_as_uint(r[2 * c].w);
                    // with the edge filter (keep q < element) a subtree whose largest element id
                    // is <= q holds no pair: it is not descended (leaf: the largest id is the element)
                    bool h = !brk && overlap4(r[2 * c], r[2 * c + 1], lo, hi) &&
                             (!filt || fk < __float_as_uint(r[2 * c + 1].w));
                    const bool leaf = (code & 0x80000000u) != 0u;
                    if (h && !leaf)
                    {
                        if (sp < kSt) push(sp, code);
                        else
                        {
                            // a full stack ends the query before the later children
                            brk = true;
                            h   = false;
                            if (a.overflow) atomicOr(a.overflow, 1u);
                        }
                    }
                    e[c] = h && leaf;
                    o[c] = code & 0x7fffffffu;
                }
                if (brk) active = false;
            }
        }
        uint64_t bal[kW];
        uint32_t cnt = 0;
#pragma unroll
        for (int c = 0; c < kW; c++)
        {
            bal[c] = __ballot(e[c]);
            cnt += (uint32_t)__popcll(bal[c]);
        }
        if (cnt)
        {
            const uint64_t lt  = lanemask_lt();
            uint32_t       off = nbuf;
#pragma unroll
            for (int c = 0; c < kW; c++) off += (uint32_t)__popcll(bal[c] & lt);
            // a sorted self-query stores each pair as (lower id, higher id), as the element-id filter does
#pragma unroll
            for (int c = 0; c < kW; c++)
                if (e[c]) buf[wv][off++] = self ? make_uint2(min(q, o[c]), max(q, o[c])) : make_uint2(q, o[c]);
            nbuf += cnt;
            if (nbuf > (uint32_t)(kBuf - 64 * kW))
            {
                flush_pairs(buf[wv], nbuf, a.count, a.capacity, a.pairs);
                nbuf = 0;
            }
        }
    }
    if (nbuf) flush_pairs(buf[wv], nbuf, a.count, a.capacity, a.pairs);
}

// Four lanes per query on the four-wide records: lane j of a group of four tests slot j, so the
// group's record is one contiguous 128 B load (16 records per wavefront load instead of 64 when
// each lane walks its own query), and the group shares one stack (64 entries, the first kS in LDS)
// and one step count. Same leaves as the other shapes; a full stack ends the query after the
// step's leaves are emitted, reported through *overflow.
template <int kS, int kBuf, int kL>
__global__ __launch_bounds__(kQueryBlock) void k_query_coop(QueryArgs a, const float4* __restrict__ packed4,
                                                             uint32_t n_inner, const uint32_t* __restrict__ roots,
                                                             const NodeBox* __restrict__ nodes,
                                                             const uint2* __restrict__ children,
                                                             uint32_t* __restrict__ spill)
{
    // kL lanes per query (4 or 2), each testing kU = 4 / kL slots of the four-wide record
    constexpr int      kU      = 4 / kL;
    constexpr int      kSt     = 2 * kStack;
    constexpr uint32_t kGroups = kQueryBlock / kL;
    constexpr uint32_t kGMask  = (1u << kL) - 1u;
    static_assert((kL == 4 || kL == 2) && kS > 0 && kS <= kSt && kBuf >= 128 + 64 * kU, "query shape");
    __shared__ uint32_t stack[kS][kGroups];
    __shared__ uint2    buf[kQueryBlock / 64][kBuf];
    const uint32_t      tid = threadIdx.x, wv = tid >> 6, grp = tid / kL, j = tid % kL;
    const size_t        gq = (size_t)blockIdx.x * kGroups + grp, groups = (size_t)gridDim.x * kGroups;
    auto put = [&](int pos, uint32_t v) {
        if (pos < kS) stack[pos][grp] = v;
        else spill[(size_t)(pos - kS) * groups + gq] = v;
    };
    auto get = [&](int pos) -> uint32_t {
        // the LDS entry read unconditionally and the spill entry (a relaxed atomic load, which the
        // compiler does not merge with the LDS one) only past it: the common read stays an LDS
        // read instead of a flat load
        uint32_t v = stack[pos < kS ? pos : kS - 1][grp];
        if (pos >= kS)
            v = __hip_atomic_load(spill + (size_t)(pos - kS) * groups + gq, __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_WAVEFRONT);
        return v;
    };
    const uint32_t qi     = xcd_block(blockIdx.x, gridDim.x) * kGroups + grp;
    bool           active = qi < a.n_queries;
    const uint32_t q      = qi;
    const bool     filt = a.edge_filter != 0;
    f3             lo = mk(0.0f, 0.0f, 0.0f), hi = mk(0.0f, 0.0f, 0.0f);
    if (active)
    {
        lo = ld3(a.boxes, 2 * q);
        hi = ld3(a.boxes, 2 * q + 1);
    }
    const uint32_t root = roots[0];  // a tree queried with boxes is one segment
    if (root == kInvalid) active = false;
    // rank of this lane among the set lanes of a ballot below it
    auto rank = [](uint64_t bal) -> uint32_t {
        return __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
    };
    auto pair_of = [&](uint32_t o) { return make_uint2(q, o); };
    int      sp     = 0;
    uint32_t visits = 0;
    uint32_t nbuf   = 0;
    // a one-leaf segment's root is a leaf: tested here, so every node the loop visits is inner
    {
        bool     e0 = false;
        uint32_t o0 = 0u;
        if (active && root >= n_inner)
        {
            if (j == 0u)
            {
                const NodeBox  B   = nodes[root];
                const uint32_t el  = children[root].x;
                                e0 = overlap4(make_float4(B.lo.x, B.lo.y, B.lo.z, 0.0f), make_float4(B.hi.x, B.hi.y, B.hi.z, 0.0f), lo,
                              hi) &&
                     (!filt || q < el);
                o0 = el;
            }
            active = false;
        }
        const uint64_t bal = __ballot(e0);
        if (e0) buf[wv][rank(bal)] = pair_of(o0);
        nbuf = (uint32_t)__popcll(bal);
    }
    for (int t = (int)j; t < kS; t += kL) stack[t][grp] = 0u;  // the group's LDS stack, zeroed
    if (active)
    {
        if (j == 0u) put(0, root);
        sp = 1;
    }
    // Every lane runs every step without a divergent branch on its common path: a lane whose
    // group has no work reads a stale stack entry and that node's record and drops the result.
    // The LDS stack starts zeroed (above) and only ever holds inner node ids, so a stale entry is
    // a node of the tree (the loop runs only while some group has an inner node to visit, so node
    // 0 exists). A query that ends early (a full stack, or more steps than inner nodes) empties
    // its stack, so the work test is one compare.
    while (true)
    {
        bool work = sp > 0;
        if (__ballot(work) == 0ull) break;
        // the top entry (an empty stack reads entry kS - 1, a stale node id whose record is dropped)
        uint32_t nd = stack[min((uint32_t)(sp - 1), (uint32_t)kS - 1u)][grp];
        if (work && sp > kS)
            nd = __hip_atomic_load(spill + (size_t)(sp - 1 - kS) * groups + gq, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WAVEFRONT);
        if (work)
        {
            sp--;
            if (++visits > n_inner + 1u)
            {
                if (a.overflow && j == 0u) atomicOr(a.overflow, 2u);
                sp   = 0;
                work = false;
            }
        }
        // 32-bit record index (a tree holds fewer than 2^28 leaves, so fewer inner nodes)
        const float4* P = packed4 + (nd * 8u + 2u * kU * j);
        float4        r[2 * kU];
#pragma unroll
        for (int u = 0; u < 2 * kU; u++) r[u] = P[u];
        uint32_t code[kU], gm[kU];
        bool     inner_hit[kU], e[kU];
        int      npush = 0;
#pragma unroll
        for (int u = 0; u < kU; u++)
        {
            // bitwise, not short-circuit, so the conditions stay lane masks in scalar registers
            code[u]      = __float_as_uint(r[2 * u].w);
            const bool h = work & overlap4(r[2 * u], r[2 * u + 1], lo, hi) &
                           ((q < __float_as_uint(r[2 * u + 1].w)) | !filt);
            inner_hit[u] = h & ((int)code[u] >= 0);
            e[u]         = h & ((int)code[u] < 0);
            gm[u]        = (uint32_t)(__ballot(inner_hit[u]) >> (lane_id() & ~(uint32_t)(kL - 1))) & kGMask;
            npush += __popc(gm[u]);
        }
        // the group's pushes (slot u of every lane, then slot u + 1)
        if (npush)
        {
            if (sp + npush > kSt)
            {
                if (a.overflow && j == 0u) atomicOr(a.overflow, 1u);
                sp = 0;
            }
            else
            {
                const uint32_t below = (1u << j) - 1u;
                int            pos   = sp;
#pragma unroll
                for (int u = 0; u < kU; u++)
                {
                    if (inner_hit[u]) put(pos + __popc(gm[u] & below), code[u]);
                    pos += __popc(gm[u]);
                }
                sp += npush;
            }
        }
#pragma unroll
        for (int u = 0; u < kU; u++)
        {
            const uint64_t bal = __ballot(e[u]);
            if (e[u]) buf[wv][nbuf + rank(bal)] = pair_of(code[u] & 0x7fffffffu);
            nbuf += (uint32_t)__popcll(bal);
        }
        if (nbuf > (uint32_t)(kBuf - 64 * kU))
        {
            flush_pairs(buf[wv], nbuf, a.count, a.capacity, a.pairs);
            nbuf = 0;
        }
    }
    if (nbuf) flush_pairs(buf[wv], nbuf, a.count, a.capacity, a.pairs);
}

// ---- The solver's own hierarchy (ClusterTree). A block is kClusterLeaves consecutive positions of the
// static order and a complete 4-ary tree over them: 256 records of four leaves, 64 of four of those, and
// so on to one, kClusterRecords records of the packed4 layout in a row, children at fixed places. Above
// the blocks there is only the list of their boxes, which a wavefront tests 64 at a time.
// Unions drop NaNs (fminf, fmaxf), so a vertex gone astray hides no other.
LCSX_D f3 umin(f3 a, f3 b) { return mk(fminf(a.x, b.x), fminf(a.y, b.y), fminf(a.z, b.z)); }
LCSX_D f3 umax(f3 a, f3 b) { return mk(fmaxf(a.x, b.x), fmaxf(a.y, b.y), fmaxf(a.z, b.z)); }
constexpr uint32_t kClusterRecords = 341;  // 256 + 64 + 16 + 4 + 1
static_assert(kClusterLeaves == 1024, "kClusterRecords");

// One workgroup per block: a thread makes the record of its four positions, then each level's boxes go
// into their parents' records, all in LDS; the block leaves as one stretch of 43 KB. Bound by the gathered
// loads of the elements' vertices. 187,000 faces and 281,000 edges: 11 us on average (the LBVH's leaves,
// treelets and top: 54).
__global__ __launch_bounds__(256) void k_cluster_refit(int arity, const uint32_t* __restrict__ prims,
                                                       const uint32_t* __restrict__ elem, const uint32_t* __restrict__ leaf_of,
                                                       const float* __restrict__ x0, const float* __restrict__ x1,
                                                       const float* __restrict__ pad, float4* __restrict__ rec,
                                                       float4* __restrict__ top)
{
    __shared__ float4 img[8 * kClusterRecords];
    const uint32_t    t = threadIdx.x, blk = blockIdx.x;
    const float       inf = __int_as_float(0x7f800000);
    f3                lo = mk(inf, inf, inf), hi = mk(-inf, -inf, -inf);
    uint32_t          key = 0;
#pragma unroll
    for (uint32_t k = 0; k < 4; k++)
    {
        const uint32_t at = blk * kClusterLeaves + 4 * t + k;
        const uint32_t el = elem[at];  // kInvalid: a position between two scenes
        float4         l  = make_float4(inf, inf, inf, __uint_as_float(0x80000000u));
        float4         h  = make_float4(-inf, -inf, -inf, 0.0f);
        if (el != kInvalid)
        {
            const NodeBox  B = leaf_box(at, arity, prims, elem, x0, x1, pad);
            const uint32_t w = leaf_of ? leaf_of[el] : el;
            l   = make_float4(B.lo.x, B.lo.y, B.lo.z, __uint_as_float(0x80000000u | el));
            h   = make_float4(B.hi.x, B.hi.y, B.hi.z, __uint_as_float(w));
            lo  = umin(lo, mk(l.x, l.y, l.z));
            hi  = umax(hi, mk(h.x, h.y, h.z));
            key = max(key, w);
        }
        img[8 * t + 2 * k]     = l;
        img[8 * t + 2 * k + 1] = h;
    }
    // this thread's box, as a slot of its parent's record; then the next level's first threads
    uint32_t node = t, base = 256, cnt = 256;
    while (true)
    {
        if (t < cnt)
        {
            const float4 l = make_float4(lo.x, lo.y, lo.z, __uint_as_float(blk * kClusterRecords + node));
            const float4 h = make_float4(hi.x, hi.y, hi.z, __uint_as_float(key));
            if (cnt == 1u)
            {
                top[2 * blk]     = l;
                top[2 * blk + 1] = h;
            }
            else
            {
                img[8 * (base + t / 4u) + 2 * (t & 3u)]     = l;
                img[8 * (base + t / 4u) + 2 * (t & 3u) + 1] = h;
            }
        }
        __syncthreads();
        if (cnt == 1u) break;
        cnt /= 4u;
        node = base + t;
        if (t < cnt)
        {
            lo  = mk(inf, inf, inf);
            hi  = mk(-inf, -inf, -inf);
            key = 0;
#pragma unroll
            for (uint32_t k = 0; k < 4; k++)
            {
                const float4 l = img[8 * node + 2 * k], h = img[8 * node + 2 * k + 1];
                lo  = umin(lo, mk(l.x, l.y, l.z));
                hi  = umax(hi, mk(h.x, h.y, h.z));
                key = max(key, __float_as_uint(h.w));
            }
        }
        base += cnt;
    }
    float4* const out = rec + (size_t)blk * (8 * kClusterRecords);
    for (uint32_t k = t; k < 8 * kClusterRecords; k += 256u) out[k] = img[k];
}

// One wavefront per 16 consecutive points or edges of the static order: they visit nearly the same nodes,
// so the wavefront walks the tree once for all of them, up to 32 nodes a step (four lanes test the slots of
// a record against the queries' joint boxes), lists the leaves met in LDS and tests each of them against
// the queries, four leaves at a time in the four quarters of the wavefront. In the LBVH (whose Morton box,
// as the reference's, covers the first third of a cloth's edges, so the rest is sorted along two axes or
// one) a query's own walk visited 15 to 250 records one after the other.
// The order's curve jumps now and then, and one joint box over a jump would cover much of the mesh: the
// queries are cut at the three largest jumps into four joint boxes (64 queries on a 161 x 161 cloth and its
// sphere met 299 leaves with one box, 152 with four, 147 with eight).
// 16 queries: 64 leave a small mesh with a few long wavefronts (a 33 x 33 cloth: 39 us, 14 with 16), and
// their 64 box tests per leaf met are mostly misses; 8 walk the top of the tree twice as often (edges
// of the batch below: 1310 us against 680, before the reservations were shared).
// kEdges: an edge keeps the leaves whose key is above its own: the LBVH's sorted leaf where the pair test
// is symmetric (sorted_ee), so that each pair is tested from the same side as in a query of the LBVH, or
// the element id.
// Per query of edges and of points: 24 scenes of 306,000 vertices, 6.5 M and 2.4 M pairs: 226 and 87 us
// (1162 and 307 in the LBVH with four lanes per query); 297 x 297 tube in wide contact bands: 273 and 92 us
// (497 and 176).
constexpr int kGroupStack = 384, kGroupLeaves = 160, kGroupBuf = 768, kGroupCuts = 3;
constexpr uint32_t kGroup = 16;  // queries of a wavefront
constexpr int kGroupWaves = 8;
constexpr int kGroupTests = 4;  // leaves read together per quarter, ahead of their tests
template <bool kEdges>
__global__ __launch_bounds__(64 * kGroupWaves) void k_query_group(ClusterQuery a, const float4* __restrict__ rec,
                                                              const float4* __restrict__ top,
                                                              const uint32_t* __restrict__ scene_block,
                                                              const uint32_t* __restrict__ leaf_of)
{
    constexpr int kWaves = kGroupWaves, kBoxes = kGroupCuts + 1;
    constexpr uint32_t kShares = 64u / kGroup;
    static_assert(kGroup <= 16 && kGroupTests * 64 <= kGroupBuf, "a pair's query takes 4 bits, its element 28 (Lbvh::init)");
    static_assert(kGroupLeaves % (kGroupTests * kShares) == 0, "the last batch of tests stays in the list");
    __shared__ uint32_t stack_[kWaves][kGroupStack];
    __shared__ float4   leaf_[kWaves][2 * kGroupLeaves];
    __shared__ uint32_t buf_[kWaves][kGroupBuf];  // pairs: query in the top 4 bits, element below
    __shared__ uint32_t n_[kWaves], base_;
    const uint32_t      wv = threadIdx.x >> 6, lane = lane_id(), g = lane >> 2, j = lane & 3u;
    const uint32_t      li = lane & (kGroup - 1u), part = lane / kGroup;  // query, share of the leaves
    uint32_t* const     stack = stack_[wv];
    float4* const       leaf  = leaf_[wv];
    uint32_t* const     buf   = buf_[wv];
    const uint32_t      at    = (xcd_block(blockIdx.x, gridDim.x) * kWaves + wv) * kGroup;
    const float         inf   = __int_as_float(0x7f800000);
    auto rank = [](uint64_t bal) -> uint32_t {
        return __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
    };
    // this lane's query (the lists are padded to whole wavefronts per scene)
    const uint32_t q = at < a.n ? a.order[at + li] : kInvalid;
    bool           live = __ballot(q != kInvalid) != 0ull;  // uniform across the wavefront
    f3       lo = mk(inf, inf, inf), hi = mk(-inf, -inf, -inf);
    uint32_t own = kInvalid, sc = 0;  // key above which leaves are kept (kEdges), scene
    if (q != kInvalid)
    {
        const uint32_t e0 = kEdges ? a.edges[2 * q] : q;
        const float    t  = a.offset[e0] + a.dhat[e0];
        if (kEdges)
        {
            const uint32_t e1 = a.edges[2 * q + 1];
            const f3       s0 = ld3(a.x0, e0), s1 = ld3(a.x0, e1), t0 = ld3(a.x1, e0), t1 = ld3(a.x1, e1);
            lo  = vmin(vmin(s0, s1), vmin(t0, t1)) - mk(t, t, t);
            hi  = vmax(vmax(s0, s1), vmax(t0, t1)) + mk(t, t, t);
            own = leaf_of ? leaf_of[q] : q;
        }
        else
        {
            const f3 p0 = ld3(a.x0, q), p1 = ld3(a.x1, q);
            lo = vmin(p0, p1) - mk(t, t, t);
            hi = vmax(p0, p1) + mk(t, t, t);
        }
        if (a.vert_scene) sc = a.vert_scene[e0];
    }
    // a scene's first position is a multiple of 64, so lane 0 holds a query of it
    sc = (uint32_t)__builtin_amdgcn_readfirstlane((int)sc);
    live = live && !(a.active && a.active[sc] == 0);
    // ---- joint boxes: lanes [start, ...) up to the next cut share one
    uint64_t cuts = 1ull;  // bit l: a joint box starts at lane l
    {
        const f3 ln = mk(__shfl_down(lo.x, 1), __shfl_down(lo.y, 1), __shfl_down(lo.z, 1));
        const f3 hn = mk(__shfl_down(hi.x, 1), __shfl_down(hi.y, 1), __shfl_down(hi.z, 1));
        const f3 e  = vmax(hi, hn) - vmin(lo, ln);
        // the extent of this lane's and the next one's joint box, with the lane in the low bits
        uint32_t d = (__float_as_uint(fmaxf(fmaxf(fmaxf(e.x, e.y), e.z), 0.0f)) & ~63u) | li;
        if (li == kGroup - 1u) d = 0u;
#pragma unroll
        for (int c = 0; c < kGroupCuts; c++)
        {
            uint32_t m = d;
            for (int o = kGroup / 2; o > 0; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o));
            const uint32_t cut = (uint32_t)__builtin_amdgcn_readfirstlane((int)(m & 63u));
            cuts |= 2ull << cut;
            if (li == cut) d = 0u;
        }
    }
    f3 ulo[kBoxes], uhi[kBoxes];
    {
        const uint32_t start = 63u - (uint32_t)__clzll((long long)(cuts & (~0ull >> (63u - li))));
        f3             l = lo, h = hi;
#pragma unroll
        for (uint32_t o = 1; o < kGroup; o <<= 1)
        {
            const f3 lp = mk(__shfl_up(l.x, o), __shfl_up(l.y, o), __shfl_up(l.z, o));
            const f3 hp = mk(__shfl_up(h.x, o), __shfl_up(h.y, o), __shfl_up(h.z, o));
            if (li >= start + o)
            {
                l = umin(l, lp);
                h = umax(h, hp);
            }
        }
        uint64_t left = cuts;
#pragma unroll
        for (int c = 0; c < kBoxes; c++)
        {
            // the box that starts at the lowest bit ends before the next one
            const bool any = left != 0ull;
            left &= left - 1ull;
            const int last = left ? __ffsll((long long)left) - 2 : (int)kGroup - 1;
            auto      part = [&](float v, float none) {
                const float r = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), last));
                return any ? r : none;
            };
            ulo[c] = mk(part(l.x, inf), part(l.y, inf), part(l.z, inf));
            uhi[c] = mk(part(h.x, -inf), part(h.y, -inf), part(h.z, -inf));
        }
    }
    uint32_t first = own;  // a subtree whose largest key is not above the smallest own one holds no pair
    if (kEdges)
        for (int o = kGroup / 2; o > 0; o >>= 1) first = min(first, (uint32_t)__shfl_xor((int)first, o));
    auto met = [&](float4 b0, float4 b1) {
        bool h = false;
#pragma unroll
        for (int c = 0; c < kBoxes; c++) h = h | overlap4(b0, b1, ulo[c], uhi[c]);
        return kEdges ? h & (first < __float_as_uint(b1.w)) : h;
    };
    uint32_t sp = 0, nleaf = 0, nbuf = 0;  // uniform across the wavefront
    auto     write = [&](uint32_t to) {
        __builtin_amdgcn_wave_barrier();
        for (uint32_t k0 = 0; k0 < nbuf; k0 += 64u)
        {
            const uint32_t k = k0 + lane, v = buf[min(k, nbuf - 1u)];
            const uint32_t e0 = __shfl(q, (int)(v >> 28)), e1 = v & 0x0fffffffu;
            if (k < nbuf && to + k < a.capacity)
            {
                a.pairs[2 * (size_t)(to + k)]     = kEdges ? min(e0, e1) : e0;
                a.pairs[2 * (size_t)(to + k) + 1] = kEdges ? max(e0, e1) : e1;
            }
        }
        __builtin_amdgcn_wave_barrier();
    };
    auto test_leaves = [&]() {
        __builtin_amdgcn_wave_barrier();
        for (uint32_t c0 = part; c0 - part < nleaf; c0 += kGroupTests * kShares)
        {
            float4   b0[kGroupTests], b1[kGroupTests];
            uint64_t bal[kGroupTests];
            uint32_t total = 0;
#pragma unroll
            for (int u = 0; u < kGroupTests; u++)  // (past the last leaf: any entry of the list, dropped)
            {
                b0[u] = leaf[2 * (c0 + u * kShares)];
                b1[u] = leaf[2 * (c0 + u * kShares) + 1];
            }
#pragma unroll
            for (int u = 0; u < kGroupTests; u++)
            {
                bool e = overlap4(b0[u], b1[u], lo, hi) & (c0 + u * kShares < nleaf);
                if (kEdges) e = e & (own < __float_as_uint(b1[u].w));
                bal[u] = __ballot(e);
                total += (uint32_t)__popcll(bal[u]);
            }
            if (nbuf + total > (uint32_t)kGroupBuf)
            {
                uint32_t to = 0;
                if (lane == 0u) to = count_reserve(a.count, nbuf);
                write(__shfl(to, 0));
                nbuf = 0;
            }
#pragma unroll
            for (int u = 0; u < kGroupTests; u++)
            {
                if ((bal[u] >> lane) & 1ull)
                    buf[nbuf + rank(bal[u])] = li << 28 | (__float_as_uint(b0[u].w) & 0x0fffffffu);
                nbuf += (uint32_t)__popcll(bal[u]);
            }
        }
        nleaf = 0;
        __builtin_amdgcn_wave_barrier();
    };
    // ---- the walk: the scene's blocks while few nodes are at hand, else up to 32 nodes a step
    uint32_t       blk = live ? scene_block[sc] : 0u;
    const uint32_t end = live ? scene_block[sc + 1] : 0u;
    while (true)
    {
        if (sp < 16u && blk < end)
        {
            bool   h  = false;
            float4 r0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (blk + lane < end)
            {
                r0 = top[2 * (blk + lane)];
                h  = met(r0, top[2 * (blk + lane) + 1]);
            }
            const uint64_t bal = __ballot(h);
            if (h) stack[sp + rank(bal)] = __float_as_uint(r0.w);
            sp += (uint32_t)__popcll(bal);
            blk += 64u;
            __builtin_amdgcn_wave_barrier();
            continue;
        }
        if (sp == 0u) break;
        // Up to 32 nodes: sp stays below 384. At most 224 entries remain under the 32, and 128 come on top of
        // them; beyond 256 one node is taken at a time, which adds at most 3 for each of the 4 levels below it.
        const uint32_t take = sp > 256u ? 1u : min(sp, 32u);
        sp -= take;
        float4 r0[2], r1[2];
#pragma unroll
        for (int u = 0; u < 2; u++)
        {
            const uint32_t k  = g + 16u * u;
            const uint32_t nd = k < take ? stack[sp + k] : 0u;
            const float4*  P  = rec + (nd * 8u + 2u * j);
            r0[u] = P[0];
            r1[u] = P[1];
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int u = 0; u < 2; u++)
        {
            const bool     h      = (g + 16u * u < take) & met(r0[u], r1[u]);
            const bool     isleaf = (int)__float_as_uint(r0[u].w) < 0;
            const uint64_t bi = __ballot(h & !isleaf), bl = __ballot(h & isleaf);
            if (h & !isleaf) stack[sp + rank(bi)] = __float_as_uint(r0[u].w);
            sp += (uint32_t)__popcll(bi);
            if (h & isleaf)
            {
                leaf[2 * (nleaf + rank(bl))]     = r0[u];
                leaf[2 * (nleaf + rank(bl)) + 1] = r1[u];
            }
            nleaf += (uint32_t)__popcll(bl);
        }
        if (nleaf > (uint32_t)kGroupLeaves - 128u) test_leaves();
        __builtin_amdgcn_wave_barrier();
    }
    if (nleaf) test_leaves();
    // one reservation for the workgroup: single ones queue at the counter, 11 ns each, which was all of the
    // time with one per wavefront (58,000 of them: 680 us)
    if (lane == 0u) n_[wv] = nbuf;
    __syncthreads();
    if (threadIdx.x == 0)
    {
        uint32_t n = 0;
        for (int w = 0; w < kWaves; w++) n += n_[w];
        base_ = n ? count_reserve(a.count, n) : 0u;
    }
    __syncthreads();
    uint32_t to = base_;
    for (uint32_t w = 0; w < wv; w++) to += n_[w];
    write(to);
}

template <int V>
void launch_query_shape(const Lbvh& t, const QueryArgs& a, uint32_t grid, hipStream_t s)
{
    constexpr QueryShape Q = kQueryShapes[V];
    if constexpr (Q.lanes >= 2)
    {
        k_query_coop<Q.lds_stack, Q.buf, Q.lanes><<<grid, kQueryBlock, 0, s>>>(
            a, t.packed4.p, t.ni, t.roots.p, t.nodes.p, t.children.p, t.spill.p);
    }
    else
        k_query<Q.wide, Q.lds_stack, Q.buf><<<grid, kQueryBlock, 0, s>>>(a, Q.wide == 4 ? t.packed4.p : t.packed.p, t.ni,
                                                                         t.roots.p, t.nodes.p, t.children.p, t.spill.p);
}
}  // namespace

void Lbvh::init(int arity_, const uint32_t* device_prims, uint32_t n_leaves, const uint32_t* seg0, uint32_t nseg_)
{
    // element ids travel in 31 bits of a leaf code and the traversal indexes 128 B records of the
    // inner nodes with 32-bit offsets
    if (n_leaves >= (1u << 28))
    {
        set_error("LBVH: at most 2^28 - 1 leaves per tree");
        throw CapacityFailure();
    }
    arity = arity_;
    n     = n_leaves;
    prims = device_prims;
    nseg  = std::max(1u, nseg_);
    seg0_h.assign(nseg + 1, 0u);
    if (seg0)
        for (uint32_t g = 0; g <= nseg; g++) seg0_h[g] = seg0[g];
    else
        seg0_h[1] = n;
    // inner-node bases, roots and per-leaf / per-inner-node segment ids
    ib_h.assign(nseg, 0u);
    roots_h.assign(nseg, kInvalid);
    cover_h.assign(nseg, 0u);
    std::vector<uint32_t> sol(n), isg;
    uint32_t              nonempty = 0;
    for (uint32_t g = 0; g < nseg; g++)
    {
        uint32_t L = seg0_h[g], ng = seg0_h[g + 1] - L;
        for (uint32_t l = L; l < L + ng; l++) sol[l] = g;
        ib_h[g] = L - nonempty;
        if (ng) nonempty++;
        for (uint32_t k = 0; k + 1 < ng; k++) isg.push_back(g);
    }
    ni = n - nonempty;
    for (uint32_t g = 0; g < nseg; g++)
    {
        uint32_t ng = seg0_h[g + 1] - seg0_h[g];
        if (ng >= 2) roots_h[g] = ib_h[g];
        else if (ng == 1) roots_h[g] = ni + seg0_h[g];
    }
    if (n == 0) return;
    hipStream_t s0 = nullptr;
    if (isg.empty()) isg.push_back(0u);
    seg_of_leaf.upload(sol, s0);
    inner_seg.upload(isg, s0);
    roots.upload(roots_h, s0);
    seg_tab.alloc(4 * (size_t)nseg);
    keys[0].alloc(n); keys[1].alloc(n); vals[0].alloc(n); vals[1].alloc(n);
    if (nseg > 1)
    {
        khi[0].alloc(n);
        khi[1].alloc(n);
    }
    hist.alloc(sort_hist_words(n));
    scan_tmp.alloc(scan_tmp_words(sort_hist_words(n)));
    center.alloc(n);
    morton_sorted.alloc(n);
    parent.alloc(n_nodes());
    object_idx.alloc(n_nodes());
    leaf_of.alloc(n);
    children.alloc(n_nodes());
    nodes.alloc(n_nodes());
    packed.alloc(4 * (size_t)(ni ? ni : 1));
    packed4.alloc(8 * (size_t)(ni ? ni : 1));
    tsize.alloc(ni ? ni : 1);
    tfirst.alloc(ni ? ni : 1);
    tleaf.alloc(ni ? ni : 1);
    troots.alloc(ni ? ni : 1);
    tcount.alloc(2);
    top_list.alloc(ni ? ni : 1);
    top_depth.alloc(ni ? ni : 1);
    top_order.alloc(ni ? ni : 1);
    top_level_ptr.alloc(kMaxLevels + 1);
    top_idx.alloc(ni ? ni : 1);
    top_child.alloc(ni ? ni : 1);
    gbox.alloc(6 * (size_t)nseg);
    sorted_to_orig = vals[0].p;
    LCSX_HIP(hipStreamSynchronize(s0));
}

void Lbvh::construct(const float* x, const uint32_t* verts_per_seg, hipStream_t s)
{
    if (n == 0) return;
    std::vector<uint32_t>& tab = tab_h;  // kept: the copy below is asynchronous
    tab.assign(4 * (size_t)nseg, 0u);
    for (uint32_t g = 0; g < nseg; g++)
    {
        uint32_t ng = seg0_h[g + 1] - seg0_h[g];
        cover_h[g]  = (uint32_t)std::min<uint64_t>(ng, ((uint64_t)verts_per_seg[g] + 255u) / 256u * 256u);
        tab[4 * g] = seg0_h[g];
        tab[4 * g + 1] = ng;
        tab[4 * g + 2] = ib_h[g];
        tab[4 * g + 3] = cover_h[g];
    }
    seg_tab.upload(tab, s);
    if (nseg == 1 && n <= kSmallLeaves)
    {
        sorted_to_orig = vals[0].p;
        auto go        = [&](auto kern) {
            kern<<<1, 1024, 0, s>>>(n, ni, arity, prims, x, cover_h[0], gbox.p, morton_sorted.p, sorted_to_orig, children.p,
                                    object_idx.p, parent.p, tcount.p, leaf_of.p);
        };
        if (n <= 4096u) go(k_build_small<4>);
        else go(k_build_small<8>);
        finish(s);
        return;
    }
    k_init_gbox<<<grid_for(6 * nseg, kBlock), kBlock, 0, s>>>(gbox.p, nseg);
    k_leaf_centers<<<grid_for(n, kBlock), kBlock, 0, s>>>(n, arity, prims, x, seg_of_leaf.p, seg_tab.p, center.p, gbox.p);
    k_morton<<<grid_for(n, kBlock), kBlock, 0, s>>>(n, center.p, seg_of_leaf.p, gbox.p, keys[0].p, vals[0].p);
    int cur = 0;
    // four passes over the Morton key, then (several segments) passes over the segment id
    for (int shift = 0; shift < 32; shift += 8)
    {
        sort_pass(n, shift, keys[cur].p, keys[cur].p, vals[cur].p, keys[1 - cur].p, vals[1 - cur].p, nullptr, nullptr,
                  hist.p, scan_tmp.p, s);
        cur = 1 - cur;
    }
    if (nseg > 1)
    {
        k_seg_keys<<<grid_for(n, kBlock), kBlock, 0, s>>>(n, vals[cur].p, seg_of_leaf.p, khi[cur].p);
        for (int shift = 0; shift < 32 && ((nseg - 1) >> shift) != 0u; shift += 8)
        {
            sort_pass(n, shift, khi[cur].p, keys[cur].p, vals[cur].p, keys[1 - cur].p, vals[1 - cur].p, khi[cur].p,
                      khi[1 - cur].p, hist.p, scan_tmp.p, s);
            cur = 1 - cur;
        }
    }
    sorted_to_orig = vals[cur].p;
    k_leaves<<<grid_for(n, kBlock), kBlock, 0, s>>>(n, ni, keys[cur].p, vals[cur].p, seg_of_leaf.p, seg_tab.p,
                                                    morton_sorted.p, children.p, object_idx.p, parent.p, leaf_of.p);
    k_fill_u32<<<1, kBlock, 0, s>>>(tcount.p, 2u, 0u);
    finish(s);
}

// From the sorted leaves (and tcount zeroed): the inner nodes, and the split into treelets and the
// nodes above them. One tree of up to kUncounted leaves stays off the host: its treelets and top nodes
// are counted on the device (about 2.5 and 1.5 per 1024 leaves on the cloth meshes, far from kTopLds).
// Larger trees and batches read the two counts back, since a top beyond kTopLds is refit with one
// launch per level.
void Lbvh::finish(hipStream_t s)
{
    if (ni == 0)
    {
        LCSX_HIP(hipGetLastError());
        return;
    }
    k_karras<<<grid_for(ni, kBlock), kBlock, 0, s>>>(ni, morton_sorted.p, inner_seg.p, seg_tab.p, parent.p, children.p,
                                                     object_idx.p, tsize.p, tfirst.p, tleaf.p);
    k_treelet_mark<<<grid_for(ni, kBlock), kBlock, 0, s>>>(ni, parent.p, tsize.p, kTreeletLeaves, tcount.p, troots.p,
                                                           top_list.p);
    counted = !(nseg == 1 && n <= kUncounted);
    ntop = ntreelets = 0;
    if (counted)
    {
        uint32_t nt[2] = {0u, 0u};
        LCSX_HIP(hipMemcpyAsync(nt, tcount.p, 2 * sizeof(uint32_t), hipMemcpyDeviceToHost, s));
        LCSX_HIP(hipStreamSynchronize(s));
        ntreelets = nt[0];
        ntop      = nt[1];
    }
    top_lvp_h.clear();
    if (n > kTreeletLeaves && (!counted || ntop))
    {
        k_top_sort<<<1, 1024, 0, s>>>(tcount.p, parent.p, top_list.p, top_depth.p, top_order.p, top_idx.p, top_level_ptr.p);
        k_top_children<<<counted ? grid_for(ntop, kBlock) : 16u, kBlock, 0, s>>>(
            ni, top_order.p, tcount.p + 1, children.p, tsize.p, kTreeletLeaves, top_idx.p, top_child.p);
        if (ntop > kTopLds)
        {
            top_lvp_h.assign(kMaxLevels + 1, 0u);
            LCSX_HIP(hipMemcpyAsync(top_lvp_h.data(), top_level_ptr.p, (kMaxLevels + 1) * sizeof(uint32_t),
                                    hipMemcpyDeviceToHost, s));
            LCSX_HIP(hipStreamSynchronize(s));
        }
    }
    LCSX_HIP(hipGetLastError());
}

void Lbvh::refit(const float* x0, const float* x1, const float* pad, hipStream_t s, bool wide)
{
    if (n == 0) return;
    k_refit_leaves<<<grid_for(n, kBlock), kBlock, 0, s>>>(n, ni, arity, prims, sorted_to_orig, x0, x1, pad, nodes.p);
    if (ni == 0) return;
    float4* const p4 = wide ? packed4.p : nullptr;
    // uncounted: about one workgroup per treelet, each taking every grid-th one
    const uint32_t tgrid = counted ? ntreelets : n / 384u + 1u;
    if (tgrid)
        k_refit_treelets<<<tgrid, kTreeletBlock, 0, s>>>(tcount.p, troots.p, tsize.p, tfirst.p, tleaf.p, parent.p, ni,
                                                         children.p, nodes.p, packed.p, p4, sorted_keys);
    // the nodes above the treelets (none up to kTreeletLeaves leaves): the levels nearest the roots that one
    // workgroup's LDS holds together in one launch, the levels below them one by one before it (24 scenes:
    // 58 us of launches per refit where every level had its own, now 25)
    if (n > kTreeletLeaves && (!counted || ntop))
    {
        uint32_t levels = kMaxLevels;
        if (counted && ntop > kTopLds)
            for (; top_lvp_h[levels] > kTopLds; levels--)
            {
                const uint32_t b = top_lvp_h[levels - 1], e = top_lvp_h[levels];
                if (e > b)
                    k_refit_range<<<grid_for(e - b, kBlock), kBlock, 0, s>>>(top_order.p + b, e - b, ni, children.p, nodes.p,
                                                                             packed.p, p4, sorted_keys);
            }
        if (levels)
            k_refit_top<<<1, 1024, 0, s>>>(top_order.p, top_level_ptr.p, levels - 1u, ni, top_child.p, children.p, nodes.p,
                                           packed.p, p4, sorted_keys);
    }
    LCSX_HIP(hipGetLastError());
    wide_ready = wide;
}

uint32_t sort_hist_words(uint32_t n)
{
    // for any count up to n: a count with smaller tiles has more of them
    auto words = [](uint32_t k) {
        const uint32_t tile = (uint32_t)(kBlock * sort_items(k));
        return 256u * ((k + tile - 1u) / tile) + 1u;
    };
    return std::max({words(n), words(std::min(n, kSort4)), words(std::min(n, kSort8))});
}

int launch_sort_key_pairs(uint32_t* lo[2], uint32_t* hi[2], uint32_t* val[2], uint32_t n, int lo_bits, int hi_bits,
                          uint32_t* hist, uint32_t* tmp, hipStream_t s)
{
    int cur = 0;
    if (n == 0) return cur;
    // the low key's digits, then the high key's (stable passes: the result is ordered by (hi, lo))
    for (int pass = 0; pass < 2; pass++)
    {
        const int bits = pass == 0 ? lo_bits : hi_bits;
        for (int shift = 0; shift < bits; shift += 8)
        {
            const uint32_t* dig = pass == 0 ? lo[cur] : hi[cur];
            sort_pass(n, shift, dig, lo[cur], val[cur], lo[1 - cur], val[1 - cur], hi[cur], hi[1 - cur], hist, tmp, s);
            cur = 1 - cur;
        }
    }
    LCSX_HIP(hipGetLastError());
    return cur;
}

void lbvh_query(const Lbvh& t, const QueryArgs& a, hipStream_t s)
{
    if (t.n == 0 || a.n_queries == 0) return;
    int v = a.variant >= 0 && a.variant < kQueryVariants ? a.variant : kQueryDefault;
    // the shapes that share a query among lanes read their boxes; vertices and edges take one lane each, with as
    // many stack entries
    if (kQueryShapes[v].lanes >= 2 && a.mode != QueryBoxes) v = kQueryElements;
    // 4-wide records exist after a level-ordered refit; otherwise the binary shape with the same
    // LDS stack and staging
    if (kQueryShapes[v].wide >= 4 && !t.wide_ready) v = kQueryShapes[v].lds_stack >= 16 ? 1 : 3;
    const QueryShape Q    = kQueryShapes[v];
    const uint32_t   per  = kQueryBlock / Q.lanes;  // queries per block
    const uint32_t   grid = (a.n_queries + per - 1) / per;
    const int        st   = Q.wide == 2 ? kStack : 2 * kStack;  // stack entries
    const size_t     need = (size_t)(st - Q.lds_stack) * grid * per;
    if (need > t.spill.n) t.spill.alloc(need);
    switch (v)
    {
    case 0: launch_query_shape<0>(t, a, grid, s); break;
    case 1: launch_query_shape<1>(t, a, grid, s); break;
    case 2: launch_query_shape<2>(t, a, grid, s); break;
    case 3: launch_query_shape<3>(t, a, grid, s); break;
    case 4: launch_query_shape<4>(t, a, grid, s); break;
    case 5: launch_query_shape<5>(t, a, grid, s); break;
    case 6: launch_query_shape<6>(t, a, grid, s); break;
    case 7: launch_query_shape<7>(t, a, grid, s); break;
    case 8: launch_query_shape<8>(t, a, grid, s); break;
    default: launch_query_shape<9>(t, a, grid, s); break;
    }
    LCSX_HIP(hipGetLastError());
}

bool query_by_clusters(int variant)
{
    const int v = variant >= 0 && variant < kQueryVariants ? variant : kQueryDefault;
    return kQueryShapes[v].lanes >= 2;
}

void ClusterTree::init(int arity_, const uint32_t* device_prims, const std::vector<uint32_t>& order,
                       const std::vector<uint32_t>& scene_block_, hipStream_t s)
{
    arity  = arity_;
    prims  = device_prims;
    blocks = (uint32_t)(order.size() / kClusterLeaves);
    if (blocks > 0xffffffffu / (8u * kClusterRecords))  // records are addressed in 32 bits
    {
        set_error("broad phase: too many elements");
        throw CapacityFailure();
    }
    elem.upload(order, s);
    scene_block.upload(scene_block_, s);
    if (!blocks) return;
    rec.alloc(8 * (size_t)kClusterRecords * blocks);
    top.alloc(2 * (size_t)blocks);
}

void ClusterTree::refit(const float* x0, const float* x1, const float* pad, const uint32_t* leaf_of, hipStream_t s)
{
    if (!blocks) return;
    k_cluster_refit<<<blocks, 256, 0, s>>>(arity, prims, elem.p, leaf_of, x0, x1, pad, rec.p, top.p);
    LCSX_HIP(hipGetLastError());
}

void ClusterTree::query(const ClusterQuery& a, const uint32_t* leaf_of, hipStream_t s) const
{
    if (!blocks || !a.n) return;
    const uint32_t per  = kGroup * kGroupWaves;  // queries of a block
    const uint32_t grid = (a.n + per - 1) / per;
    if (a.edges) k_query_group<true><<<grid, 64 * kGroupWaves, 0, s>>>(a, rec.p, top.p, scene_block.p, leaf_of);
    else k_query_group<false><<<grid, 64 * kGroupWaves, 0, s>>>(a, rec.p, top.p, scene_block.p, leaf_of);
    LCSX_HIP(hipGetLastError());
}

}  // namespace lcsx
