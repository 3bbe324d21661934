// Shared device/host helpers for the lcsx HIP kernels (gfx950, wave64).
//
// All kernels are compiled with -ffp-contract=off: every floating-point expression below is
// evaluated exactly in the written order (left to right), which is what makes the per-element
// results reproducible bit for bit.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define LCSX_HD __host__ __device__ __forceinline__
#define LCSX_D __device__ __forceinline__

namespace lcsx
{

constexpr float kEpsilon        = 1.19209290E-7f;  // FLT_EPSILON (reference Core/constant_value.h:12)
constexpr float kLineSearchMaxT = 1.25f;           // ACCD step cap (reference accd.hpp:47)
constexpr float kCcdReduction   = 0.01f;           // ACCD gap reduction (reference accd.hpp:46)
constexpr uint32_t kInvalid     = 0xffffffffu;
constexpr uint32_t kClusterLeaves = 1024;  // positions of a block of the solver's hierarchies (ClusterTree)

struct f3
{
    float x, y, z;
};
LCSX_HD f3 mk(float a, float b, float c) { return f3{a, b, c}; }
LCSX_HD f3 operator+(f3 a, f3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
LCSX_HD f3 operator-(f3 a, f3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
LCSX_HD f3 operator-(f3 a) { return {-a.x, -a.y, -a.z}; }
LCSX_HD f3 operator*(float s, f3 a) { return {s * a.x, s * a.y, s * a.z}; }
LCSX_HD f3 operator*(f3 a, float s) { return {a.x * s, a.y * s, a.z * s}; }
LCSX_HD f3 operator/(f3 a, float s) { return {a.x / s, a.y / s, a.z / s}; }
LCSX_HD float dot(f3 a, f3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
LCSX_HD f3 cross(f3 a, f3 b) { return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x}; }
LCSX_HD float length(f3 a) { return sqrtf(dot(a, a)); }
LCSX_HD f3 normalize(f3 a) { return a * (1.0f / length(a)); }
// min/max with std::min / std::max semantics ((b < a) ? b : a), so signed zeros and ties
// resolve the same way on the device and on the host.
LCSX_HD float smin(float a, float b) { return (b < a) ? b : a; }
LCSX_HD float smax(float a, float b) { return (a < b) ? b : a; }
LCSX_HD f3 vmin(f3 a, f3 b) { return {smin(a.x, b.x), smin(a.y, b.y), smin(a.z, b.z)}; }
LCSX_HD f3 vmax(f3 a, f3 b) { return {smax(a.x, b.x), smax(a.y, b.y), smax(a.z, b.z)}; }
LCSX_HD float clampf(float v, float lo, float hi) { return smax(smin(v, hi), lo); }
LCSX_HD float get(f3 a, int i) { return i == 0 ? a.x : (i == 1 ? a.y : a.z); }

LCSX_HD f3 ld3(const float* p, uint32_t i) { return {p[3 * (size_t)i], p[3 * (size_t)i + 1], p[3 * (size_t)i + 2]}; }
LCSX_HD void st3(float* p, uint32_t i, f3 v)
{
    p[3 * (size_t)i]     = v.x;
    p[3 * (size_t)i + 1] = v.y;
    p[3 * (size_t)i + 2] = v.z;
}

// Row-major 3x3.
struct m3
{
    float m[9];
};
LCSX_HD m3 m3_zero()
{
    m3 a;
    for (int i = 0; i < 9; i++) a.m[i] = 0.0f;
    return a;
}
LCSX_HD f3 mul(const m3& a, f3 x)
{
    return {a.m[0] * x.x + a.m[1] * x.y + a.m[2] * x.z, a.m[3] * x.x + a.m[4] * x.y + a.m[5] * x.z,
            a.m[6] * x.x + a.m[7] * x.y + a.m[8] * x.z};
}

// ---------------------------------------------------------------- ordered float atomics
// Map a float to an unsigned key with the same order (used for global min/max of AABBs
// and of step bounds; min/max is order-independent, so the result is deterministic).
LCSX_HD uint32_t f2ord(float f)
{
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
LCSX_HD float ord2f(uint32_t u) { return __builtin_bit_cast(float, (u & 0x80000000u) ? (u & 0x7fffffffu) : ~u); }
LCSX_HD unsigned long long d2ord(double d)
{
    unsigned long long u = __builtin_bit_cast(unsigned long long, d);
    return (u >> 63) ? ~u : (u | (1ull << 63));
}
LCSX_HD double ord2d(unsigned long long u)
{
    return __builtin_bit_cast(double, (u >> 63) ? (u & ~(1ull << 63)) : ~u);
}

// ---------------------------------------------------------------- wave64 primitives
LCSX_D uint32_t lane_id() { return __lane_id(); }
LCSX_D uint64_t lanemask_lt() { return (1ull << __lane_id()) - 1ull; }

// List counters saturate near kCountCeil: a reservation that finds the counter at or past it
// takes its amount back, so a counter never wraps (it stays below kCountCeil plus what the waves
// in flight add at once) and a host reading >= kCountCeil knows the list overflowed beyond any
// capacity (capacities stay below kCountCeil).
constexpr uint32_t kCountCeil = 0x80000000u;

// Capacity of a list after `need` entries did not fit in `cap`: 1.5 x need, at least cap, at most
// limit. 0 when the need cannot be met: above the limit, or at the counters' saturation point
// (the true count is then unknown).
inline uint64_t grown_capacity(uint64_t cap, uint64_t need, uint64_t limit)
{
    if (need >= kCountCeil || need > limit) return 0;
    const uint64_t g = need + need / 2;
    const uint64_t c = cap < g ? g : cap;
    return c < limit ? c : limit;
}
LCSX_D uint32_t count_reserve(uint32_t* counter, uint32_t k)
{
    uint32_t base = atomicAdd(counter, k);
    if (base >= kCountCeil) atomicSub(counter, k);
    return base;
}

// Appends `pred` lanes to a global list with one atomic per wave; returns this lane's slot.
LCSX_D uint32_t wave_append(uint32_t* counter, bool pred)
{
    uint64_t mask = __ballot(pred);
    if (mask == 0) return 0;
    int      leader = __ffsll((unsigned long long)mask) - 1;
    uint32_t base   = 0;
    if ((int)lane_id() == leader) base = count_reserve(counter, (uint32_t)__popcll(mask));
    base = __shfl(base, leader);
    return base + (uint32_t)__popcll(mask & lanemask_lt());
}

// v + (v of the lane whose index differs in bit O), without a trip through LDS: rows and halves of
// the wavefront are swapped by v_permlane16/32_swap, lanes within a row of 16 by DPP. Addition
// commutes, so both lanes of a pair get the same bits as from __shfl_xor.
template <int O>
LCSX_D float xor_add(float v)
{
    const int i = __float_as_int(v);
    if constexpr (O == 32 || O == 16)
    {
        const auto r = O == 32 ? __builtin_amdgcn_permlane32_swap(i, i, false, false)
                               : __builtin_amdgcn_permlane16_swap(i, i, false, false);
        return __int_as_float((int)r[0]) + __int_as_float((int)r[1]);
    }
    else
    {
        int o;
        if constexpr (O == 8) o = __builtin_amdgcn_mov_dpp(i, 0x128, 0xf, 0xf, true);  // row_ror:8
        else if constexpr (O == 4)
        {
            // row_half_mirror (lane ^ 7), then quad_perm [3, 2, 1, 0] (lane ^ 3)
            o = __builtin_amdgcn_mov_dpp(i, 0x141, 0xf, 0xf, true);
            o = __builtin_amdgcn_mov_dpp(o, 0x1b, 0xf, 0xf, true);
        }
        else if constexpr (O == 2) o = __builtin_amdgcn_mov_dpp(i, 0x4e, 0xf, 0xf, true);  // [2, 3, 0, 1]
        else o = __builtin_amdgcn_mov_dpp(i, 0xb1, 0xf, 0xf, true);                        // [1, 0, 3, 2]
        return v + __int_as_float(o);
    }
}
template <int O>
LCSX_D f3 xor_add(f3 v)
{
    return {xor_add<O>(v.x), xor_add<O>(v.y), xor_add<O>(v.z)};
}
template <class T>
LCSX_D T wave_sum(T v)
{
    for (int o = 32; o > 0; o >>= 1) v = v + __shfl_xor(v, o);
    return v;
}
LCSX_D float wave_sum(float v)
{
    return xor_add<1>(xor_add<2>(xor_add<4>(xor_add<8>(xor_add<16>(xor_add<32>(v))))));
}
LCSX_D float wave_min(float v)
{
    for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o));
    return v;
}
LCSX_D float wave_max(float v)
{
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}

inline unsigned grid_for(size_t n, unsigned block) { return (unsigned)((n + block - 1) / block); }

// Work block of launch block b when a launch of n blocks is spread over the 8 XCDs of the part:
// workgroups are dispatched to the XCDs in turn (b mod 8), so XCD x gets the contiguous range of
// work blocks [x q + min(x, r), ...) with q = n / 8, r = n mod 8 (a bijection of [0, n)). Data
// that neighbouring work blocks share (gathered rows, BVH subtrees of nearby queries) then stays
// in one XCD's L2 instead of being fetched by all eight.
LCSX_D uint32_t xcd_block(uint32_t b, uint32_t n)
{
    const uint32_t x = b & 7u, idx = b >> 3, q = n >> 3, r = n & 7u;
    return x < r ? x * (q + 1u) + idx : r * (q + 1u) + (x - r) * q + idx;
}

}  // namespace lcsx
