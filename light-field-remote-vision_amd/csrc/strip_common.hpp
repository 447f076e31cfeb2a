// Pieces of the marching-strip kernels (k_sr.hip, k_cg.hip): a wave owns a
// strip of 64 columns with its halo and walks down its rows.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <type_traits>

namespace lfrv {

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>)
template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for(F &&f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>());
        static_for<N, I + 1>(f);
    }
}

constexpr int kStripGroup = 3;  // rows per turn of the loop

// The lane's left (x - 1) / right (x + 1) neighbour's value, 0 past the wave
// (every lane has to take part: never inside a select).
__device__ __forceinline__ float from_left(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));  // wave_shr:1
}
__device__ __forceinline__ float from_right(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));  // wave_shl:1
}

// v where the mask is -1, and 0, whatever v, where it is 0.  A mask is one register where a condition is a pair of
// the scalar ones, of which the strips have none to spare; the compiler is kept from seeing the condition in it.
__device__ __forceinline__ float where(int mask, float v) { return __int_as_float(__float_as_int(v) & mask); }
__device__ __forceinline__ int lane_mask(bool in)
{
    int m = in ? -1 : 0;
    asm("" : "+v"(m));
    return m;
}
__device__ __forceinline__ int mask_below(int y, int end) { return (~y & (y - end)) >> 31; }  // of 0 <= y < end

// a b, rounded: not to be contracted with a sum that it goes into (where the product is also stored, the sum is of
// what is stored).
__device__ __forceinline__ float product(float a, float b)
{
#pragma clang fp contract(off)
    return a * b;
}

constexpr int kOutside = (int)0x80000000;
constexpr size_t kNarrowBytes = (size_t)1 << 31;  // kOutside lies past any buffer below this size
constexpr int kStripOverrun = 16;  // a strip names fewer rows than this past its planes (with kOutside)

// Whether the strips need a descriptor per row: where the scalar offset of a
// row past the last of `planes` planes of h rows of w values would reach
// `limit` (kNarrowBytes; int arithmetic, and added to kOutside it would wrap).
constexpr bool strip_wide(int planes, int w, int h, size_t limit)
{
    return 4 * (size_t)w * ((size_t)planes * h + kStripOverrun) >= limit;
}
static_assert(strip_wide(5, 10361, 10363, kNarrowBytes),
              "planes that fit one descriptor, the rows past whose end overflow the offset");
static_assert(!strip_wide(5, 10360, 10363 - kStripOverrun, kNarrowBytes) &&
                  4ll * (4 * 10360ll * (10363 - kStripOverrun) + 10360ll * 10363) < (1ll << 31),
              "the largest narrow planes");

// Planes of `w`-wide rows, `stride` values apart.  Narrow: one descriptor for
// all of them (unless strip_wide), the row and plane in the scalar offset.
// WIDE: a descriptor per row.
template <bool WIDE>
struct Planes {
    const float *base;
    size_t stride;
    int w;
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ Planes(const float *b, int n, size_t st, int width) : base(b), stride(st), w(width)
    {
        if constexpr (!WIDE) r = __builtin_amdgcn_make_buffer_rsrc((void *)b, 0, b ? (int)(4 * n * st) : 0, 0x00020000);
    }
    // plane c, row y (clamped at 0; a row outside comes with vo = kOutside)
    __device__ __forceinline__ float load(int c, int y, int vo) const
    {
        if constexpr (WIDE) return __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(row(c, y), vo, 0, 0));
        else return __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, vo, 4 * (c * (int)stride + max(y, 0) * w), 0));
    }
    __device__ __forceinline__ void store(float v, int c, int y, int vo) const
    {
        if constexpr (WIDE) __builtin_amdgcn_raw_buffer_store_b32(__float_as_int(v), row(c, y), vo, 0, 0);
        else __builtin_amdgcn_raw_buffer_store_b32(__float_as_int(v), r, vo, 4 * (c * (int)stride + max(y, 0) * w), 0);
    }
    __device__ __forceinline__ __amdgpu_buffer_rsrc_t row(int c, int y) const
    {
        return __builtin_amdgcn_make_buffer_rsrc((void *)(base + c * stride + (size_t)max(y, 0) * w), 0, base ? 4 * w : 0,
                                                 0x00020000);
    }
};

// n / d, correctly rounded but for quotients and dividends within some 2^24 of
// the smallest normal number (an ulp there): a Newton step for the reciprocal,
// which several quotients of one divisor share, then two for the quotient.
// Divisors away from 1 are brought there by a power of two, and the fix-up
// gives what division gives for zeros, infinities and NaN, and where it overflows.
struct Divisor {
    float d, r, scale;
    __device__ __forceinline__ explicit Divisor(float div)
        : Divisor(div, fabsf(div) < 0x1p-64f ? 0x1p64f : fabsf(div) > 0x1p64f ? 0x1p-64f : 1.0f)
    {
    }
    __device__ __forceinline__ Divisor(float div, float sc) : d(div * sc), scale(sc)
    {
        r = __builtin_amdgcn_rcpf(d);
        r = fmaf(fmaf(-d, r, 1.0f), r, r);
    }
    // whether a divisor can go without a scale: between 2^-126 and 2^125
    __device__ __forceinline__ static bool plain(float div)
    {
        return (unsigned)(__float_as_int(div) - 0x00800000) < 0x7d800000u;
    }
    // the quotient of n / scale (which the caller knows to be 1, or has multiplied into n)
    __device__ __forceinline__ float of_scaled(float n) const
    {
        float q = n * r;
        q = fmaf(fmaf(-d, q, n), r, q);
        return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q, n), r, q), d, n);
    }
};

// n / d for d = 1, 2, 3 or 4 and r = 1 / d: with a rounded reciprocal one correction rounds the quotient (checked for
// every mantissa of n, for n above 2^-102).
__device__ __forceinline__ float small_quotient(float n, float d, float r)
{
    const float q = n * r;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q, n), r, q), d, n);
}

}  // namespace lfrv
