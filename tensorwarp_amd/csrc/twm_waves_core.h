// Device helpers of the kernels for 5 .. 32 rows with exact weights (twm_waves_exact.hip, twm_batch_range.hip).
#pragma once
#include "twm_device.h"

namespace twm {

namespace {

__device__ __forceinline__ const TWM_GLOBAL char *we_scalar_base(const void *p, size_t byte_offset)
{
    uint64_t v = (uint64_t)p + byte_offset;
    asm("" : "+s"(v));  // a uniform base kept in scalar registers: loads take saddr + 32-bit lane offset
    return (const TWM_GLOBAL char *)v;
}

struct WeConsts {
    uint32_t mask_lo, mask_hi, magic_lo, magic_hi;
};

// eight nibbles of word w -> eight f16 values (q - 8), exact
__device__ __forceinline__ half8 we_unpack(uint32_t w, const WeConsts &c)
{
    union { uint32_t u[4]; half2v h2[4]; half8 h; } r;
    const half2v b_lo = {(_Float16)-1032.0f, (_Float16)-1032.0f};
    const half2v b_hi = {(_Float16)-72.0f, (_Float16)-72.0f};
    const uint32_t w8 = w >> 8;
    r.u[0] = (w & c.mask_lo) | c.magic_lo;
    r.u[1] = (w & c.mask_hi) | c.magic_hi;
    r.u[2] = (w8 & c.mask_lo) | c.magic_lo;
    r.u[3] = (w8 & c.mask_hi) | c.magic_hi;
    r.h2[0] += b_lo;
    r.h2[1] += b_hi;
    r.h2[2] += b_lo;
    r.h2[3] += b_hi;
    return r.h;
}

constexpr int kWeRow = 128;  // halves per LDS row (256 bytes)

// What kind of rows: f16; up to eight f32 rows, whose second f16 terms are rows 8 .. 15 of the one block (which costs what
// eight f16 rows cost); f32 rows as two tiles
enum { kRowsF16 = 0, kRowsF32Few = 1, kRowsF32 = 2 };

// the largest magnitude of eight values
__device__ __forceinline__ float we_max8(const uint4v &a, const uint4v &b)
{
    float x[8], t;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        x[q] = __uint_as_float(a[q]);
        x[4 + q] = __uint_as_float(b[q]);
    }
    asm("v_max3_f32 %0, |%1|, |%2|, |%3|" : "=v"(t) : "v"(x[0]), "v"(x[1]), "v"(x[2]));
    asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(t) : "v"(t), "v"(x[3]), "v"(x[4]));
    asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(t) : "v"(t), "v"(x[5]), "v"(x[6]));
    asm("v_max_f32 %0, %1, |%2|" : "=v"(t) : "v"(t), "v"(x[7]));
    return t;
}

// The power of two that brings a largest magnitude to [2^13, 2^14), and its inverse.  (An infinity or a NaN stays one.)
struct WeFactor {
    float down, back;
};
__device__ __forceinline__ WeFactor we_factor(float largest)
{
    uint32_t e = __float_as_uint(largest) & 0x7F800000u;
    e = e > (16u << 23) ? e : (16u << 23);
    return WeFactor{__uint_as_float((267u << 23) - e), __uint_as_float(e - (13u << 23))};
}

// four f32 values as two f16 terms each: hi = f16(x * down), lo = f16(x * down - hi)
__device__ __forceinline__ void we_terms(const uint4v &a, float down, uint2v &hi_out, uint2v &lo_out)
{
    union { half2v h[2]; uint2v u; } hi, lo;
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const float f0 = __uint_as_float(a[2 * q]), f1 = __uint_as_float(a[2 * q + 1]);
        hi.h[q] = half2v{(_Float16)(f0 * down), (_Float16)(f1 * down)};
        asm("" : "+v"(hi.u[q]));        // (one conversion of the pair; its halves are read from the packed register)
        float r0 = __builtin_fmaf(f0, down, -(float)hi.h[q][0]), r1 = __builtin_fmaf(f1, down, -(float)hi.h[q][1]);
        asm("" : "+v"(r0), "+v"(r1));   // (v_fma_mixlo_f16, which would do both steps, issues at half the rate)
        lo.h[q] = half2v{(_Float16)r0, (_Float16)r1};
    }
    hi_out = hi.u;
    lo_out = lo.u;
}

}  // namespace

}  // namespace twm
