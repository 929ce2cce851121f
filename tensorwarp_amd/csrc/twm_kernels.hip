// gfx950 (CDNA4, wave64) kernels for the TW-Marlin W4A16 quantized-linear path.
//
// Reference semantics (crates/kernels/src/quantize.rs in the reference checkout):
//   GEMV arithmetic ............ :1186-1298   (warp_gemm_tw_marlin_m1[_direct])
//   Q4 unpack to FP16 .......... :534-571     (warp_dequant_q4_to_f16)
//   quantizer .................. :414-474, crates/loader/src/gemma_moe_q4.rs:218-254
//   reorder / fuse ............. :912-956, :1018-1063
//   split_qkv / split_gate_up .. crates/kernels/src/ops.rs:2255-2297
// This file holds the format operations, the GEMV on the reference layout and the repacks into
// the two streaming orders; the MFMA kernels that stream the repacked weights are in twm_gemv4*.hip,
// twm_stream.hip, twm_batch.hip and twm_prefill.hip.
#include "twm_device.h"

namespace twm {

__device__ __forceinline__ float f16_bits_to_f32(uint16_t h)
{
    union { uint16_t u; _Float16 f; } x;
    x.u = h;
    return (float)x.f;  // v_cvt_f32_f16: exact, subnormals kept
}

// scale * q for the Q4 unpack.  The value is pinned in a register between the convert and the
// multiply: left alone, the compiler folds both into v_fma_mix*(s, q, +0), and x*y + (+0) turns
// the product -0.0 (zero scale, negative q) into +0.0, which is not the reference's bit pattern.
__device__ __forceinline__ float scale_times_q(uint16_t scale_bits, int q)
{
    float s = f16_bits_to_f32(scale_bits);
    asm volatile("" : "+v"(s));
    float w = s * (float)q;
    asm volatile("" : "+v"(w));
    return w;
}

__device__ __forceinline__ uint16_t f32_to_f16_bits(float f)
{
    union { uint16_t u; _Float16 h; } x;
    x.h = (_Float16)f;  // v_cvt_f16_f32: round to nearest even
    return x.u;
}

// ---------------------------------------------------------------------------------
// fill
// ---------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_fill_zero(uint32_t *p, size_t words)
{
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    size_t stride = (size_t)gridDim.x * 256;
    for (; i < words; i += stride) p[i] = 0u;
}

hipError_t launch_fill_zero(hipStream_t s, void *ptr, size_t bytes)
{
    size_t words = bytes / 4;
    if (words == 0) return hipSuccess;
    size_t blocks = (words + 255) / 256;
    if (blocks > 2048) blocks = 2048;
    hipLaunchKernelGGL(k_fill_zero, dim3((unsigned)blocks), dim3(256), 0, s, (uint32_t *)ptr, words);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------
// casts between f32 and f16 rows (crates/kernels/src/fp16.rs:133-166): round to nearest even, as __float2half
// ---------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_cast_f32_f16(const float *__restrict__ src, _Float16 *__restrict__ dst, size_t count)
{
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    size_t stride = (size_t)gridDim.x * 256;
    for (; i < count; i += stride) dst[i] = (_Float16)src[i];
}
__global__ __launch_bounds__(256) void k_cast_f16_f32(const _Float16 *__restrict__ src, float *__restrict__ dst, size_t count)
{
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    size_t stride = (size_t)gridDim.x * 256;
    for (; i < count; i += stride) dst[i] = (float)src[i];
}

hipError_t launch_cast(hipStream_t s, const void *src, void *dst, size_t count, bool to_f16)
{
    if (count == 0) return hipSuccess;
    size_t blocks = (count + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    if (to_f16) hipLaunchKernelGGL(k_cast_f32_f16, dim3((unsigned)blocks), dim3(256), 0, s, (const float *)src, (_Float16 *)dst, count);
    else hipLaunchKernelGGL(k_cast_f16_f32, dim3((unsigned)blocks), dim3(256), 0, s, (const _Float16 *)src, (float *)dst, count);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------
// quantizer: one thread per (group, column)
// ---------------------------------------------------------------------------------
struct QGroup {
    float scale;
    uint32_t w[4];
};

// One thread per (group, column) of a matrix, columns next to each other, groups one after the other without a gap whatever
// the width: blockIdx.x counts the places of `slab` groups, as many as 31 bits index, and blockIdx.y the slabs, so that a
// thread divides 32 bits and not 64.  (A workgroup on 256 columns of one group leaves most of its threads idle on narrow
// matrices and behind the last 256 columns: 1048576 x 1 quantized 20.4 us, now 7.0, 18944 x 260 7.0, now 5.0.)
struct Place {
    uint32_t group, column;
};
__device__ __forceinline__ bool place_of(uint32_t groups, uint32_t columns, uint32_t slab, Place &p)
{
    const uint32_t at = blockIdx.x * 256u + threadIdx.x, q = at / columns;
    p.group = blockIdx.y * slab + q;
    p.column = at - q * columns;
    return q < slab && p.group < groups;
}
static uint32_t place_slab(uint32_t groups, uint32_t columns)
{
    const uint32_t most = columns < 0x80000000u ? 0x7FFFFFFFu / columns : 1u;
    return groups < most ? groups : most;
}
static dim3 place_grid(uint32_t groups, uint32_t columns)
{
    const uint32_t slab = place_slab(groups, columns);
    return dim3((unsigned)(((uint64_t)slab * columns + 255) / 256), (groups + slab - 1) / slab);
}

// The general form: any values, NaN and infinity among them.
__device__ __forceinline__ void quantize_words(const float *vals, float inv, uint32_t *w)
{
#pragma unroll
    for (int wi = 0; wi < 4; wi++) {
        uint32_t word = 0;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            float rv = roundf(vals[wi * 8 + j] * inv);     // half away from zero
            int q = (rv != rv) ? 0 : (int)fminf(fmaxf(rv, -64.0f), 64.0f);
            q += 8;
            q = q < 0 ? 0 : (q > 15 ? 15 : q);
            word |= (uint32_t)q << (4 * j);
        }
        w[wi] = word;
    }
}

// Finite values and a finite factor: |x| <= 7 (1 + 2^-23), so the rounded value is -7 .. 7 and needs no clamp.  Half away
// from zero is the integer part of x + 0.49999997 with x's sign (the largest f32 below a half: x = 0.5 still reaches 1 by
// the sum's own rounding and 0.49999997 does not), which leaves five instructions per value instead of about fourteen.
__device__ __forceinline__ void quantize_words_finite(const float *vals, float inv, uint32_t *w)
{
#pragma clang fp contract(off)
#pragma unroll
    for (int wi = 0; wi < 4; wi++) {
        uint32_t word = 0x88888888u;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float x = vals[wi * 8 + j] * inv;
            const int r = (int)(x + copysignf(0.49999997f, x));
            word += (uint32_t)r << (4 * j);
        }
        w[wi] = word;
    }
}

__device__ __forceinline__ QGroup quantize_group32(const float *vals)
{
    float amax = 0.0f;
    bool odd = false;  // an infinity or a NaN
#pragma unroll
    for (int i = 0; i < 32; i++) {
        float a = fabsf(vals[i]);
        odd = odd || !(a <= 3.40282347e38f);
        if (a > amax) amax = a;  // NaN never wins, as with Rust's f32::max fold
    }
    QGroup r;
    r.scale = amax / 7.0f;                                 // correctly rounded division
    float inv = (r.scale != 0.0f) ? 7.0f / amax : 0.0f;
    odd = odd || !(inv <= 3.40282347e38f);
    if (__builtin_amdgcn_ballot_w64(odd) != 0) quantize_words(vals, inv, r.w);
    else quantize_words_finite(vals, inv, r.w);
    return r;
}

// One thread per (group, column) of a [K,N] matrix: lanes take neighbouring columns.
__global__ __launch_bounds__(256) void k_quantize_q4_0(const float *__restrict__ w, uint32_t k, uint32_t n,
                                                        uint8_t *__restrict__ q4, uint32_t slab)
{
    const uint32_t groups = k / 32;
    Place at;
    if (!place_of(groups, n, slab, at)) return;
    const uint32_t g = at.group, col = at.column;
    float vals[32];
#pragma unroll
    for (int i = 0; i < 32; i++) vals[i] = w[((size_t)g * 32 + i) * n + col];
    QGroup r = quantize_group32(vals);
    uint32_t *dst = (uint32_t *)(q4 + ((size_t)col * groups + g) * 20);  // 20-byte blocks are 4-byte aligned
    dst[0] = __float_as_uint(r.scale);
    dst[1] = r.w[0]; dst[2] = r.w[1]; dst[3] = r.w[2]; dst[4] = r.w[3];
}

__global__ __launch_bounds__(256) void k_quantize_twm_kn(const float *__restrict__ w, uint32_t groups, uint32_t n, uint4v *__restrict__ packed,
                                                          uint16_t *__restrict__ scales, uint32_t slab)
{
    Place at;
    if (!place_of(groups, n, slab, at)) return;
    const uint32_t g = at.group, col = at.column;
    float vals[32];
#pragma unroll
    for (int i = 0; i < 32; i++) vals[i] = __builtin_nontemporal_load(w + ((size_t)g * 32 + i) * n + col);
    QGroup r = quantize_group32(vals);
    packed[(size_t)g * n + col] = uint4v{r.w[0], r.w[1], r.w[2], r.w[3]};
    scales[(size_t)g * n + col] = f32_to_f16_bits(r.scale);
}

// [N,K]: a column's values lie along K and its neighbours K floats away, so a workgroup takes 64 columns x four groups
// (bits = 6; NARROW: of matrices with fewer columns 2^bits of them x more groups: 1048576 x 1 22.4 us on 64, now 3.4) through LDS:
// 32 lanes read 512 contiguous bytes of a column (with a thread reading its own 128 bytes every load touched 64 lines:
// 3584 x 18944, 314 MB, 80 us, now 52.2 at 6.0 TB/s), then a thread per (group, column) quantizes.  A column's 32 slots of
// 16 bytes stand 33 apart, so that the 64 columns of a read fall on different banks.  The f32 matrix is read once and passes
// the caches (61 us through them).  blockIdx.y and .z count the groups (.y holds at most 65535).
template <bool NARROW>
__global__ __launch_bounds__(256) void k_quantize_twm_nk(const float *__restrict__ w, uint32_t k, uint32_t n,
                                                          uint4v *__restrict__ packed, uint16_t *__restrict__ scales, uint32_t narrow_bits)
{
    const uint32_t bits = NARROW ? narrow_bits : 6u;
    __shared__ float4v tile[64 * 33];  // (2^bits columns of 2^(11 - bits) slots and one more: 2048 + 2^bits of them)
    const uint32_t groups = k / 32, tall = 256u >> bits, g0 = (blockIdx.z * gridDim.y + blockIdx.y) * tall, col0 = blockIdx.x << bits;
    if (g0 >= groups) return;
    const uint32_t slots = (groups - g0 < tall ? groups - g0 : tall) * 8u;  // 16-byte slots of a column in this tile
    const uint32_t slot_bits = 11u - bits, slot_mask = (1u << slot_bits) - 1u, stride = slot_mask + 2u;
    float4v v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint32_t at = i * 256u + threadIdx.x, c = at >> slot_bits, slot = at & slot_mask;
        const uint32_t col = col0 + c < n ? col0 + c : n - 1;
        v[i] = __builtin_nontemporal_load((const float4v *)(w + (size_t)col * k + (size_t)g0 * 32) + (slot < slots ? slot : 0u));
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint32_t at = i * 256u + threadIdx.x;
        tile[(at >> slot_bits) * stride + (at & slot_mask)] = v[i];
    }
    __syncthreads();
    const uint32_t c = threadIdx.x & ((1u << bits) - 1u), row = threadIdx.x >> bits, g = g0 + row, col = col0 + c;
    if (g >= groups) return;
    float vals[32];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const float4v x = tile[c * stride + row * 8u + i];
#pragma unroll
        for (int j = 0; j < 4; j++) vals[4 * i + j] = x[j];
    }
    QGroup r = quantize_group32(vals);
    if (col >= n) return;
    packed[(size_t)g * n + col] = uint4v{r.w[0], r.w[1], r.w[2], r.w[3]};
    scales[(size_t)g * n + col] = f32_to_f16_bits(r.scale);
}

hipError_t launch_quantize_q4_0(hipStream_t s, const float *w_kn, uint32_t k, uint32_t n, uint8_t *q4)
{
    if (k / 32 == 0 || n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_quantize_q4_0, place_grid(k / 32, n), dim3(256), 0, s, w_kn, k, n, q4, place_slab(k / 32, n));
    return hipGetLastError();
}

hipError_t launch_quantize_twm(hipStream_t s, const float *w, int w_is_nk, uint32_t k, uint32_t n, uint8_t *packed,
                               uint16_t *scales)
{
    const uint32_t groups = k / 32;
    if (groups == 0 || n == 0) return hipSuccess;
    if (w_is_nk) {
        uint32_t bits = 0;
        while (bits < 6 && (1u << bits) < n) bits++;
        const uint32_t tall = 256u >> bits, blocks = (groups + tall - 1) / tall, y = blocks < 65535u ? blocks : 65535u;
        const dim3 grid((n >> bits) + ((n & ((1u << bits) - 1u)) != 0), y, (blocks + y - 1) / y);
        if (bits < 6) hipLaunchKernelGGL(k_quantize_twm_nk<true>, grid, dim3(256), 0, s, w, k, n, (uint4v *)packed, scales, bits);
        else hipLaunchKernelGGL(k_quantize_twm_nk<false>, grid, dim3(256), 0, s, w, k, n, (uint4v *)packed, scales, bits);
    } else {
        hipLaunchKernelGGL(k_quantize_twm_kn, place_grid(groups, n), dim3(256), 0, s, w, groups, n, (uint4v *)packed, scales, place_slab(groups, n));
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------
// reorder Q4_0 column-major -> TW-Marlin; fuse along N
// ---------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_reorder(const uint8_t *__restrict__ q4, uint32_t groups, uint32_t n,
                                                  uint4v *__restrict__ packed, uint16_t *__restrict__ scales)
{
    size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;  // g * n + col (coalesced writes)
    if (idx >= (size_t)groups * n) return;
    uint32_t g = (uint32_t)(idx / n), col = (uint32_t)(idx % n);
    const uint32_t *src = (const uint32_t *)(q4 + ((size_t)col * groups + g) * 20);
    float scale = __uint_as_float(src[0]);
    uint4v o = {src[1], src[2], src[3], src[4]};
    packed[idx] = o;
    scales[idx] = f32_to_f16_bits(scale);
}

hipError_t launch_reorder(hipStream_t s, const uint8_t *q4, uint32_t k, uint32_t n, uint8_t *packed, uint16_t *scales)
{
    size_t total = (size_t)(k / 32) * n;
    if (total == 0) return hipSuccess;
    hipLaunchKernelGGL(k_reorder, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, q4, k / 32, n,
                       (uint4v *)packed, scales);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_fuse_one(const uint4v *__restrict__ pin, const uint16_t *__restrict__ sin,
                                                   uint32_t groups, uint32_t ni, uint32_t total_n,
                                                   uint32_t col_off, uint4v *__restrict__ pout, uint16_t *__restrict__ sout,
                                                   uint32_t slab)
{
    Place at;
    if (!place_of(groups, ni, slab, at)) return;
    const uint32_t g = at.group, c = at.column;
    const size_t idx = (size_t)g * ni + c, dst = (size_t)g * total_n + col_off + c;
    pout[dst] = pin[idx];
    sout[dst] = sin[idx];
}

hipError_t launch_fuse_one(hipStream_t s, const uint8_t *packed_in, const uint16_t *scales_in, uint32_t groups,
                           uint32_t ni, uint32_t total_n, uint32_t col_off, uint8_t *packed_out, uint16_t *scales_out)
{
    if (groups == 0 || ni == 0) return hipSuccess;
    hipLaunchKernelGGL(k_fuse_one, place_grid(groups, ni), dim3(256), 0, s, (const uint4v *)packed_in,
                       scales_in, groups, ni, total_n, col_off, (uint4v *)packed_out, scales_out, place_slab(groups, ni));
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------
// Q4 unpack from the reference layout
// ---------------------------------------------------------------------------------
// Memory bound.  A thread takes COLS neighbouring columns of one group: their 16-byte records once, then 32 rows of COLS
// values.  3584 x 37888 to f16, 352 MB: 49.8 us, 7.1 TB/s (an element per thread, each reading its record's byte and
// dividing its 64-bit index, took 235; four columns 52.3, eight 127).  The stores pass the caches, or the write-back falls
// on whatever runs next; records loaded past the caches as well cost 25 us of the gain, since they are often just written.
template <int COLS, bool F16OUT>
__global__ __launch_bounds__(256) void k_dequant(const uint4v *__restrict__ packed, const uint16_t *__restrict__ scales,
                                                  uint32_t groups, uint32_t n, void *__restrict__ out)
{
    typedef uint16_t halves __attribute__((ext_vector_type(COLS)));
    typedef float floats __attribute__((ext_vector_type(COLS)));
    const uint32_t g = blockIdx.z * gridDim.y + blockIdx.y, col = (blockIdx.x * 256u + threadIdx.x) * COLS;
    if (g >= groups || col >= n) return;
    const size_t rec = (size_t)g * n + col;
    uint4v w[COLS];
    float sc[COLS];
#pragma unroll
    for (int c = 0; c < COLS; c++) {
        w[c] = packed[rec + c];
        sc[c] = f16_bits_to_f32(scales[rec + c]);
        asm volatile("" : "+v"(sc[c]));
    }
    const size_t at = (size_t)g * 32 * n + col;
#pragma unroll
    for (int wi = 0; wi < 4; wi++) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            halves h;
            floats f;
#pragma unroll
            for (int c = 0; c < COLS; c++) {
                // (the product is exact in f32: 11-bit x 4-bit significands; see scale_times_q for the pins)
                const uint32_t nibbles = ((e & 1) ? w[c][wi] >> 4 : w[c][wi]) & 0x0F0F0F0Fu;
                float x = sc[c] * ((float)((nibbles >> (8 * (e >> 1))) & 0xFFu) - 8.0f);
                asm volatile("" : "+v"(x));
                f[c] = x;
                h[c] = f32_to_f16_bits(x);
            }
            const size_t o = at + (size_t)(wi * 8 + e) * n;
            if (F16OUT) __builtin_nontemporal_store(h, (halves *)((uint16_t *)out + o));
            else __builtin_nontemporal_store(f, (floats *)((float *)out + o));
        }
    }
}

// records at any address: a byte and an element per thread
template <bool F16OUT>
__global__ __launch_bounds__(256) void k_dequant_bytes(const uint8_t *__restrict__ packed, const uint16_t *__restrict__ scales,
                                                        uint32_t k, uint32_t n, void *__restrict__ out, uint32_t slab)
{
    Place at;
    if (!place_of(k, n, slab, at)) return;
    const uint32_t row = at.group, col = at.column;
    const uint32_t g = row / 32, e = row % 32;
    const size_t idx = (size_t)row * n + col;
    uint8_t byte = packed[((size_t)g * n + col) * 16 + e / 2];
    int q = (e & 1) ? (byte >> 4) : (byte & 0xF);
    float w = scale_times_q(scales[(size_t)g * n + col], q - 8);
    if (F16OUT) ((uint16_t *)out)[idx] = f32_to_f16_bits(w);
    else ((float *)out)[idx] = w;
}

hipError_t launch_dequant(hipStream_t s, const uint8_t *packed, const uint16_t *scales, uint32_t k, uint32_t n,
                          void *out, bool f16_out)
{
    if (k == 0 || n == 0) return hipSuccess;
    // An element per thread where the records are not aligned -- and where a record per thread would be few workgroups (4096 x
    // 64: 2.6 us and here 2.2) or leave most of one idle (1048576 x 1: 16.5, here 3.2; 262144 x 16: 7.7, here 7.5, to f32 11.4
    // and 7.9).
    if (((uintptr_t)packed & 15) != 0 || n <= 16 || (uint64_t)(k / 32) * n < 32768u) {
        const dim3 grid = place_grid(k, n);
        const uint32_t slab = place_slab(k, n);
        if (f16_out) hipLaunchKernelGGL(k_dequant_bytes<true>, grid, dim3(256), 0, s, packed, scales, k, n, out, slab);
        else hipLaunchKernelGGL(k_dequant_bytes<false>, grid, dim3(256), 0, s, packed, scales, k, n, out, slab);
        return hipGetLastError();
    }
    // two columns per thread where a row's columns keep the alignment of the paired stores
    const bool pairs = n % 2 == 0 && ((uintptr_t)out & (f16_out ? 3 : 7)) == 0;
    const uint32_t groups = k / 32, y = groups < 65535u ? groups : 65535u;
    const dim3 grid((n + (pairs ? 511 : 255)) / (pairs ? 512 : 256), y, (groups + y - 1) / y);
    const uint4v *rec = (const uint4v *)packed;
    if (pairs && f16_out) hipLaunchKernelGGL((k_dequant<2, true>), grid, dim3(256), 0, s, rec, scales, groups, n, out);
    else if (pairs) hipLaunchKernelGGL((k_dequant<2, false>), grid, dim3(256), 0, s, rec, scales, groups, n, out);
    else if (f16_out) hipLaunchKernelGGL((k_dequant<1, true>), grid, dim3(256), 0, s, rec, scales, groups, n, out);
    else hipLaunchKernelGGL((k_dequant<1, false>), grid, dim3(256), 0, s, rec, scales, groups, n, out);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------
// split_qkv / split_gate_up
// ---------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_split_qkv(const float *__restrict__ qkv, float *__restrict__ q,
                                                    float *__restrict__ kk, float *__restrict__ v, uint32_t h,
                                                    uint32_t kv, uint32_t batch)
{
    uint32_t per = h + 2 * kv;
    size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)batch * per) return;
    uint32_t b = (uint32_t)(idx / per), d = (uint32_t)(idx % per);
    float x = qkv[idx];
    if (d < h) q[(size_t)b * h + d] = x;
    else if (d < h + kv) kk[(size_t)b * kv + (d - h)] = x;
    else v[(size_t)b * kv + (d - h - kv)] = x;
}

__global__ __launch_bounds__(256) void k_split_gate_up(const float *__restrict__ gu, float *__restrict__ g,
                                                        float *__restrict__ u, uint32_t ffn, uint32_t batch)
{
    size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)batch * 2 * ffn) return;
    uint32_t b = (uint32_t)(idx / (2 * ffn)), d = (uint32_t)(idx % (2 * ffn));
    float x = gu[idx];
    if (d < ffn) g[(size_t)b * ffn + d] = x;
    else u[(size_t)b * ffn + (d - ffn)] = x;
}

// silu(gate) * up, elementwise (warp_fused_silu_mul, crates/kernels/src/ops.rs:966-976).
__global__ __launch_bounds__(256) void k_silu_mul(const float *__restrict__ gate, const float *__restrict__ up,
                                                   float *__restrict__ out, size_t count)
{
    size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx < count) out[idx] = silu_mul_f32(gate[idx], up[idx]);
}

// out[b][j] = silu(gate_up[b][gate column j]) * gate_up[b][up column j]: the split of
// k_split_gate_up and the SwiGLU gate in one pass.  PAIRED selects where the two columns are:
// [gate | up] halves (the reference's fused order) or the 32-column interleave of paired_col().
template <bool PAIRED>
__global__ __launch_bounds__(256) void k_swiglu_rows(const float *__restrict__ gu, float *__restrict__ out,
                                                      uint32_t ffn, uint32_t batch)
{
    size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)batch * ffn) return;
    uint32_t b = (uint32_t)(idx / ffn), j = (uint32_t)(idx % ffn);
    const float *row = gu + (size_t)b * 2 * ffn;
    float g, u;
    if (PAIRED) {
        uint32_t c = paired_col(j);
        g = row[c];
        u = row[c + kPairWidth];
    } else {
        g = row[j];
        u = row[ffn + j];
    }
    out[idx] = silu_mul_f32(g, u);
}

// TW-Marlin arrays of gate and up ([G][ffn] records and scales each) -> one [G][2*ffn] pair of
// arrays in the paired column order.  Pure byte moves; one thread per (group, output column).
__global__ __launch_bounds__(256) void k_pair_gate_up(const uint4v *__restrict__ gp, const uint16_t *__restrict__ gs,
                                                       const uint4v *__restrict__ up, const uint16_t *__restrict__ us,
                                                       uint32_t groups, uint32_t ffn, uint4v *__restrict__ pout,
                                                       uint16_t *__restrict__ sout)
{
    size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;  // g * 2*ffn + c
    size_t n2 = (size_t)2 * ffn;
    if (idx >= (size_t)groups * n2) return;
    uint32_t g = (uint32_t)(idx / n2), c = (uint32_t)(idx % n2);
    uint32_t j = (c >> 6) * kPairWidth + (c & 31u);
    size_t src = (size_t)g * ffn + j;
    bool is_up = (c & kPairWidth) != 0;
    pout[idx] = is_up ? up[src] : gp[src];
    sout[idx] = is_up ? us[src] : gs[src];
}

// ArgMax along the last dimension with the reference's rule (crates/kernels/src/missing_ops.rs:24-39): the
// first index whose value is greater than every earlier candidate, starting from -1e30 at index 0 (so
// values <= -1e30 and NaNs are never chosen, and an empty or all-small row yields 0).
//
// A workgroup takes a span of sixteen columns a thread, all loads in flight; of a row's several spans each leaves its
// candidate in the scratch, and the workgroup that arrives last picks among them and clears the row's counter.  Bound: latency.
// Workgroups of 512 and 1024 threads hold rows of up to 8192 and 16384 columns whole, since a hand-over costs a microsecond.
// A value and its index are one 64-bit key, larger for a larger value and, among equal values, for the smaller index; the
// largest of a wave's keys is found half by half, values and then indices, by DPP steps and four scalar reads.
// (152064 columns: two launches, of 8192 columns a workgroup each merging through an LDS tree of ten steps and of one workgroup a
// row for the candidates, 5.7 us in a graph, now 3.9; 16 rows 6.8, now 4.3; 512 rows of 32000 16.7, now 12.7.)
constexpr uint32_t kArgmaxEach = 16;
constexpr uint32_t kArgmaxCounterStep = 32;   // a row's counter has a cache line of its own (16 rows in one line: 10.5 us, now 4.3)

// a number that orders as the float does (-0 as 0)
__device__ __forceinline__ uint32_t argmax_order(float v)
{
    const uint32_t u = __float_as_uint(v + 0.0f);
    return u ^ ((uint32_t)((int)u >> 31) | 0x80000000u);
}

__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v)
{
#define TWM_MAX_STEP(N) v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x120 + N, 0xf, 0xf, true))   // row_ror:N
    TWM_MAX_STEP(8);
    TWM_MAX_STEP(4);
    TWM_MAX_STEP(2);
    TWM_MAX_STEP(1);
#undef TWM_MAX_STEP
    const uint32_t a = __builtin_amdgcn_readlane(v, 0), b = __builtin_amdgcn_readlane(v, 16);
    const uint32_t c = __builtin_amdgcn_readlane(v, 32), d = __builtin_amdgcn_readlane(v, 48);
    return max(max(a, b), max(c, d));
}

__device__ __forceinline__ uint64_t wave_max_key(uint64_t key)
{
    const uint32_t hi = wave_max_u32((uint32_t)(key >> 32));
    return (uint64_t)hi << 32 | wave_max_u32((uint32_t)(key >> 32) == hi ? (uint32_t)key : 0u);
}

template <uint32_t THREADS>
__global__ __launch_bounds__(THREADS) void k_argmax(const float *__restrict__ in, uint32_t cols, uint32_t spans, uint64_t *__restrict__ candidates,
                                                    unsigned *__restrict__ counters, int *__restrict__ out)
{
    constexpr uint32_t kWaves = THREADS / 64, kSpan = THREADS * kArgmaxEach;
    __shared__ uint64_t found[kWaves];
    __shared__ uint32_t last;
    const uint32_t row = blockIdx.x, lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const float *src = in + (size_t)row * cols;
    float best = -1e30f;
    uint32_t idx = 0xFFFFFFFFu;  // "none yet"
    for (uint64_t c0 = (uint64_t)blockIdx.y * kSpan; c0 < cols; c0 += (uint64_t)spans * kSpan) {
        // past the end the last column again, under a larger index than its own
        const float *from = src + c0;
        const uint32_t most = cols - (uint32_t)c0 - 1u;
        float v[kArgmaxEach];
#pragma unroll
        for (uint32_t j = 0; j < kArgmaxEach; j++) {
            const uint32_t c = threadIdx.x + THREADS * j;
            v[j] = from[c < most ? c : most];
        }
#pragma unroll
        for (uint32_t j = 0; j < kArgmaxEach; j++) {  // (in increasing index order)
            if (v[j] > best) {
                best = v[j];
                idx = (uint32_t)c0 + threadIdx.x + THREADS * j;
            }
        }
    }
    // (no candidate: a key of -1e30 and index part 0, below every candidate's)
    uint64_t key = wave_max_key((uint64_t)argmax_order(best) << 32 | (0xFFFFFFFFu - idx));
    if (lane == 0) found[wave] = key;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (uint32_t w = 1; w < kWaves; w++) key = found[w] > key ? found[w] : key;
        last = 1u;
        if (spans > 1) {
            __hip_atomic_store(&candidates[(size_t)row * spans + blockIdx.y], key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __builtin_amdgcn_s_waitcnt(0);  // vmcnt(0): the candidate is in place
            last = __hip_atomic_fetch_add(&counters[row * kArgmaxCounterStep], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == spans - 1u;
        } else {
            out[row] = (uint32_t)key == 0u ? 0 : (int)(0xFFFFFFFFu - (uint32_t)key);
        }
    }
    if (spans == 1) return;
    __syncthreads();
    if (!last || wave != 0) return;
    key = 0;
    for (uint32_t s = lane; s < spans; s += 64u) {
        const uint64_t other = __hip_atomic_load(&candidates[(size_t)row * spans + s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        key = other > key ? other : key;
    }
    key = wave_max_key(key);
    if (lane == 0) {
        out[row] = (uint32_t)key == 0u ? 0 : (int)(0xFFFFFFFFu - (uint32_t)key);
        __hip_atomic_store(&counters[row * kArgmaxCounterStep], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// `scratch` (scratch_bytes) holds the spans' candidates and `counters` (zero between launches) their arrivals; without enough of
// either, or for short rows, one workgroup per row takes all its spans in turn.
hipError_t launch_argmax(hipStream_t s, const float *in, uint32_t rows, uint32_t cols, int *out, void *scratch,
                         size_t scratch_bytes, unsigned *counters, uint32_t n_counters)
{
    if (rows == 0) return hipSuccess;
    // Whole rows in one workgroup up to 16384 columns of up to 512 rows (1 x 5000 3.4 us in two spans, 2.35 whole, 1 x 16384 3.4 and
    // 2.9, 512 x 9000 5.1 and 4.4; beyond that many rows the larger workgroups wait for room on the CUs: 600 x 9000 4.2 and 5.2)
    const uint32_t threads = rows > 512u || cols <= 256u * kArgmaxEach || cols > 1024u * kArgmaxEach ? 256u : cols <= 512u * kArgmaxEach ? 512u : 1024u;
    const uint32_t span = threads * kArgmaxEach;
    uint32_t spans = (uint32_t)(((uint64_t)cols + span - 1) / span);
    // about a thousand workgroups at most: with many rows a workgroup takes several spans
    const uint32_t most = rows < 1024u ? 1024u / rows : 1u;
    if (spans > most) spans = most;
    if (spans == 0 || !scratch || !counters || (uint64_t)rows * kArgmaxCounterStep > n_counters || (size_t)rows * spans * 8 > scratch_bytes) spans = 1;
    auto kernel = threads == 256u ? k_argmax<256> : threads == 512u ? k_argmax<512> : k_argmax<1024>;
    hipLaunchKernelGGL(kernel, dim3(rows, spans), dim3(threads), 0, s, in, cols, spans, (uint64_t *)scratch, counters, out);
    return hipGetLastError();
}

hipError_t launch_split_qkv(hipStream_t s, const float *qkv, float *q, float *kk, float *v, uint32_t h, uint32_t kv,
                            uint32_t batch)
{
    size_t total = (size_t)batch * (h + 2 * kv);
    if (total == 0) return hipSuccess;
    hipLaunchKernelGGL(k_split_qkv, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, qkv, q, kk, v, h, kv, batch);
    return hipGetLastError();
}

hipError_t launch_split_gate_up(hipStream_t s, const float *gu, float *g, float *u, uint32_t ffn, uint32_t batch)
{
    size_t total = (size_t)batch * 2 * ffn;
    if (total == 0) return hipSuccess;
    hipLaunchKernelGGL(k_split_gate_up, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, gu, g, u, ffn, batch);
    return hipGetLastError();
}

hipError_t launch_silu_mul(hipStream_t s, const float *gate, const float *up, float *out, size_t count)
{
    if (count == 0) return hipSuccess;
    hipLaunchKernelGGL(k_silu_mul, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, s, gate, up, out, count);
    return hipGetLastError();
}

hipError_t launch_swiglu_rows(hipStream_t s, const float *gu, float *out, uint32_t ffn, uint32_t batch, bool paired)
{
    size_t total = (size_t)batch * ffn;
    if (total == 0) return hipSuccess;
    dim3 grid((unsigned)((total + 255) / 256));
    if (paired) hipLaunchKernelGGL(k_swiglu_rows<true>, grid, dim3(256), 0, s, gu, out, ffn, batch);
    else hipLaunchKernelGGL(k_swiglu_rows<false>, grid, dim3(256), 0, s, gu, out, ffn, batch);
    return hipGetLastError();
}

hipError_t launch_pair_gate_up(hipStream_t s, const uint8_t *gate_packed, const uint16_t *gate_scales,
                               const uint8_t *up_packed, const uint16_t *up_scales, uint32_t groups, uint32_t ffn,
                               uint8_t *packed_out, uint16_t *scales_out)
{
    size_t total = (size_t)groups * 2 * ffn;
    if (total == 0) return hipSuccess;
    hipLaunchKernelGGL(k_pair_gate_up, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s,
                       (const uint4v *)gate_packed, gate_scales, (const uint4v *)up_packed, up_scales, groups, ffn,
                       (uint4v *)packed_out, scales_out);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------
// GEMV on the reference layout, f32 activations (no repack, exact f32 products).
// One lane per output column: a wave reads 64 x 16 B = 1 KiB contiguous per group.
// The activation index is wave-uniform, so A comes in through scalar loads.
// ---------------------------------------------------------------------------------
// ALIGN16: the records are 16-byte aligned (one 128-bit load); otherwise four 32-bit loads, the alignment the
// reference's own kernel needs (quantize.rs:1227-1228).
template <bool ATOMIC, bool ALIGN16>
__global__ __launch_bounds__(256) void k_ref_gemv(float *__restrict__ c, const float *__restrict__ a,
                                                   const uint32_t *__restrict__ packed,
                                                   const uint16_t *__restrict__ scales, uint32_t n, uint32_t groups,
                                                   uint32_t gps)
{
    uint32_t col = blockIdx.x * 256 + threadIdx.x;
    if (col >= n) return;
    uint32_t g0 = blockIdx.y * gps;
    uint32_t g1 = g0 + gps < groups ? g0 + gps : groups;
    float dot = 0.0f;
    for (uint32_t g = g0; g < g1; g++) {
        float s = f16_bits_to_f32(scales[(size_t)g * n + col]);
        const uint32_t *rec = packed + ((size_t)g * n + col) * 4u;
        uint4v v;
        if (ALIGN16) v = *(const uint4v *)rec;
        else v = uint4v{rec[0], rec[1], rec[2], rec[3]};
        const float *ab = a + g * 32;
        float gdot = 0.0f;
#pragma unroll
        for (int wi = 0; wi < 4; wi++) {
            uint32_t w = v[wi];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                int q = (int)((w >> (4 * j)) & 0xFu) - 8;
                gdot = fmaf(ab[wi * 8 + j], (float)q, gdot);
            }
        }
        dot = fmaf(gdot, s, dot);
    }
    if (ATOMIC) atomicAdd(&c[col], dot);
    else c[col] = dot;
}

hipError_t launch_ref_gemv(hipStream_t s, const float *a, const uint8_t *packed, const uint16_t *scales, float *c,
                           uint32_t n, uint32_t k, uint32_t splits, uint32_t groups_per_split)
{
    if (n == 0) return hipSuccess;
    dim3 grid((n + 255) / 256, splits);
    const bool align16 = ((uintptr_t)packed & 15) == 0;
    if (splits > 1) {
        hipError_t e = launch_fill_zero(s, c, (size_t)n * 4);
        if (e != hipSuccess) return e;
    }
#define TWM_REF_GEMV(AT, AL) \
    hipLaunchKernelGGL((k_ref_gemv<AT, AL>), grid, dim3(256), 0, s, c, a, (const uint32_t *)packed, scales, n, k / 32, groups_per_split)
    if (splits > 1) {
        if (align16) TWM_REF_GEMV(true, true);
        else TWM_REF_GEMV(true, false);
    } else {
        if (align16) TWM_REF_GEMV(false, true);
        else TWM_REF_GEMV(false, false);
    }
#undef TWM_REF_GEMV
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------
// repack: reference layout -> wave tile order (see twm_internal.h)
// ---------------------------------------------------------------------------------
// bit position 4*p of the result holds the nibble of k-offset j, p = j/2 for even j, 4 + j/2 for odd j
__device__ __forceinline__ uint32_t permute_word(uint32_t w)
{
    uint32_t r = 0;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        int p = (j & 1) ? 4 + (j >> 1) : (j >> 1);
        r |= ((w >> (4 * j)) & 0xFu) << (4 * p);
    }
    return r;
}

__global__ __launch_bounds__(256) void k_repack_q(const uint32_t *__restrict__ packed, uint32_t groups, uint32_t n,
                                                   uint32_t n_tiles, uint32_t k_chunks, uint4v *__restrict__ qw)
{
    size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;  // (kc * n_tiles + nt) * 64 + lane
    if (idx >= (size_t)n_tiles * k_chunks * 64) return;
    uint32_t lane = (uint32_t)(idx & 63);
    size_t tile = idx >> 6;
    uint32_t nt = (uint32_t)(tile % n_tiles), kc = (uint32_t)(tile / n_tiles);
    uint32_t col = nt * 16 + (lane & 15), kb = lane >> 4;
    uint4v o;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        uint32_t g = kc * 4 + i;
        uint32_t w = 0x88888888u;
        if (g < groups && col < n) w = packed[((size_t)g * n + col) * 4 + kb];
        o[i] = permute_word(w);
    }
    qw[idx] = o;
}

__global__ __launch_bounds__(256) void k_repack_s(const uint16_t *__restrict__ scales, uint32_t groups, uint32_t n,
                                                   uint32_t n_tiles, uint32_t k_chunks, uint2v *__restrict__ sc)
{
    size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;  // (kc * n_tiles + nt) * 16 + c
    if (idx >= (size_t)n_tiles * k_chunks * 16) return;
    uint32_t c = (uint32_t)(idx & 15);
    size_t tile = idx >> 4;
    uint32_t nt = (uint32_t)(tile % n_tiles), kc = (uint32_t)(tile / n_tiles);
    uint32_t col = nt * 16 + c;
    uint32_t h[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        uint32_t g = kc * 4 + i;
        h[i] = (g < groups && col < n) ? scales[(size_t)g * n + col] : 0u;
    }
    uint2v o = {h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
    sc[idx] = o;
}

hipError_t launch_repack(hipStream_t s, const uint8_t *packed, const uint16_t *scales, uint32_t k, uint32_t n, void *qw,
                         void *sc, uint32_t n_tiles, uint32_t k_chunks)
{
    size_t tq = (size_t)n_tiles * k_chunks * 64, ts = (size_t)n_tiles * k_chunks * 16;
    if (tq == 0) return hipSuccess;
    hipLaunchKernelGGL(k_repack_q, dim3((unsigned)((tq + 255) / 256)), dim3(256), 0, s, (const uint32_t *)packed, k / 32,
                       n, n_tiles, k_chunks, (uint4v *)qw);
    hipLaunchKernelGGL(k_repack_s, dim3((unsigned)((ts + 255) / 256)), dim3(256), 0, s, scales, k / 32, n, n_tiles,
                       k_chunks, (uint2v *)sc);
    return hipGetLastError();
}

// Q4 unpack straight from the wave tile order (used to prove the repack lossless).
__global__ __launch_bounds__(256) void k_weight_dequant_f16(const uint32_t *__restrict__ qw,
                                                             const uint16_t *__restrict__ sc, uint32_t k, uint32_t n,
                                                             uint32_t n_tiles, uint16_t *__restrict__ out)
{
    size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;  // row * n + col
    if (idx >= (size_t)k * n) return;
    uint32_t row = (uint32_t)(idx / n), col = (uint32_t)(idx % n);
    uint32_t g = row / 32, e = row % 32;
    uint32_t nt = col / 16, c = col % 16, kc = g / 4, i = g % 4, kb = e / 8, j = e % 8;
    size_t tile = (size_t)kc * n_tiles + nt;
    uint32_t w = qw[(tile * 64 + kb * 16 + c) * 4 + i];
    int p = (j & 1) ? 4 + (j >> 1) : (j >> 1);
    int q = (int)((w >> (4 * p)) & 0xFu) - 8;
    out[idx] = f32_to_f16_bits(scale_times_q(sc[(tile * 16 + c) * 4 + i], q));
}

hipError_t launch_weight_dequant_f16(hipStream_t s, const WeightView &w, uint16_t *out_kn)
{
    size_t total = (size_t)w.k * w.n;
    if (total == 0) return hipSuccess;
    hipLaunchKernelGGL(k_weight_dequant_f16, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s,
                       (const uint32_t *)w.qw, (const uint16_t *)w.sc, w.k, w.n, w.n_tiles, out_kn);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------
// column-lane copy (layout in twm_gemv4.hip): 4608-byte blocks [tile64][k_chunk], each
// [4 groups][64 columns][16 B nibbles, permuted inside each word] + [64 columns][4 f16 scales]
// ---------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_repack_col(const uint4v *__restrict__ packed, const uint16_t *__restrict__ scales,
                                                     uint32_t groups, uint32_t n, uint32_t k_chunks, uint32_t tiles64,
                                                     char *__restrict__ cw, uint32_t pair_ffn)
{
    size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;  // ((tile * k_chunks + kc) * 4 + g) * 64 + lane
    if (idx >= (size_t)tiles64 * k_chunks * 256) return;
    uint32_t lane = (uint32_t)(idx & 63), gi = (uint32_t)((idx >> 6) & 3);
    size_t blk = idx >> 8;
    uint32_t kc = (uint32_t)(blk % k_chunks), tile = (uint32_t)(blk / k_chunks);
    uint32_t g = kc * 4 + gi, col = tile * 64 + lane;
    uint4v w = {0x88888888u, 0x88888888u, 0x88888888u, 0x88888888u};
    uint32_t sbits = 0;
    if (g < groups && col < n) {
        // pair_ffn != 0: the source is [gate | up] (n = 2 * pair_ffn) and the copy takes the paired order
        uint32_t src = pair_ffn ? (col >> 6) * kPairWidth + (col & 31u) + ((col & kPairWidth) ? pair_ffn : 0u) : col;
        w = packed[(size_t)g * n + src];
        sbits = scales[(size_t)g * n + src];
    }
    uint4v o = {permute_word(w[0]), permute_word(w[1]), permute_word(w[2]), permute_word(w[3])};
    char *base = cw + blk * kColBlockBytes;
    *(uint4v *)(base + gi * 1024u + lane * 16u) = o;
    *(uint16_t *)(base + 4096u + lane * 8u + gi * 2u) = (uint16_t)sbits;
}

hipError_t launch_repack_col(hipStream_t s, const uint8_t *packed, const uint16_t *scales, uint32_t k, uint32_t n,
                             void *cq, uint32_t n_pad, uint32_t k_chunks, uint32_t pair_ffn)
{
    size_t total = (size_t)(n_pad / 64) * k_chunks * 256;
    if (total == 0) return hipSuccess;
    hipLaunchKernelGGL(k_repack_col, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, (const uint4v *)packed,
                       scales, k / 32, n, k_chunks, n_pad / 64, (char *)cq, pair_ffn);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_weight_dequant_f16_col(const char *__restrict__ cw, uint32_t k, uint32_t n,
                                                                 uint32_t k_chunks, uint16_t *__restrict__ out)
{
    size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;  // row * n + col
    if (idx >= (size_t)k * n) return;
    uint32_t row = (uint32_t)(idx / n), col = (uint32_t)(idx % n);
    uint32_t g = row / 32, e = row % 32, j = e % 8;
    const char *base = cw + ((size_t)(col / 64) * k_chunks + g / 4) * kColBlockBytes;
    uint32_t lane = col % 64, gi = g % 4;
    uint32_t w = *(const uint32_t *)(base + gi * 1024u + lane * 16u + (e / 8) * 4u);
    int p = (j & 1) ? 4 + (j >> 1) : (j >> 1);
    int q = (int)((w >> (4 * p)) & 0xFu) - 8;
    uint16_t sbits = *(const uint16_t *)(base + 4096u + lane * 8u + gi * 2u);
    out[idx] = f32_to_f16_bits(scale_times_q(sbits, q));
}

hipError_t launch_weight_dequant_f16_col(hipStream_t s, const WeightView &w, uint16_t *out_kn)
{
    size_t total = (size_t)w.k * w.n;
    if (total == 0) return hipSuccess;
    hipLaunchKernelGGL(k_weight_dequant_f16_col, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s,
                       (const char *)w.cq, w.k, w.n, w.k_chunks, out_kn);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------
// One repacked copy from the other.  Both hold every 32-bit word of the reference's records with the same nibble
// permutation, so the conversion moves words: word kb of column c's record of group g is
//   tile copy:        qw[(kc * n_tiles + c / 16) * 64 + kb * 16 + c % 16][g % 4]
//   column-lane copy: block (c / 64, kc), group row g % 4, lane c % 64, word kb
// ---------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_col_to_tile(const char *__restrict__ cw, uint32_t n_tiles, uint32_t k_chunks,
                                                      uint4v *__restrict__ qw, uint2v *__restrict__ sc)
{
    size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;  // (kc * n_tiles + nt) * 64 + lane
    if (idx >= (size_t)n_tiles * k_chunks * 64) return;
    const uint32_t lane = (uint32_t)(idx & 63), c = lane & 15, kb = lane >> 4;
    const size_t tile = idx >> 6;
    const uint32_t nt = (uint32_t)(tile % n_tiles), kc = (uint32_t)(tile / n_tiles);
    const char *blk = cw + ((size_t)(nt / 4) * k_chunks + kc) * kColBlockBytes;
    const uint32_t col = (nt % 4) * 16 + c;
    uint4v o;
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] = *(const uint32_t *)(blk + i * 1024u + col * 16u + kb * 4u);
    qw[idx] = o;
    if (kb == 0) sc[tile * 16 + c] = *(const uint2v *)(blk + 4096u + col * 8u);
}

__global__ __launch_bounds__(256) void k_tile_to_col(const uint32_t *__restrict__ qw, const uint2v *__restrict__ sc,
                                                      uint32_t n_tiles, uint32_t k_chunks, char *__restrict__ cw)
{
    size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;  // ((tile64 * k_chunks + kc) * 4 + g) * 64 + lane
    if (idx >= (size_t)(n_tiles / 4) * k_chunks * 256) return;
    const uint32_t lane = (uint32_t)(idx & 63), gi = (uint32_t)((idx >> 6) & 3);
    const size_t blk = idx >> 8;
    const uint32_t kc = (uint32_t)(blk % k_chunks), tile64 = (uint32_t)(blk / k_chunks);
    const size_t tile = (size_t)kc * n_tiles + tile64 * 4 + lane / 16;
    uint4v o;
#pragma unroll
    for (int kb = 0; kb < 4; kb++) o[kb] = qw[(tile * 64 + kb * 16 + lane % 16) * 4 + gi];
    char *base = cw + blk * kColBlockBytes;
    *(uint4v *)(base + gi * 1024u + lane * 16u) = o;
    if (gi == 0) *(uint2v *)(base + 4096u + lane * 8u) = sc[tile * 16 + lane % 16];
}

hipError_t launch_col_to_tile(hipStream_t s, const void *cq, uint32_t n_tiles, uint32_t k_chunks, void *qw, void *sc)
{
    size_t total = (size_t)n_tiles * k_chunks * 64;
    if (total == 0) return hipSuccess;
    hipLaunchKernelGGL(k_col_to_tile, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, (const char *)cq, n_tiles,
                       k_chunks, (uint4v *)qw, (uint2v *)sc);
    return hipGetLastError();
}

hipError_t launch_tile_to_col(hipStream_t s, const void *qw, const void *sc, uint32_t n_tiles, uint32_t k_chunks, void *cq)
{
    size_t total = (size_t)(n_tiles / 4) * k_chunks * 256;
    if (total == 0) return hipSuccess;
    hipLaunchKernelGGL(k_tile_to_col, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, (const uint32_t *)qw,
                       (const uint2v *)sc, n_tiles, k_chunks, (char *)cq);
    return hipGetLastError();
}

}  // namespace twm
