// The second launch of a GEMM whose K is split over workgroups: out[row][col] = sum over splits of partials[split][row][col].
#include "twm_prefill_core.h"

namespace twm {

namespace {

// The partial sums of one place, added in split order (deterministic): up to eight loads in flight.  (Byte offsets: the partial
// sums of a launch fit the context's scratch, 256 MB.)
__device__ __forceinline__ float4v splitk_sum(const float *partials, uint32_t offset, uint32_t stride, uint32_t splits)
{
    const TWM_GLOBAL char *base = (const TWM_GLOBAL char *)partials;
    float4v s = *(const TWM_GLOBAL float4v *)(base + offset);
    for (uint32_t z = 1; z < splits; z += 8u) {
        float4v v[8];
#pragma unroll
        for (uint32_t j = 0; j < 8u; j++) {
            if (z + j < splits) {
                offset += stride;
                v[j] = *(const TWM_GLOBAL float4v *)(base + offset);
            }
        }
#pragma unroll
        for (uint32_t j = 0; j < 8u; j++)
            if (z + j < splits) s += v[j];
    }
    return s;
}

}  // namespace

// One thread per four padded columns, one grid row per output row; stride: bytes from one split's sums to the next.  Bound:
// latency: a launch takes about 1.8 us with a single load and store, this one 2.4 for four splits of 8 x 3584 and 3.1 for seven
// of 96 x 4608 in a graph.  A grid row per output row instead of a division by the quads of a row, the arguments of the loads
// preloaded, and eight loads in flight instead of four: 0.2 - 0.4 us a launch (3584 -> 4608 at 96 rows on seven splits 16.56 ->
// 16.25, 18944 -> 3584 at 8 f32 rows on four 16.1 -> 15.9; a decode layer with one such launch 64.3 -> 63.7 at 32 rows, 45.3 ->
// 44.8 at 8).  Sixteen in flight were no faster.
template <RowStore ROWS, uint32_t BLOCK>
__global__ __launch_bounds__(BLOCK) void k_splitk_reduce(const float *__restrict__ partials, uint32_t n_ld, uint32_t splits, uint32_t stride,
                                                         uint32_t n, const float *__restrict__ row_scale, uint32_t row0, OutSpec out)
{
    const uint32_t col = (blockIdx.x * BLOCK + threadIdx.x) * 4u, row = row0 + blockIdx.y;
    if (col >= n_ld) return;
    float4v s = splitk_sum(partials, (row * n_ld + col) * 4u, stride, splits);
    if (row_scale) s *= row_scale[row];  // (f32 rows scaled into the f16 range)
    if constexpr (ROWS == kRowsPlain) {
        if (col < n) *(float4v *)(out.seg[0].ptr + (size_t)row * n + col) = s;
    } else if constexpr (ROWS == kRowsSegments) {
        uint32_t ld = 0;
        float4v bias = {0.f, 0.f, 0.f, 0.f};
        float *dst = col < n ? pf_quad_of(out, col, ld, bias) : nullptr;
        if (out.seg[0].bias) s += bias;
        if (dst) *(float4v *)(dst + (size_t)row * ld) = s;
    } else {
#pragma unroll
        for (uint32_t j = 0; j < 4; j++)
            if (col + j < n) pf_store_out(out, row, col + j, s[j]);
    }
}

// The same sum for a paired gate/up weight: one thread per four features adds the gate and the up partials
// (32 columns apart) in split order and stores silu(gate) * up.
template <uint32_t BLOCK>
__global__ __launch_bounds__(BLOCK) void k_splitk_reduce_swiglu(const float *__restrict__ partials, uint32_t n_ld, uint32_t splits, uint32_t stride,
                                                                uint32_t ffn, const float *__restrict__ row_scale, uint32_t row0,
                                                                uint32_t act, float *__restrict__ gate_out)
{
    const uint32_t feat = (blockIdx.x * BLOCK + threadIdx.x) * 4u, row = row0 + blockIdx.y;
    if (feat >= ffn) return;   // (ffn is a multiple of 32)
    const uint32_t at = (row * n_ld + paired_col(feat)) * 4u;
    float4v g = splitk_sum(partials, at, stride, splits), u = splitk_sum(partials, at + kPairWidth * 4u, stride, splits);
    if (row_scale) {
        const float scale = row_scale[row];
        g *= scale;
        u *= scale;
    }
    float4v o;
#pragma unroll
    for (int j = 0; j < 4; j++) o[j] = gated_mul(act, g[j], u[j]);
    *(float4v *)(gate_out + (size_t)row * ffn + feat) = o;
}

hipError_t launch_splitk_reduce(hipStream_t s, const float *partials, const OutSpec &out, uint32_t m, uint32_t n,
                                uint32_t n_ld, uint32_t splits)
{
    const uint32_t quads = (out.swiglu ? n / 2 : n_ld) / 4;
    if (m == 0 || quads == 0) return hipSuccess;
    if (out.swiglu && n % (2 * kPairWidth) != 0) return hipErrorInvalidValue;
    if ((uint64_t)splits * m * n_ld * 4 > 0xFFFFFFFFull) return hipErrorInvalidValue;   // (32-bit byte offsets)
    // few places: one wave per workgroup, so that they spread over the CUs
    const bool few = (size_t)m * quads < 256u * 256u;
    const uint32_t block = few ? 64u : 256u, rows = row_store_of(out, n), stride = m * n_ld * 4u;
    auto gated = few ? k_splitk_reduce_swiglu<64> : k_splitk_reduce_swiglu<256>;
    auto plain = rows == kRowsPlain      ? (few ? k_splitk_reduce<kRowsPlain, 64> : k_splitk_reduce<kRowsPlain, 256>)
                 : rows == kRowsSegments ? (few ? k_splitk_reduce<kRowsSegments, 64> : k_splitk_reduce<kRowsSegments, 256>)
                                         : (few ? k_splitk_reduce<kRowsNone, 64> : k_splitk_reduce<kRowsNone, 256>);
    for (uint32_t row0 = 0; row0 < m; row0 += 65535u) {   // (the most rows of a grid)
        const dim3 grid((quads + block - 1) / block, m - row0 < 65535u ? m - row0 : 65535u);
        if (out.swiglu) hipLaunchKernelGGL(gated, grid, dim3(block), 0, s, partials, n_ld, splits, stride, n / 2, out.row_scale, row0, out.gate_act, out.swiglu);
        else hipLaunchKernelGGL(plain, grid, dim3(block), 0, s, partials, n_ld, splits, stride, n, out.row_scale, row0, out);
    }
    return hipGetLastError();
}

}  // namespace twm
