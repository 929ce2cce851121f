// The second launch of a GEMM whose K is split over workgroups: out[row][col] = sum over splits of partials[split][row][col].
#include "twm_prefill_core.h"

namespace twm {

namespace {

// N more partial sums of P places kPairWidth columns apart, all loads in flight, added by pairs (a chain of additions in split order
// had a tenth more rounding error in the whole result on seventeen splits)
template <int N, int P> __device__ __forceinline__ void splitk_add(float4v (&s)[P], const TWM_GLOBAL char *base, uint32_t &offset, uint32_t stride)
{
    float4v v[N + 1][P];
#pragma unroll
    for (int j = 1; j <= N; j++) {
        offset += stride;
#pragma unroll
        for (int p = 0; p < P; p++) v[j][p] = *(const TWM_GLOBAL float4v *)(base + offset + p * kPairWidth * 4u);
    }
#pragma unroll
    for (int p = 0; p < P; p++) {
        v[0][p] = s[p];
#pragma unroll
        for (int step = 1; step <= N; step *= 2)
#pragma unroll
            for (int j = 0; j + step <= N; j += 2 * step) v[j][p] += v[j + step][p];
        s[p] = v[0][p];
    }
}

// The partial sums of P places, added in an order that their number alone decides.  (Byte offsets: the partial sums of a launch fit the
// context's scratch, 256 MB.)
template <int P> __device__ __forceinline__ void splitk_sum(float4v (&s)[P], const float *partials, uint32_t offset, uint32_t stride, uint32_t splits)
{
    const TWM_GLOBAL char *base = (const TWM_GLOBAL char *)partials;
#pragma unroll
    for (int p = 0; p < P; p++) s[p] = *(const TWM_GLOBAL float4v *)(base + offset + p * kPairWidth * 4u);
    uint32_t left = splits - 1u;
    for (; left >= 8u; left -= 8u) splitk_add<8>(s, base, offset, stride);
    switch (left) {
    case 1: splitk_add<1>(s, base, offset, stride); break;
    case 2: splitk_add<2>(s, base, offset, stride); break;
    case 3: splitk_add<3>(s, base, offset, stride); break;
    case 4: splitk_add<4>(s, base, offset, stride); break;
    case 5: splitk_add<5>(s, base, offset, stride); break;
    case 6: splitk_add<6>(s, base, offset, stride); break;
    case 7: splitk_add<7>(s, base, offset, stride); break;
    }
}

}  // namespace

// One thread per four padded columns; stride: bytes from one split's sums to the next.  Bound: latency, and on many rows the
// traffic: a launch takes about 1.8 us with a single load and store, this one 2.4 for four splits of 8 x 3584 and 3.1 for seven of
// 96 x 4608 in a graph.  A 32-bit division by the quads of a row in place of a 64-bit one, the arguments of the loads preloaded, and
// all loads of up to nine splits in flight instead of one, four or two in turn: 0.2 - 0.6 us a launch (3584 -> 4608 at 96 rows on
// seven splits 16.6 -> 16.0, 18944 -> 3584 at 8 f32 rows on four 16.1 -> 15.9, the four launches of a layer of 1152 values at 394
// f32 rows 87.0 -> 85.6 with three of these; a decode layer with one 64.3 -> 63.7 at 32 rows, 45.3 -> 44.8 at 8).  Sixteen loads
// in flight were no faster; eight under conditions instead of a form per remainder 1.5 % behind on few splits of many rows; a grid
// row per output row instead of the division left most lanes of a row's last workgroup idle.
template <RowStore ROWS, uint32_t BLOCK>
__global__ __launch_bounds__(BLOCK) void k_splitk_reduce(const float *__restrict__ partials, uint32_t n_ld, uint32_t splits, uint32_t stride,
                                                         uint32_t n, const float *__restrict__ row_scale, uint32_t m_rows, OutSpec out)
{
    const uint32_t idx = blockIdx.x * BLOCK + threadIdx.x, quads = n_ld / 4u, row = idx / quads, col = (idx - row * quads) * 4u;
    if (row >= m_rows) return;
    uint32_t ld = 0;
    float4v bias = {0.f, 0.f, 0.f, 0.f};
    float *dst = nullptr, scale = 1.f;
    // (the factor and the bias are on their way during the sum)
    if (row_scale) scale = row_scale[row];
    if (ROWS == kRowsSegments && col < n) dst = pf_quad_of(out, col, ld, bias);
    float4v sum[1];
    splitk_sum(sum, partials, (row * n_ld + col) * 4u, stride, splits);
    float4v s = sum[0];
    if (row_scale) s *= scale;  // (f32 rows scaled into the f16 range)
    if constexpr (ROWS == kRowsPlain) {
        if (col < n) *(float4v *)(out.seg[0].ptr + (size_t)row * n + col) = s;
    } else if constexpr (ROWS == kRowsSegments) {
        if (out.seg[0].bias) s += bias;
        if (dst) *(float4v *)(dst + (size_t)row * ld) = s;
    } else {
#pragma unroll
        for (uint32_t j = 0; j < 4; j++)
            if (col + j < n) pf_store_out(out, row, col + j, s[j]);
    }
}

// The same sum for a paired gate/up weight: one thread per four features adds the gate and the up partials
// (32 columns apart) and stores silu(gate) * up.  The loads of both places are in flight together, also the only ones of one split, which
// f32 prompt rows under a gate come as (one place after the other cost a second latency: 160 -> 2 x 64 at 204 f32 rows 11.5, now 11.0 us).
template <uint32_t BLOCK>
__global__ __launch_bounds__(BLOCK) void k_splitk_reduce_swiglu(const float *__restrict__ partials, uint32_t n_ld, uint32_t splits, uint32_t stride,
                                                                uint32_t ffn, const float *__restrict__ row_scale, uint32_t m_rows,
                                                                uint32_t act, float *__restrict__ gate_out)
{
    const uint32_t idx = blockIdx.x * BLOCK + threadIdx.x, quads = ffn / 4u, row = idx / quads, feat = (idx - row * quads) * 4u;   // (ffn is a multiple of 32)
    if (row >= m_rows) return;
    const uint32_t at = (row * n_ld + paired_col(feat)) * 4u;
    const float scale = row_scale ? row_scale[row] : 1.f;
    float4v sum[2];
    splitk_sum(sum, partials, at, stride, splits);
    float4v g = sum[0], u = sum[1];
    if (row_scale) {
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
    const dim3 grid((unsigned)(((uint64_t)m * quads + block - 1) / block));
    if (out.swiglu) hipLaunchKernelGGL(gated, grid, dim3(block), 0, s, partials, n_ld, splits, stride, n / 2, out.row_scale, m, out.gate_act, out.swiglu);
    else hipLaunchKernelGGL(plain, grid, dim3(block), 0, s, partials, n_ld, splits, stride, n, out.row_scale, m, out);
    return hipGetLastError();
}

}  // namespace twm
