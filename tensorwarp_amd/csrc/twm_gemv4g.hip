// One to four rows on small and on narrow matrices: a lane per column and 32-deep group.
//
// Semantics: k_gemv4s (crates/kernels/src/quantize.rs:1186-1298): per group the products a * (q - 8) summed in f32 by the 4x4x4
// MFMA, scaled once by f32(scale), added to the running f32 sum.
//
// What bounds these launches is the chain of one wave: a matrix of 0.5 .. 8 MB is spread over a few thousand waves that all run
// at once, and a launch takes a hand-over (1.6 us from node to node of a graph with nothing in them, 1.8 with a load and a
// store) plus that chain.  So the chain is short: a workgroup owns 16 columns, a wave a chunk of 128 values at a time, lane =
// (group l / 16, column l % 16) with 16 bytes of nibbles, one scale and one 8-wide piece of the activations -- four words to
// unpack and eight MFMAs in turn where k_gemv4s's lane has sixteen and thirty-two.  All loads of a wave's up to four chunks are
// issued up front; no split over workgroups, whose division would stand in front of the first load; where wave 0 will store,
// and the bias there, is fetched while the weights are on their way.
// (us in a graph, k_gemv4s or k_gemv4 -> here: one f16 row 896 -> 1152 2.53 -> 2.23, 896 -> 896 2.76 -> 2.41, 1536 -> 12288
// 4.47 -> 3.87, 4096 -> 4096 3.88 -> 3.58, gated 896 -> 2 x 4864 3.58 -> 3.27, 2048 -> 2 x 5632 4.92 -> 4.49; two rows 1536 ->
// 2048 4.20 -> 2.70; four 4.47 -> 2.96; one f32 row 896 -> 1152 2.80 -> 2.39.)
// 16 columns gated read 128-byte runs, which is no loss while the whole matrix is in flight at once; 32 columns were slower on
// every narrow shape (896 -> 1152 2.56, 4096 -> 4096 4.58, 2816 -> 2 x 704 3.9 against 3.1 on 16).
#include "twm_gemv4_core.h"
#include "twm_internal.h"

namespace twm {

// RL: rows (1, 2, 4); AF32: one row of f32 activations, as two f16 terms in rows 0 and 1 of the MFMA's A block; NP: chunks per wave;
// GATED: 8 gate columns and the 8 up columns of the same features.  TRACE: four words per workgroup as in k_gemv4s_traced.
template <int RL, bool AF32, int NP, bool GATED, bool TRACE>
__global__ __launch_bounds__(1024) void k_gemv4g(const char *__restrict__ cw, const void *__restrict__ a_any, uint32_t waves_rows,
                                                uint32_t k, uint32_t k_chunks, uint32_t sub_tiles, uint32_t n, uint32_t *__restrict__ trace, OutSpec out)
{
    constexpr int SUB = 16, E = RL * SUB;
    static_assert(E <= 64 && (!AF32 || RL == 1), "wave 0 finishes");
    __shared__ float red[16 * E];
    const uint32_t waves = waves_rows >> 8, m_rows = waves_rows & 255u;
    if constexpr (TRACE) {
        if (threadIdx.x == 0) {
            trace[4u * blockIdx.x] = (uint32_t)__builtin_amdgcn_s_memrealtime();
            trace[4u * blockIdx.x + 1u] = 0u;
            trace[4u * blockIdx.x + 3u] = (__builtin_amdgcn_s_getreg((31 << 11) | 4) & 0xFFFFu) | (__builtin_amdgcn_s_getreg((3 << 11) | 20) << 16);
        }
    }
    // each XCD a contiguous run of sub-tiles (workgroups reach the eight XCDs in turn)
    const uint32_t st = (blockIdx.x & 7u) * ((sub_tiles + 7u) >> 3) + (blockIdx.x >> 3);
    if (st >= sub_tiles) return;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const uint32_t cl = lane % SUB, gl = lane / SUB;
    const uint32_t tile = st / (64 / SUB), part = st % (64 / SUB);
    const uint32_t col = GATED ? (cl / (SUB / 2)) * 32u + part * (SUB / 2) + cl % (SUB / 2) : part * SUB + cl;
    const char *tbase = cw + (size_t)tile * k_chunks * kColBlockBytes;
    uint32_t arow = RL == 1 ? 0u : cl & 3u;
    if (arow > m_rows - 1u) arow = m_rows - 1u;

    uint4v wq[NP], a[NP], a2[NP];
    uint16_t sc[NP];
#pragma unroll
    for (int i = 0; i < NP; i++) {
        const uint32_t kc0 = wave + i * waves, kc = kc0 < k_chunks ? kc0 : k_chunks - 1u;   // (past the end: replayed and left out)
        uint32_t k0 = kc * 128u + gl * 32u + (cl >> 2) * 8u;
        if (k0 > k - 8u) k0 = k - 8u;   // only the zero-padded groups of a last partial chunk get here
        if (AF32) {
            const uint4v *p = (const uint4v *)((const float *)a_any + k0);
            a[i] = p[0];
            a2[i] = p[1];
        } else {
            a[i] = *(const uint4v *)((const _Float16 *)a_any + (size_t)arow * k + k0);
        }
        const char *blk = tbase + (size_t)kc * kColBlockBytes;
        wq[i] = ld_once((const uint4v *)(blk + gl * 1024u + col * 16u));
        sc[i] = ld_once((const uint16_t *)(blk + 4096u + col * 8u + gl * 2u));
    }
    __builtin_amdgcn_sched_barrier(0);
    // where wave 0 will store, and the bias, fetched while the weights are on their way
    float *dst = nullptr;
    uint32_t ld = 0;
    float bias = 0.f;
    bool has_bias = false;
    if (wave == 0) {
        if (GATED) {
            const uint32_t ffn = n >> 1, feat = tile * 32u + part * (SUB / 2) + cl;
            if (cl < SUB / 2 && feat < ffn) dst = out.swiglu + feat;
            ld = ffn;
        } else {
            const uint32_t on = tile * 64u + col;
            if (on < n) {
#pragma unroll
                for (uint32_t s = 0; s < kMaxSegs; s++) {
                    if (s < out.count) {
                        const uint32_t rel = on - out.seg[s].start;
                        if (rel < out.seg[s].width) {
                            dst = out.seg[s].ptr + rel;
                            ld = out.seg[s].width;
                            if (out.seg[s].bias) {
                                bias = out.seg[s].bias[rel];
                                has_bias = true;
                            }
                        }
                    }
                }
            }
        }
    }
    const Gemv4Consts dq = make_gemv4_consts();
    float acc[RL];
#pragma unroll
    for (int r = 0; r < RL; r++) acc[r] = 0.f;
#pragma unroll
    for (int i = 0; i < NP; i++) {
        // A chunk past the end and a padded group replay other values of the row: their sums are left out, not scaled by zero
        // (an infinity among those values would come out as NaN in every column).
        const bool live = ((wave + i * waves) * 4u + gl) * 32u < k;
        float inv[4] = {1.f, 1.f, 1.f, 1.f};
        union { uint4v u; half4v h[2]; } av;
        av.u = a[i];
        if (AF32) {
            uint4v hi, lo;
            gemv4s_split_a_f32_piece<false>(a[i], a2[i], hi, lo, inv);
            const bool second = (lane & 1u) != 0;
#pragma unroll
            for (int w = 0; w < 4; w++) av.u[w] = second ? lo[w] : hi[w];
        }
        half4v lo4, hi4;
        float4v d = {0.f, 0.f, 0.f, 0.f};
#define TWM_4G_PIECE(W)                                     \
    gemv4_dequant_word(wq[i][W], dq, lo4, hi4);            \
    d = mfma_sub<SUB, W>(av.h[0], lo4, d);                 \
    d = mfma_sub<SUB, W>(av.h[1], hi4, d);
        TWM_4G_PIECE(0) TWM_4G_PIECE(1) TWM_4G_PIECE(2) TWM_4G_PIECE(3)
#undef TWM_4G_PIECE
        union { uint16_t u; _Float16 h; } sv;
        sv.u = sc[i];
        const float s = (float)sv.h;
        if (AF32) acc[0] = live ? fmaf(d[0] + d[1], s * inv[0], acc[0]) : acc[0];
        else {
#pragma unroll
            for (int r = 0; r < RL; r++) acc[r] = live ? fmaf(d[r], s, acc[r]) : acc[r];
        }
    }
    if constexpr (TRACE) {
        if (threadIdx.x == 0) trace[4u * blockIdx.x + 1u] = (uint32_t)__builtin_amdgcn_s_memrealtime();
    }
    // sums: the wave's four groups by lane swaps, the waves through LDS, read by 64 / E lanes per entry
#pragma unroll
    for (int r = 0; r < RL; r++) acc[r] = sum_lane_groups<SUB>(acc[r]);
    if (gl == 0) {
#pragma unroll
        for (int r = 0; r < RL; r++) red[wave * E + r * SUB + cl] = acc[r];
    }
    __syncthreads();
    if (wave != 0) return;
    constexpr int PARTS = 64 / E;
    const uint32_t e = lane % E, first = lane / E;
    float t = 0.f;
    float x[16 / PARTS];
#pragma unroll
    for (int j = 0; j < 16 / PARTS; j++) {
        const uint32_t w = first + j * PARTS;
        x[j] = red[(w < waves ? w : 0u) * E + e];
    }
#pragma unroll
    for (int j = 0; j < 16 / PARTS; j++) t += first + j * PARTS < waves ? x[j] : 0.f;
    t = sum_lane_groups<E>(t);
    const uint32_t r = e / SUB;
    if (GATED) {
        const float up = __shfl_down(t, SUB / 2, 64);
        if (lane < E && dst && r < m_rows) dst[(size_t)r * ld] = gated_mul(out.gate_act, t, up);
    } else {
        if (lane < E && dst && r < m_rows) dst[(size_t)r * ld] = has_bias ? t + bias : t;
    }
    if constexpr (TRACE) {
        if (threadIdx.x == 0) trace[4u * blockIdx.x + 2u] = (uint32_t)__builtin_amdgcn_s_memrealtime();
    }
}

// Waves per workgroup, 0 where the other kernels of up to four rows are ahead.  From forced sweeps of 35 shapes (us, this kernel /
// the best other form):
// * f16: K up to 3072 at one row, 2688 at two, 2560 at four, up to 512, 512 and 400 column tiles of 64 (2048 -> 32000 at one row
//   8.1 / 8.2, at four 9.4 / 8.9; 3072 -> 2 x 8192 at two rows 7.4 / 7.3, 2560 -> 8192 at four level), and up to K = 8192 on 64
//   column tiles (3584 -> 3584 3.44 / 3.66, at four rows 3.95 / 4.12; 8192 -> 1024 4.28 / 4.32; 3584 -> 4608 at four 5.13 /
//   4.88; 3584 -> 2 x 18944 16.3 / 16.0; gated at four rows 2240 -> 2 x 7776 7.25 / 6.55).
// * f32, one row: every lane splits a piece of its own for each group, four times what k_gemv4s's lanes do: K up to 1536 on 200
//   column tiles (896 -> 151936 18.4 / 15.5, 2048 -> 2048 level), gated up to 3072 on 64 (2816 -> 2 x 704 3.54 / 3.88; 1472 -> 2 x 6048 4.97 / 4.79).
//   On 150 column tiles and more the waves take two to four chunks; where those do not come out even many tiles stay with the other
//   forms: two chunks gated (256 -> 2 x 7328 at three rows 3.68 / 3.34, 544 -> 2 x 14048 at one 5.24 / 4.59), five to seven (544 ->
//   2 x 12544 at four rows 5.49 / 4.95, 576 -> 28479 at one 4.96 / 4.50), nine and thirteen to fifteen at one row (1088 -> 26584
//   6.08 / 5.66, 1600 -> 30792 7.61 / 7.13); gated at two rows from nine chunks on (1088 -> 2 x 16352 7.69 / 6.86, 2048 -> 2 x 11136
//   7.42 / 6.91).
// One chunk per wave up to eleven of them on 150 column tiles, else up to four (4096 -> 4096 on 8 / 16 waves 3.58 / 3.62, 1536 ->
// 12288 on 4 / 12 3.87 / 4.9; 3072 -> 5120 on 8 / 6 4.04 / 4.23), from 25 chunks on on an even number of waves; f32 one chunk up
// to sixteen, then two.
uint32_t plan_gemv4g(uint32_t tiles64, uint32_t k_chunks, uint32_t m, bool a_f32, bool gated)
{
    if (m == 0 || m > 4 || k_chunks == 0) return 0;
    if (a_f32) {
        if (m != 1 || !(gated ? k_chunks <= 24 && tiles64 <= 64 : k_chunks <= 12 && tiles64 <= 200)) return 0;
        return k_chunks <= 16 ? k_chunks : (k_chunks + 1) / 2;
    }
    const uint32_t deep = m == 1 ? 24u : m == 2 ? 21u : 20u, wide = m <= 2 ? 512u : 400u;
    if (gated && m >= 2 && k_chunks > (m == 2 ? 20u : 16u) && tiles64 > (m == 2 ? 256u : 200u)) return 0;
    if (!(k_chunks <= deep && tiles64 <= wide) && !(k_chunks <= 64 && tiles64 <= 64)) return 0;
    if (k_chunks == 2 && tiles64 > (gated ? (m >= 3 ? 150u : m == 2 ? 400u : 330u) : m == 1 ? 440u : 512u)) return 0;
    if (k_chunks == 5 && tiles64 > (gated ? (m >= 3 ? 150u : m == 2 ? 300u : 200u) : m == 1 ? 340u : 360u)) return 0;
    if ((k_chunks == 6 || k_chunks == 7) && tiles64 > 340 && (gated || m == 1)) return 0;
    if (gated && m == 2 && k_chunks >= 9 && tiles64 > 340) return 0;
    if (m == 1 && ((k_chunks == 9 && tiles64 > (gated ? 260u : 320u)) || (k_chunks >= 13 && k_chunks <= 15 && tiles64 > (gated ? 320u : 430u)))) return 0;
    if (k_chunks <= 11 && tiles64 <= 150) return k_chunks;
    if (k_chunks > 24) return ((k_chunks + 3) / 4 + 1u) & ~1u;
    // three or four chunks per wave, whichever leaves fewer replayed; two where both leave several
    const uint32_t w4 = (k_chunks + 3) / 4, w3 = (k_chunks + 2) / 3;
    if (k_chunks <= 20 && w4 * 4 <= k_chunks + 1) return w4 < 4 ? 4u : w4;
    if (k_chunks > 20 || w3 * 3 <= k_chunks + 1) return w3 < 4 ? 4u : w3;
    return (k_chunks + 1) / 2;
}

// m <= 4 with f16 rows, m = 1 with f32 ones; up to 16 waves with up to four chunks each.
hipError_t launch_gemv4g(hipStream_t s, const WeightView &w, const void *a, bool a_f32, uint32_t m, const OutSpec &out, uint32_t waves, TraceBuf trace)
{
    if (m == 0 || w.n == 0) return hipSuccess;
    if (!w.cq || m > 4 || (a_f32 && m != 1) || waves < 1 || waves > 16 || w.k_chunks == 0) return hipErrorInvalidValue;
    if (out.swiglu && w.n % 64 != 0) return hipErrorInvalidValue;
    const uint32_t sub_tiles = w.n_tiles, blocks = (sub_tiles + 7) / 8 * 8, np = (w.k_chunks + waves - 1) / waves;
    const bool gated = out.swiglu != nullptr, traced = trace.ptr && !a_f32 && m == 1 && blocks <= trace.capacity;
#define TWM_4G(RL, AF, NP, GT, TR)                                                                                              \
    hipLaunchKernelGGL((k_gemv4g<RL, AF, NP, GT, TR>), dim3(blocks), dim3(waves * 64), 0, s, (const char *)w.cq, a, (waves << 8) | m, \
                       w.k, w.k_chunks, sub_tiles, w.n, trace.ptr, out)
#define TWM_4G_NP(RL, AF, GT, TR)                     \
    do {                                              \
        if (np == 1) TWM_4G(RL, AF, 1, GT, TR);       \
        else if (np == 2) TWM_4G(RL, AF, 2, GT, TR);  \
        else if (np == 3) TWM_4G(RL, AF, 3, GT, TR);  \
        else if (np == 4) TWM_4G(RL, AF, 4, GT, TR);  \
        else return hipErrorInvalidValue;             \
    } while (0)
#define TWM_4G_GATE(RL, AF, TR)                       \
    do {                                              \
        if (gated) TWM_4G_NP(RL, AF, true, TR);       \
        else TWM_4G_NP(RL, AF, false, TR);            \
    } while (0)
    if (a_f32) TWM_4G_GATE(1, true, false);
    else if (traced) TWM_4G_GATE(1, false, true);
    else if (m == 1) TWM_4G_GATE(1, false, false);
    else if (m == 2) TWM_4G_GATE(2, false, false);
    else TWM_4G_GATE(4, false, false);
#undef TWM_4G_GATE
#undef TWM_4G_NP
#undef TWM_4G
    return hipGetLastError();
}

}  // namespace twm
