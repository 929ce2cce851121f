// GEMM for 5 .. 32 rows: waves that share nothing until the end, each on k-chunks of its own, exact weights.
//
// Semantics: per 32-deep group the products a * (q - 8) are summed in f32 by one v_mfma_f32_16x16x32_f16 with a zero
// accumulator, the group sum is scaled once by f32(scale) and added to the running f32 sum
// (crates/kernels/src/quantize.rs:1219-1238; M > 1 has the meaning of gemm_q4_0, quantize.rs:1825-1858).  f32 rows enter as
// two f16 terms, split in here: each row's stretch of a 128-deep chunk is scaled by the power of two that brings its largest
// magnitude to [2^13, 2^14), hi = f16(x), lo = f16(x - hi), and the chunk's sums of that row are scaled back before they join
// the running sum (exact: any finite f32 row keeps 22 bits per value relative to the largest of 128 neighbours).
//
// What bounds these launches: HBM on wide matrices, latency on narrow ones, and in between the vector ALU (unpack 9, scaling 4
// or 8 instructions per eight weights, a conversion of f32 rows that every workgroup repeats).  So:
// * a workgroup owns 16 NT columns for all rows and, mostly, the whole K; NT is chosen so that one round of workgroups fills
//   the CUs; its eight waves deal the 128-deep chunks among themselves.  There is no barrier in the main loop -- the kernels
//   that share an activation tile among waves spend longer on their barrier-and-load chain -- and one at the end, where all
//   waves add the partial sums;
// * a wave loads its chunk's activation tile into registers a chunk ahead (sixteen lanes per row), writes it to an LDS region of
//   its own (256-byte rows, XOR-swizzled 16-byte slots) and reads the MFMA operands of the four groups back once for all its
//   tiles -- from memory in operand order they cost 3.5 times as much, 37 against 130 bytes per ns and CU;
// * tile after tile, a tile's weight registers take the next chunk's loads as soon as its last group is unpacked: with up to
//   four tiles two chunks are in flight, with more one, 92 KB per CU on ten tiles;
// * the rows are loaded by quads, as many as there are (NV: 8, 12, 16, 24 or 32 rows): each costs the CU's load path, which
//   delivers some 6.4 TB/s in all, weights and rows alike, once the weights come from HBM (16 and 32 rows whatever their number
//   before: 3584 -> 3584 at 8 rows 5.45 -> 5.1, at 24 6.9 -> 6.4, 8192 -> 8192 at 8 11.5 -> 10.7, at 24 15.4 -> 14.7; with the
//   conversion of f32 rows 4096 -> 12288 at 24 18.4 -> 16.5, 4096 -> 4096 at 20 12.2 -> 11.3);
// * nothing in the store waits for a kernel argument: the output description is fetched behind the first loads (-0.3 us on
//   896 -> 1152), and up to ten sums per lane four waves finish a tile, one register each (-0.5 us there).
// f32 rows in one launch instead of a conversion launch and a GEMM on its two f16 arrays (us, before -> now): 4096 -> 2 x 11008
// gated at 8 rows 22.3 -> 13.6, at 13 22.4 -> 15.8; 18944 -> 3584 at 8 20.2 -> 14.5, at 32 30.3 -> 25.9; 4096 -> 12288 at 13
// 15.3 -> 12.3; 4096 -> 4096 at 13 9.9 -> 8.4; 11008 -> 4096 at 13 15.9 -> 13.6; 896 -> 1152 at 8 5.6 -> 3.3.
// f16 rows, against the kernels with shared activation tiles: 4096 -> 2 x 11008 at 32 rows 20.0 -> 16.4, at 16 15.9 -> 12.8;
// 3584 -> 2 x 18944 at 32 24.4 -> 22.2, at 13 20.1 -> 17.8; 4096 -> 12288 at 32 14.3 -> 12.4.
// Measured and not kept: activations two chunks ahead (896 -> 1152 at 8 rows 3.5 / 3.6, 4096 -> 4096 at 32 rows 8.0 / 8.5),
// v_fma_mixlo_f16 for the two terms (it issues at half the rate of v_fma_mix_f32 and v_cvt_pk_f16_f32).
#include "twm_waves_core.h"

#include <type_traits>

namespace twm {

namespace {

// The largest of m[j] over each sixteen lanes, in each of them, for NV values at once.  (A value read through DPP must have
// been written two instructions before: the steps of several values are interleaved.)
template <int NV>
__device__ __forceinline__ void rows16_max(float (&m)[NV])
{
#define TWM_MAX4(N)                                                             \
    "v_max_f32_dpp %0, %0, %0 row_ror:" #N " row_mask:0xf bank_mask:0xf\n"      \
    "v_max_f32_dpp %1, %1, %1 row_ror:" #N " row_mask:0xf bank_mask:0xf\n"      \
    "v_max_f32_dpp %2, %2, %2 row_ror:" #N " row_mask:0xf bank_mask:0xf\n"      \
    "v_max_f32_dpp %3, %3, %3 row_ror:" #N " row_mask:0xf bank_mask:0xf\n"
#define TWM_MAX3(N)                                                             \
    "v_max_f32_dpp %0, %0, %0 row_ror:" #N " row_mask:0xf bank_mask:0xf\n"      \
    "v_max_f32_dpp %1, %1, %1 row_ror:" #N " row_mask:0xf bank_mask:0xf\n"      \
    "v_max_f32_dpp %2, %2, %2 row_ror:" #N " row_mask:0xf bank_mask:0xf\n"
#define TWM_MAX2(N)                                                             \
    "s_nop 1\n"                                                                 \
    "v_max_f32_dpp %0, %0, %0 row_ror:" #N " row_mask:0xf bank_mask:0xf\n"      \
    "v_max_f32_dpp %1, %1, %1 row_ror:" #N " row_mask:0xf bank_mask:0xf\n"
#pragma unroll
    for (int j = 0; j + 4 <= NV; j += 4)
        asm("s_nop 1\n" TWM_MAX4(8) TWM_MAX4(4) TWM_MAX4(2) TWM_MAX4(1) : "+v"(m[j]), "+v"(m[j + 1]), "+v"(m[j + 2]), "+v"(m[j + 3]));
    constexpr int L = NV / 4 * 4;
    if constexpr (NV % 4 == 3) asm("s_nop 1\n" TWM_MAX3(8) TWM_MAX3(4) TWM_MAX3(2) TWM_MAX3(1) : "+v"(m[L]), "+v"(m[L + 1]), "+v"(m[L + 2]));
    if constexpr (NV % 4 == 2) asm(TWM_MAX2(8) TWM_MAX2(4) TWM_MAX2(2) TWM_MAX2(1) : "+v"(m[L]), "+v"(m[L + 1]));
    static_assert(NV % 4 != 1, "");
#undef TWM_MAX4
#undef TWM_MAX3
#undef TWM_MAX2
}

}  // namespace

// grid: K-splits x column groups (the splits of a group are neighbours, so that with eight of them each XCD reads one stretch
// of the activations).  The first arguments, which the loads need, arrive preloaded (thirteen words).
template <int MT, int NT, int MODE, int W, int NV>
__global__ __launch_bounds__(64 * W) void k_waves_exact(const uint4v *__restrict__ qw, const uint2v *__restrict__ sc,
                                                 const void *__restrict__ a_any, uint32_t m_rows, uint32_t k, uint32_t n_tiles,
                                                 uint32_t k_chunks, uint32_t chunks_per_split, uint32_t gated_u, uint32_t n,
                                                 float *__restrict__ partials, OutSpec out)
{
    constexpr bool F32 = MODE != kRowsF16;
    constexpr int TERMS = MODE == kRowsF32 ? 2 : 1;
    constexpr int SLOTS = NT <= 4 && !(MT == 2 && TERMS == 2) ? 2 : 1;
    constexpr int kTile = 16 * MT * kWeRow;                          // halves of one term's activation tile
    constexpr int kRegion = TERMS * kTile + (F32 ? 32 * MT : 0);     // halves of a wave's LDS region (behind the tiles: a factor per row)
    constexpr int LD = F32 ? 2 : 1;                                  // 16-byte loads per lane and row quad
    extern __shared__ __attribute__((aligned(16))) _Float16 lds_all[];

    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t c = lane & 15u, kb = lane >> 4;
    _Float16 *region = lds_all + wave * kRegion;

    const uint32_t group = blockIdx.y, split = blockIdx.x;
    const uint32_t kc0 = split * chunks_per_split;
    const uint32_t nchunks = k_chunks - kc0 < chunks_per_split ? k_chunks - kc0 : chunks_per_split;
    const uint32_t count = nchunks > wave ? (nchunks - wave + W - 1u) / W : 0u;  // this wave's chunks: wave, wave + W, ...

    // This group's tiles; with the gated store, gate tiles and then the up tiles of the same features.  Tiles past the end
    // replay the last one and are never stored.
    const bool gated = NT % 2 == 0 && gated_u != 0u;
    auto tile_at = [&](uint32_t t) {
        if (NT % 2 == 0 && gated) {
            const uint32_t pair = group * (NT / 2) + t % (NT / 2);
            return (pair >> 1) * 4u + (pair & 1u) + (t >= NT / 2 ? 2u : 0u);
        }
        return group * NT + t;
    };
    uint32_t tile_of[NT];
#pragma unroll
    for (int i = 0; i < NT; i++) {
        const uint32_t t = tile_at(i);
        tile_of[i] = t < n_tiles ? t : n_tiles - 1u;
    }

    WeConsts dq = {0x000F000Fu, 0x00F000F0u, 0x64006400u, 0x54005400u};
    asm volatile("" : "+s"(dq.mask_lo), "+s"(dq.mask_hi), "+v"(dq.magic_lo), "+v"(dq.magic_hi));

    float4v acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int i = 0; i < NT; i++) acc[mt][i] = float4v{0.f, 0.f, 0.f, 0.f};

    // f16: load j takes rows 4 j .. 4 j + 3: lane L row 4 j + L / 16, vector (L % 16) ^ (row % 16), written to slot L % 16.
    // f32: the same rows, lane L values 4 p .. 4 p + 3 of each half of the row's 128 (p = L % 16; odd lane groups the second
    // half first, so that the 8-byte LDS writes of two rows take different banks).  Rows past m_rows replay the last row and
    // are never stored.  Vectors past K read other values of the row; f32 rows and up to sixteen f16 rows stage them as zeros
    // (an infinity there times the zero of a padded weight would make the row's sums NaN; above that k_batch and k_prefill,
    // which take such rows on other shapes, replay a vector as well, and there the masks cost 1 % of the launch).
    uint32_t a_off[NV], a_vec[4];
    const uint32_t p = lane & 15u, odd = (lane >> 4) & 1u;
#pragma unroll
    for (int j = 0; j < 4; j++) a_vec[j] = p ^ (4u * j + (lane >> 4));
#pragma unroll
    for (int j = 0; j < NV; j++) {
        uint32_t row = 4u * j + (lane >> 4);
        row = row < m_rows ? row : m_rows - 1;
        a_off[j] = F32 ? row * k * 4u : (row * k + a_vec[j & 3] * 8u) * 2u;
    }
    const uint32_t q_off = lane * 16u, s_off = c * 8u;
    uint4v ar[NV][LD];
    uint4v wq[SLOTS][NT];
    uint2v ws[SLOTS][NT];
    // Chunk i of this wave.  Past the end every lane reads the first bytes of the wave's first chunk instead (one line per load,
    // never used): the loads are unconditional, so the compiler's count of loads in flight stays exact.
    auto chunk_at = [&](uint32_t i) { return kc0 + wave + (i < count ? i : 0u) * (uint32_t)W; };
    auto load_a = [&](uint32_t i) {
        const uint32_t kg = chunk_at(i), on = i < count ? 0xFFFFFFFFu : 0u;
        const TWM_GLOBAL char *src = we_scalar_base(a_any, (size_t)kg * (F32 ? 512u : 256u));
        if constexpr (F32) {
            const uint32_t most = (k - kg * 128u) * 4u - 16u;   // the row's last 16 bytes, for places past its end (staged as zeros)
#pragma unroll
            for (int l = 0; l < 2; l++) {
                uint32_t col = 16u * p + (((uint32_t)l ^ odd) << 8);
                col = col < most ? col : most;
#pragma unroll
                for (int j = 0; j < NV; j++) ar[j][l] = *(const TWM_GLOBAL uint4v *)(src + ((a_off[j] + col) & on));
            }
        } else {
#pragma unroll
            for (int j = 0; j < NV; j++) {
                const uint32_t back = kg * 128u + a_vec[j & 3] * 8u < k ? 0u : a_vec[j & 3] * 16u;
                ar[j][0] = *(const TWM_GLOBAL uint4v *)(src + ((a_off[j] - back) & on));
            }
        }
    };
    auto load_b = [&](int slot, int t, uint32_t i) {
        const uint32_t kg = chunk_at(i), on = i < count ? 0xFFFFFFFFu : 0u;
        const size_t tile = (size_t)kg * n_tiles + tile_of[t];
        wq[slot][t] = __builtin_nontemporal_load((const TWM_GLOBAL uint4v *)(we_scalar_base(qw, tile * 1024u) + (q_off & on)));
        ws[slot][t] = __builtin_nontemporal_load((const TWM_GLOBAL uint2v *)(we_scalar_base(sc, tile * 128u) + (s_off & on)));
    };
    auto stage_a = [&](uint32_t i) {
        const uint32_t left = k - chunk_at(i) * 128u;  // the row's values from this chunk on
        if constexpr (!F32) {
            if (MT == 1 && left < 128u) {
#pragma unroll
                for (int j = 0; j < NV; j++) ar[j][0] = a_vec[j & 3] * 8u < left ? ar[j][0] : uint4v{0u, 0u, 0u, 0u};
            }
#pragma unroll
            for (int j = 0; j < NV; j++) *(uint4v *)(region + j * 512 + lane * 8u) = ar[j][0];
        } else {
            if (left < 128u) {
                asm volatile("");   // (a branch, not selects in every chunk)
#pragma unroll
                for (int l = 0; l < 2; l++)
#pragma unroll
                    for (int j = 0; j < NV; j++) ar[j][l] = (((uint32_t)l ^ odd) * 64u + 4u * p) < left ? ar[j][l] : uint4v{0u, 0u, 0u, 0u};
            }
            float m[NV];
#pragma unroll
            for (int j = 0; j < NV; j++) m[j] = we_max8(ar[j][0], ar[j][1]);
            rows16_max<NV>(m);
#pragma unroll
            for (int j = 0; j < NV; j++) {
                const WeFactor factor = we_factor(m[j]);
                const uint32_t row = 4u * j + (lane >> 4);
#pragma unroll
                for (int l = 0; l < 2; l++) {
                    uint2v hi, lo;
                    we_terms(ar[j][l], factor.down, hi, lo);
                    const uint32_t vec = (((uint32_t)l ^ odd) << 3) + (p >> 1);
                    *(uint2v *)(region + row * kWeRow + ((vec ^ (row & 15u)) * 8u) + (p & 1u) * 4u) = hi;
                    if constexpr (MODE == kRowsF32Few)
                        *(uint2v *)(region + (row + 8u) * kWeRow + ((vec ^ (row + 8u)) * 8u) + (p & 1u) * 4u) = lo;
                    else
                        *(uint2v *)(region + kTile + row * kWeRow + ((vec ^ (row & 15u)) * 8u) + (p & 1u) * 4u) = lo;
                }
                if (p == 0) {
                    float *f = (float *)(region + TERMS * kTile);
                    f[row] = factor.back;
                    if (MODE == kRowsF32Few) f[row + 8u] = factor.back;
                }
            }
        }
    };
    uint32_t rd_off[4];  // row c of a row block, vector 4 g + kb of the chunk -> slot (4 g + kb) ^ c
#pragma unroll
    for (int g = 0; g < 4; g++) rd_off[g] = c * kWeRow + (((4u * g + kb) ^ c) * 8u);

    // The chunk's 4 NT (tile, group) units in turn: a unit's MFMAs are followed by the next unit's unpack and then by its own
    // scaling, so that the matrix pipe's latency passes under the unpack.  f32 rows: a tile's four groups are summed first and
    // join the running sums through the rows' factors, one multiply-add more per chunk.
    auto compute = [&](int slot, uint32_t next) {
        half8 af[TERMS][4][MT];
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
            for (int t = 0; t < TERMS; t++)
#pragma unroll
                for (int mt = 0; mt < MT; mt++) af[t][g][mt] = *(const half8 *)(region + t * kTile + mt * 16 * kWeRow + rd_off[g]);
        float4v back[MT];
        if constexpr (F32) {
#pragma unroll
            for (int mt = 0; mt < MT; mt++) back[mt] = *(const float4v *)((const float *)(region + TERMS * kTile) + 16 * mt + 4u * kb);
        }
        auto scale_of = [&](int u) {
            union { uint32_t u32; half2v h; } pair;
            pair.u32 = ws[slot][u / 4][(u & 3) >> 1];
            return (float)pair.h[u & 1];
        };
        half8 bf = we_unpack(wq[slot][0][0], dq);
        float4v sum[MT];
#pragma unroll
        for (int u = 0; u < 4 * NT; u++) {
            const int t = u / 4, g = u % 4;
            float4v d[MT];
#pragma unroll
            for (int mt = 0; mt < MT; mt++) d[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[0][g][mt], bf, float4v{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            if constexpr (TERMS == 2) {
#pragma unroll
                for (int mt = 0; mt < MT; mt++) d[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[1][g][mt], bf, d[mt], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            half8 bn = bf;
            if (u + 1 < 4 * NT) bn = we_unpack(wq[slot][(u + 1) / 4][(u + 1) % 4], dq);
            const float scale = scale_of(u);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    if constexpr (F32) {
                        sum[mt][r] = g == 0 ? d[mt][r] * scale : __builtin_fmaf(d[mt][r], scale, sum[mt][r]);
                        if (g == 3) acc[mt][t][r] = __builtin_fmaf(sum[mt][r], back[mt][r], acc[mt][t][r]);
                    } else {
                        acc[mt][t][r] += d[mt][r] * scale;
                    }
                }
            __builtin_amdgcn_sched_barrier(0);
            if (g == 3) {
                load_b(slot, t, next);
                __builtin_amdgcn_sched_barrier(0);
            }
            bf = bn;
        }
    };

    if (count) {
        load_a(0);
#pragma unroll
        for (int s = 0; s < SLOTS; s++)
#pragma unroll
            for (int t = 0; t < NT; t++) load_b(s, t, (uint32_t)s);
        __builtin_amdgcn_sched_barrier(0);
        // (the store's arguments, fetched while the loads are on their way)
        asm volatile("" ::"s"(out.seg[0].ptr), "s"(out.seg[2].ptr), "s"(out.count));
        __builtin_amdgcn_sched_barrier(0);
        auto step = [&](int slot, uint32_t i) {
            stage_a(i);
            __builtin_amdgcn_sched_barrier(0);
            load_a(i + 1u);
            __builtin_amdgcn_sched_barrier(0);
            compute(slot, i + SLOTS);
        };
        if constexpr (SLOTS == 1) {
            for (uint32_t i = 0; i < count; i++) step(0, i);
        } else {
            for (uint32_t i = 0;; i += 2u) {
                step(0, i);
                if (i + 1u >= count) break;
                step(1, i + 1u);
                if (i + 2u >= count) break;
            }
        }
    }

    // ---- the W waves' sums: [wave][mt * NT + t][lane] of four rows each
    constexpr int kItems = MT * NT;
    constexpr bool OWN = kItems * 1024 <= kRegion * 2;              // a wave's sums fit over its own staging region
    constexpr uint32_t kWaveVecs = OWN ? kRegion / 8 : kItems * 64;
    // few sums: four waves finish a tile, a register (row of four) each, so that the eight reads of a sum are all there is in turn
    constexpr bool FINE = kItems <= 10;
    float4v *red = (float4v *)lds_all;
    if constexpr (!OWN) __syncthreads();   // (the sums lie over the staging regions of other waves)
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int i = 0; i < NT; i++) {
            if constexpr (FINE) {
#pragma unroll
                for (int r = 0; r < 4; r++) ((float *)lds_all)[(wave * kWaveVecs + (mt * NT + i) * 64u) * 4u + r * 64u + lane] = acc[mt][i][r];
            } else {
                red[wave * kWaveVecs + (mt * NT + i) * 64u + lane] = acc[mt][i];
            }
        }
    __syncthreads();
    auto total = [&](uint32_t item) {
        float4v s = red[item * 64u + lane];
#pragma unroll
        for (int w = 1; w < W; w++) s += red[w * kWaveVecs + item * 64u + lane];
        if constexpr (MODE == kRowsF32Few) {
            // rows 8 .. 15 hold the second terms, two row groups (32 lanes) further
#pragma unroll
            for (int w = 0; w < W; w++) s += red[w * kWaveVecs + item * 64u + (lane | 32u)];
        }
        return s;
    };
    auto total_of = [&](uint32_t item, uint32_t r) {
        const float *at = (const float *)lds_all + item * 256u + r * 64u;
        float s = at[lane];
#pragma unroll
        for (int w = 1; w < W; w++) s += at[w * kWaveVecs * 4u + lane];
        if constexpr (MODE == kRowsF32Few) {
#pragma unroll
            for (int w = 0; w < W; w++) s += at[w * kWaveVecs * 4u + (lane | 32u)];
        }
        return s;
    };
    const uint32_t n_ld = n_tiles * 16u;
    if (gated && !partials) {
        const uint32_t ffn = n >> 1;
        for (uint32_t unit = wave; unit < (FINE ? 4u : 1u) * MT * (NT / 2); unit += W) {
            const uint32_t it = FINE ? unit >> 2 : unit, mt = it / (NT / 2 ? NT / 2 : 1), t = it % (NT / 2 ? NT / 2 : 1);
            const float4v g = FINE ? float4v{total_of(mt * NT + t, unit & 3u), 0.f, 0.f, 0.f} : total(mt * NT + t);
            const float4v u = FINE ? float4v{total_of(mt * NT + t + NT / 2, unit & 3u), 0.f, 0.f, 0.f} : total(mt * NT + t + NT / 2);
            const uint32_t tile = tile_at(t), feat = paired_feature(tile * 16u + c);
            if (tile >= n_tiles || feat >= ffn || (MODE == kRowsF32Few && kb > 1u)) continue;
#pragma unroll
            for (int r = 0; r < (FINE ? 1 : 4); r++) {
                const uint32_t row = 16u * mt + 4u * kb + (FINE ? unit & 3u : (uint32_t)r);
                if (row < m_rows) out.swiglu[(size_t)row * ffn + feat] = gated_mul(out.gate_act, g[r], u[r]);
            }
        }
        return;
    }
    for (uint32_t unit = wave; unit < (FINE ? 4u : 1u) * kItems; unit += W) {
        const uint32_t it = FINE ? unit >> 2 : unit, mt = it / NT, t = it % NT;
        const float4v s = FINE ? float4v{total_of(it, unit & 3u), 0.f, 0.f, 0.f} : total(it);
        const uint32_t tile = tile_at(t), on = tile * 16u + c;
        if (tile >= n_tiles || (MODE == kRowsF32Few && kb > 1u)) continue;
        float *dst = nullptr;
        uint32_t ld = 0;
        float b = 0.f;
        bool has_b = false;
        if (partials) {
            dst = partials + (size_t)split * m_rows * n_ld + on;
            ld = n_ld;
        } else if (on < n) {
#pragma unroll
            for (uint32_t sg = 0; sg < kMaxSegs; sg++) {
                if (sg < out.count) {
                    const uint32_t rel = on - out.seg[sg].start;
                    if (rel < out.seg[sg].width) {
                        dst = out.seg[sg].ptr + rel;
                        ld = out.seg[sg].width;
                        if (out.seg[sg].bias) {
                            b = out.seg[sg].bias[rel];
                            has_b = true;
                        }
                    }
                }
            }
        }
        if (!dst) continue;
#pragma unroll
        for (int r = 0; r < (FINE ? 1 : 4); r++) {
            const uint32_t row = 16u * mt + 4u * kb + (FINE ? unit & 3u : (uint32_t)r);
            if (row < m_rows) dst[(size_t)row * ld] = has_b ? s[r] + b : s[r];
        }
    }
}

namespace {

template <int MT, int NT, int MODE, int W, int NV> struct WavesExact {
    static constexpr size_t staging = (size_t)W * ((MODE == kRowsF32 ? 2 : 1) * 16 * MT * kWeRow + (MODE ? 32 * MT : 0)) * sizeof(_Float16);
    static constexpr size_t sums = (size_t)W * MT * NT * 1024;
    static constexpr size_t lds = staging > sums ? staging : sums;
    static_assert(lds <= 160 * 1024, "");
    static hipError_t init()
    {
        if (lds <= 64 * 1024) return hipSuccess;
        return hipFuncSetAttribute((const void *)k_waves_exact<MT, NT, MODE, W, NV>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    }
    static hipError_t launch(hipStream_t s, const WeightView &w, const void *a, uint32_t m, const OutSpec &out, uint32_t splits, float *partials)
    {
        const uint32_t cps = (w.k_chunks + splits - 1) / splits;
        splits = (w.k_chunks + cps - 1) / cps;  // no empty split
        const bool gated = out.swiglu != nullptr;
        const uint32_t groups = (w.n_tiles + NT - 1) / NT;
        hipLaunchKernelGGL((k_waves_exact<MT, NT, MODE, W, NV>), dim3(splits, groups), dim3(64 * W), lds, s, (const uint4v *)w.qw, (const uint2v *)w.sc,
                           a, m, w.k, w.n_tiles, w.k_chunks, cps, gated && splits == 1 ? 1u : 0u, w.n, splits > 1 ? partials : nullptr, out);
        if (splits > 1) return launch_splitk_reduce(s, partials, out, m, w.n, w.n_tiles * 16, splits);
        return hipGetLastError();
    }
};

// The forms that exist, eight waves each; the two-tile f32 rows' registers end at eight column tiles (four with 17 .. 32 rows).
// fn gets the one of the runtime parameters (false: there is none), or every one in turn (mt = 0, until fn fails).
template <typename F> bool waves_exact_form(uint32_t mt, uint32_t nt, uint32_t mode, uint32_t quads, hipError_t &e, F &&fn)
{
    bool found = false;
    e = hipSuccess;
#define TWM_WAVES_ROWS(MT, NT, MODE, NV)                                                              \
    if (e == hipSuccess && (mt == 0 || (mt == MT && nt == NT && mode == MODE && quads == NV))) {      \
        found = true;                                                                                 \
        e = fn(WavesExact<MT, NT, MODE, 8, NV>{});                                                    \
    }
#define TWM_WAVES(MT, NT, MODE)                                                       \
    if constexpr (MT == 2) { TWM_WAVES_ROWS(MT, NT, MODE, 6) TWM_WAVES_ROWS(MT, NT, MODE, 8) }              \
    else if constexpr (MODE == kRowsF32Few) { TWM_WAVES_ROWS(MT, NT, MODE, 2) }                             \
    else if constexpr (MODE == kRowsF32) { TWM_WAVES_ROWS(MT, NT, MODE, 3) TWM_WAVES_ROWS(MT, NT, MODE, 4) } \
    else { TWM_WAVES_ROWS(MT, NT, MODE, 2) TWM_WAVES_ROWS(MT, NT, MODE, 3) TWM_WAVES_ROWS(MT, NT, MODE, 4) }
#define TWM_WAVES_4(MT, MODE) TWM_WAVES(MT, 1, MODE) TWM_WAVES(MT, 2, MODE) TWM_WAVES(MT, 3, MODE) TWM_WAVES(MT, 4, MODE)
#define TWM_WAVES_8(MT, MODE) TWM_WAVES_4(MT, MODE) TWM_WAVES(MT, 5, MODE) TWM_WAVES(MT, 6, MODE) TWM_WAVES(MT, 8, MODE)
    TWM_WAVES_8(1, kRowsF16) TWM_WAVES(1, 10, kRowsF16)
    TWM_WAVES_8(2, kRowsF16) TWM_WAVES(2, 10, kRowsF16)
    TWM_WAVES_8(1, kRowsF32Few) TWM_WAVES(1, 10, kRowsF32Few)
    TWM_WAVES_8(1, kRowsF32)
    TWM_WAVES_4(2, kRowsF32)
#undef TWM_WAVES_8
#undef TWM_WAVES_4
#undef TWM_WAVES
#undef TWM_WAVES_ROWS
    return found;
}

}  // namespace

// Once per device, outside any stream capture: the forms that ask for more than 64 KB of LDS.
hipError_t init_waves_exact()
{
    hipError_t e;
    waves_exact_form(0, 0, 0, 0, e, [](auto form) { return decltype(form)::init(); });
    return e;
}

// Whether this kernel takes a GEMM of 5 .. 32 rows (nt = 0: it does not), with how many tiles per workgroup and K-splits.
// Lines from forced sweeps of 72 projection shapes, 5 .. 32 rows, f16 and f32 (us, this kernel / the best other form):
// * vocabularies (more than 4096 tiles) stay with the forms whose workgroups are short-lived, except up to eight f32 rows
//   (3584 -> 152064 at 8 f16 rows 66 / 54, at 32 92 / 78, at 8 f32 rows 73 / 82), as do wide matrices of up to eight chunks
//   (896 -> 32000 at 16 rows 8.1 / 6.5);
// * so do f16 rows from where ten tiles each are more than one round of workgroups, 2560 tiles, at 9 .. 16 rows 2816 (2592 -> 51736
//   at 28 rows 35.6 / 25.2, 3840 -> 52422 at 17 38.0 / 32.7, 2496 -> 64331 at 10 24.0 / 19.4, 2592 -> 2 x 28832 at 5 23.5 / 18.9), and
//   f32 rows on a K that is shallow for it: up to eight rows four chunks, sixteen from 3840 tiles on (22 and 32 of them where the
//   last round of ten-tile groups is the emptiest, eight between 8000 and 9000 tiles, where the other form's is: 12 chunks 0.78 of its
//   time; 64 -> 84583 at 6 rows 19.2 / 10.2, 1184 -> 63459 at 8 18.6 / 17.0, 2080 -> 2 x 52384 at 6 39.1 / 36.1, 2400 -> 82295 at 5
//   42.4 / 36.9), nine and more 5 .. 9 chunks, to 18 from 2700 tiles on, to 31 from 3328 (576 -> 2 x 24608 at 10 rows 13.5 / 12.4,
//   1984 -> 59058 at 12 24.6 / 23.0);
// * 17 .. 32 f32 rows end at the four tiles their registers allow (1856 -> 2 x 9312 at 32 rows 20.9 / 17.3; 1024 tiles and
//   fewer are 5 - 50 % ahead) and at K of about 20000, 12800 above 340 tiles (17536 -> 5504 at 25 rows 36.5 / 31.6), 8192 above
//   680 and 5120 on 513 .. 680, whose groups of three leave the CUs 70 - 85 % full (28672 -> 8192 64 / 55, 8064 -> 9792 at 23
//   rows 30.5 / 25.6, 7296 -> 2 x 5280 at 27 30.7 / 27.0); nine rows and more on three chunks at 2048 tiles (128 -> 39553 at 16
//   rows 8.1 / 7.3);
// * f16, up to eight rows: the lane-per-column and streaming kernels keep 513 .. 1100 tiles (896 -> 2 x 4864 4.9 / 4.2; 820 .. 1024
//   tiles 2 - 17 % ahead) but for a deeper K on up to 820 of them (up to 700 tiles nine chunks and more: 3072 -> 8922 at 8 rows 7.2
//   / 8.1, 8448 -> 10775 at 8 13.3 / 16.8, gated from 33 on 0.97; up to 768, three tiles each, 33 and more: 5760 -> 11678 at 6 10.7 /
//   12.5; up to 820, four each, 49 and more: 9856 -> 12562 at 5 17.6 / 18.6, but 4640 -> 12716 at 5 11.1 / 10.6) and 17 chunks and
//   more above 1024, where their second round of workgroups is nearly empty (0.67 .. 0.89); 1537 .. 2048 tiles (3104 -> 28833 at 6
//   rows 14.1 / 12.8: eight tiles each leave the CUs 75 - 90 % full); K of 16 .. 32 chunks on 257 .. 512 tiles (2784 -> 4611 at 5 rows
//   5.45 / 5.0; but gated up to 340 tiles 0.89 .. 1.01 of k_gemv4s's time, 3200 -> 2 x 2336 at 8 rows 5.8 / 6.5, and up to 18 chunks
//   0.93); and up to six rows, seven up to K = 4096, every K from 2200 on with up to 256 tiles (3584 -> 3584 at 5 rows
//   5.2 / 4.6) but for more than 64 chunks on up to 128 (0.75 .. 0.87 of k_stream's time), gated 2048 .. 4096 at eight rows too,
//   where pairs of tiles are half as many workgroups (3072 -> 2 x 96 at 8 rows 4.75 / 4.24);
// * f16, 9 .. 12 and 17 .. 24 rows, whose row blocks are not loaded whole: a few more of the shapes below, against k_batch: three and
//   four chunks on up to 768 tiles (512 -> 12208 at 10 rows 4.2 / 4.5, 448 -> 11338 at 21 5.1 / 5.6; three chunks 0.91 .. 1.02), two
//   under a gate from 19 rows on (160 -> 2 x 4672 at 21 4.4 / 4.7; without one 160 -> 12385 at 24 5.2 / 4.6, and at 17 rows 160 -> 2 x
//   6080 4.5 / 4.3), nine to sixteen on 701 .. 768 tiles (2048 -> 11391 at 9 6.5 / 7.4, 1408 -> 12134 at 21 7.1 / 8.3), up to 820
//   under a gate and from 21 rows on (2016 -> 2 x 6464 at 21 8.9 / 10.2; but 1600 -> 12768 at 9 7.0 / 6.7), 33 and more on 1801 .. 2048
//   (5312 -> 29504 at 12 20.3 / 22.2, 8416 -> 2 x 15328 at 24 35.9 / 41.4);
// * f16, deep K on 129 .. 256 tiles: from 72 chunks on up to sixteen rows (12192 -> 3584 at 8 rows 11.0 / 10.0), up to 340 tiles
//   from 67 on (9216 -> 4352 at 11 rows 10.9 / 9.8, 13600 -> 2 x 2720 at 7 14.4 / 12.9), from 65 on above (17824 -> 3584 at 17 rows
//   16.8 / 15.6), gated from 61 on with 321 .. 400 tiles (10848 -> 2 x 2848 at 31 rows 20.0 / 17.9); f16 on a few
//   chunks: four on 513 tiles and more (256 -> 14049 at 10 rows 4.0 / 3.75), nine to sixteen on 701 .. 1000 (1600 -> 2 x 6560 at
//   11 rows 6.75 / 6.5, 1600 -> 14798 at 30 9.6 / 8.9), up to eighteen above 1600, 1536 up to sixteen rows and 1300 up to eight
//   (those up to ten): a wave has one to three chunks, unevenly, on seven to ten tiles (1152 -> 33728 at 19 rows 13.1 / 11.0, 1664
//   -> 24966 at 9 10.4 / 8.9, 1152 -> 38272 at 9 10.6 / 9.4); 1801 .. 2048 tiles (2752 -> 2 x 15104 at 17 rows 16.0 / 15.0)
//   and, up to sixteen rows, 961 .. 1024 (2752 -> 2 x 8192 at 12 rows 9.1 / 8.7).
// Within those lines the form comes from a small cost model, fitted to the same sweeps (root mean square error 6.5 %; its forms
// are 0.3 % above the best ones in the mean): a chunk costs a wave `fixed` + `tile` x nt us, more the longer the row of chunks;
// a launch takes the larger of that and of its weights at 5.8 TB/s; a K-split adds the launch of the sum kernel and its
// traffic, 1.2 us more under a gate (5344 -> 2 x 2784 at 13 f32 rows 12.8 split, 11.3 not).  Up to four tiles (3 excepted) a
// K-split is taken only up to 128 groups; from 32 chunks on, with f32 rows 28 up to sixteen rows and 16 above (3072 -> 128 at 25
// f16 rows 5.5 split, 5.0 not; 2336 -> 2 x 608 at 5 f32 rows 6.2 / 5.1; but 3712 -> 448 at 11 f32 rows 6.2 / 7.5), and with eight
// chunks and more to a range.  With the gated store as without it: the kernel that adds the ranges applies the gate (17824 -> 2 x
// 128 at 24 f32 rows 45.0 us on 8 workgroups, 11.4 on eight ranges of 16).
// 4000 random calls against the kernels of before, in the mean: f16 rows 0.95, gated 0.91, f32 rows 0.74, gated 0.71; 9 of them
// more than 6 % slower.
WavesPlan plan_waves_exact(uint32_t n_tiles, uint32_t k_chunks, uint32_t m, bool a_f32, bool gated)
{
    const WavesPlan none = {0, 0, 0};
    if (m < 5 || m > 32) return none;
    const bool few_f32 = a_f32 && m <= 8;
    if (n_tiles > 4096 && !few_f32) return none;
    if (few_f32 && n_tiles > 3840) {
        const uint32_t from = n_tiles > 8000 && n_tiles <= 9000 ? 8u : n_tiles > 5120 && n_tiles <= 5400 ? 32u : n_tiles > 6000 && n_tiles <= 7000 ? 22u : 16u;
        if (k_chunks <= from) return none;
    }
    if (a_f32) {
        if (few_f32 && n_tiles > 2560 && k_chunks <= 4) return none;
        if (!few_f32 && ((n_tiles > 2560 && k_chunks >= 5 && k_chunks <= 9) || (n_tiles > 2700 && k_chunks >= 10 && k_chunks <= 18) ||
                         (n_tiles > 3328 && k_chunks >= 19 && k_chunks <= 31))) return none;
        if (m > 16 && (n_tiles > 1024 || k_chunks > (n_tiles > 680 ? 64u : n_tiles > 512 ? 40u : n_tiles > 340 ? 100u : 160u))) return none;
        if (m > 8 && n_tiles > 2048 && k_chunks <= 3) return none;
    } else {
        if (n_tiles > (m <= 8 || m > 16 ? 2560u : 2816u)) return none;
        const bool part = (m >= 9 && m <= 12) || (m >= 17 && m <= 24);   // (a row block that is not loaded whole)
        if (k_chunks <= 8 && n_tiles > (k_chunks > 4 ? 1024u : part && k_chunks > (gated && m > 18 ? 1u : 2u) ? 768u : 512u)) return none;
        if (n_tiles > 128 && n_tiles <= (m <= 16 ? 340u : 256u) && k_chunks > (m > 16 ? 64u : n_tiles > 256 ? 66u : 71u)) return none;
        if (gated && m > 16 && n_tiles > 320 && n_tiles <= 400 && k_chunks > 60) return none;
        if (n_tiles > (!part ? 700u : gated || m > 20 ? 820u : 768u) && n_tiles <= 1000 && k_chunks > 8 && k_chunks <= 16) return none;
        if (n_tiles > 1800 && n_tiles <= 2048 && !(part && k_chunks > 32)) return none;
        if (n_tiles > (m <= 8 && k_chunks <= 10 ? 1300u : m <= 16 ? 1536u : 1600u) && k_chunks <= 18) return none;
        if (m <= 16 && n_tiles > 960 && n_tiles <= 1024) return none;
        if (m <= 8) {
            const bool deep = n_tiles > 1024 ? k_chunks > 16 : n_tiles <= 700 ? k_chunks > (gated ? 32u : 8u) : n_tiles <= 820 && k_chunks > (n_tiles <= 768 ? 32u : 48u) && !gated;
            if ((n_tiles > 512 && n_tiles <= 1100 && !deep) || (n_tiles > 1536 && n_tiles <= 2048)) return none;
            if (n_tiles > 256 && n_tiles <= 512 && k_chunks >= 16 && k_chunks <= 32 && !(gated && (n_tiles <= 340 || k_chunks <= 18))) return none;
            if (n_tiles <= 256 && k_chunks > 17 && (m <= 6 || (m == 7 && k_chunks <= 32)) && !(n_tiles <= 128 && k_chunks > 64)) return none;
            if (n_tiles <= 256 && gated && k_chunks >= 16 && k_chunks <= 31) return none;
        }
    }
    static const struct { double fixed, tile, longer, split, split_mb; } kCost[] = {
        {0.12, 0.31, 0.045, 1.9, 1.0}, {0.37, 0.42, 0.026, 1.2, 1.0}, {0.20, 0.35, 0.026, 1.4, 1.0}, {0.54, 0.39, 0.05, 1.7, 0.5}, {1.5, 0.55, 0.02, 1.7, 0.5}};
    const auto &cost = kCost[!a_f32 ? (m <= 16 ? 0 : 1) : few_f32 ? 2 : m <= 16 ? 3 : 4];
    const double bytes_us = (double)n_tiles * k_chunks * 1152.0 / 5.8e6;
    const uint32_t shallow = !a_f32 ? 32u : m <= 16 ? 28u : 16u;   // (K is not split below)
    WavesPlan best = none;
    double best_us = 1e30;
    for (uint32_t nt : {1u, 2u, 3u, 4u, 5u, 6u, 8u, 10u}) {
        if ((nt == 10 && a_f32 && !few_f32) || (nt > 4 && a_f32 && m > 16)) continue;
        const uint32_t groups = (n_tiles + nt - 1) / nt;
        const bool whole = nt == 1 || nt == 2 || nt == 4;
        if (whole && groups > 256 && !(nt == 4 && a_f32 && m > 16)) continue;
        for (uint32_t sp = 1; sp <= 8 && sp <= k_chunks; sp++) {
            const uint32_t cps = (k_chunks + sp - 1) / sp;
            if ((k_chunks + cps - 1) / cps != sp) continue;   // same work as a smaller factor
            if (gated && sp == 1 && nt % 2) continue;         // (a gate tile and its up tile lie in one workgroup)
            if (sp > 1 && (groups * sp > 256 || k_chunks < shallow || k_chunks / sp < 8 || (whole && groups > 128))) continue;
            const double e = 0.1 * ((cps + 7) / 8) + 0.9 * cps / 8.0;
            const double rounds = (double)((groups * sp + 255) / 256);
            const double work = rounds * e * (cost.fixed + cost.tile * nt) * (1.0 + cost.longer * e / nt);
            const double t4 = work * work * work * work + bytes_us * bytes_us * bytes_us * bytes_us;
            double t = __builtin_sqrt(__builtin_sqrt(t4));
            if (sp > 1) t += cost.split + (gated ? 1.2 : 0.0) + cost.split_mb * sp * m * n_tiles * 128.0e-6;
            if (t < best_us) {
                best_us = t;
                best = WavesPlan{nt, 8, sp};
            }
        }
    }
    return best;
}

// The largest count of column tiles up to nt that there is a form of at this row count and type.
uint32_t waves_exact_tiles(uint32_t nt, uint32_t m, bool a_f32)
{
    const uint32_t most = !a_f32 || m <= 8 ? 10u : m <= 16 ? 8u : 4u;
    if (nt > most) nt = most;
    return nt == 7 || nt == 9 ? nt - 1u : nt < 1 ? 1u : nt;
}

// Up to 32 rows.  nt: 16-column tiles per workgroup (1 .. 6, 8, 10 as the form has them; a gated store without a K-split needs an
// even number).  `scratch` holds the split-K sums; the split factor is cut to what fits.
hipError_t launch_waves_exact(hipStream_t s, const WeightView &w, const void *a, bool a_f32, uint32_t m, const OutSpec &out, uint32_t nt,
                              uint32_t splits, void *scratch, size_t scratch_bytes)
{
    if (m == 0 || w.n == 0) return hipSuccess;
    if (w.k_chunks == 0 || w.n_tiles % 4 != 0 || m > 32) return hipErrorInvalidValue;
    if (a_f32 && (uint64_t)m * w.k * 2 > 0x7FFFFFFFu) return hipErrorInvalidValue;   // (32-bit offsets into the rows)
    const uint32_t mode = !a_f32 ? kRowsF16 : m <= 8 ? kRowsF32Few : kRowsF32;
    const size_t per_split = (size_t)m * w.n_tiles * 16 * 4, left = scratch ? scratch_bytes : 0;
    if (splits > left / per_split) splits = (uint32_t)(left / per_split);
    if (splits > w.k_chunks) splits = w.k_chunks;
    if (splits < 1) splits = 1;
    if (out.swiglu && splits == 1 && nt % 2) nt++;
    hipError_t e;
    const uint32_t quads = m <= 8 ? 2u : m <= 12 ? 3u : m <= 16 ? 4u : m <= 24 ? 6u : 8u;
    const bool found = waves_exact_form(m <= 16 ? 1u : 2u, nt, mode, quads, e, [&](auto form) {
        return decltype(form)::launch(s, w, a, m, out, splits, (float *)scratch);
    });
    return found ? e : hipErrorInvalidValue;
}

}  // namespace twm
