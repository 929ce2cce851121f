// GEMM for 5 .. 192 rows on narrow matrices: waves that share nothing until the end, each on k-chunks of its own.
//
// Semantics: the kernels of twm_batch.hip.  Exact (RND = false, up to 32 rows): per 32-deep group the products a * (q - 8)
// are summed in f32 by one v_mfma_f32_16x16x32_f16 with a zero accumulator, the group sum is scaled once by f32(scale) and
// added to the running f32 sum (crates/kernels/src/quantize.rs:1219-1238); f32 rows enter as two f16 terms.  RND: the B
// operand is f16_rne(f32(scale) * (q - 8)) and the MFMAs accumulate over K (the reference's dequant-then-FP16-GEMM route,
// quantize.rs:534-571, 1825-1858; the arithmetic of the prefill GEMM).
//
// What bounds these launches is latency: 4 .. 20 MB of weights are read in one to three microseconds, and the kernels of
// twm_batch.hip and twm_prefill.hip spend longer on a chain of barriers, a K-split's partial sums and the launch that adds
// them.  So: a workgroup owns 16 NT columns for up to 16 MT rows and (nearly always) the whole K, with NT chosen so that
// one round of workgroups fills the CUs; its eight waves deal the 128-deep chunks among themselves.  A wave loads its
// chunk's activation tile (16 MT x 128 f16, sixteen lanes per row) into registers, writes it to an LDS region of its own
// (256-byte rows, XOR-swizzled 16-byte slots) and reads the MFMA operands back -- reading them from memory in operand order
// costs 3.5 times as much, 37 against 130 bytes per ns and CU, because sixteen lanes of a load then touch sixteen lines.
// No other wave reads that region, so the main loop has no barrier; one at the end, then all waves add the partial sums.
// Measured against the forms that ran before (f16 rows, us): 3584 -> 3584 at 16 rows 7.4 -> 5.6, 32 rows 9.5 -> 7.2, 64 rows
// 13.8 -> 10.3, 96 rows 16.1 -> 10.0; 4096 -> 6144 at 32 rows 12.0 -> 10.0; 2048 -> 2048 at 32 rows 9.3 -> 5.3, 128 rows
// 13.1 -> 7.7; 896 -> 1152 at 32 rows 6.6 -> 4.1; f32 rows: 3584 -> 3584 at 8 rows 10.7 -> 8.1, 2048 -> 2048 at 16 10.7 -> 7.7.
// Wider matrices have enough columns to share an activation tile between more of them and stay where they were.
#include "twm_device.h"

#include <type_traits>

namespace twm {

namespace {

__device__ __forceinline__ const TWM_GLOBAL char *wv_scalar_base(const void *p, size_t byte_offset)
{
    uint64_t v = (uint64_t)p + byte_offset;
    asm("" : "+s"(v));  // a uniform base kept in scalar registers: loads take saddr + 32-bit lane offset
    return (const TWM_GLOBAL char *)v;
}

struct WvConsts {
    uint32_t mask_lo, mask_hi, magic_lo, magic_hi;
};

// eight nibbles of word w -> eight f16 values (q - 8), exact
__device__ __forceinline__ half8 wv_unpack(uint32_t w, const WvConsts &c)
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

constexpr int kWvRow = 128;  // halves per LDS row (256 bytes)

}  // namespace

// TERMS = 2: f32 rows as two f16 tiles.  (Up to eight f32 rows need no second tile: `stacked`, the second terms are rows
// 8 .. 15 of the one block, which costs what eight f16 rows cost.)
template <int MT, int NT, int TERMS, int W, bool RND>
__global__ __launch_bounds__(64 * W) void k_waves(const uint4v *__restrict__ qw, const uint2v *__restrict__ sc,
                                                  const void *__restrict__ a_any, uint32_t m_total, uint32_t k, uint32_t n,
                                                  uint32_t n_tiles, uint32_t k_chunks, uint32_t chunks_per_split,
                                                  uint32_t row_blocks, uint32_t lo_offset, uint32_t stacked, float *__restrict__ partials, OutSpec out)
{
    constexpr int kTile = 16 * MT * kWvRow;      // halves of one term's activation tile
    constexpr int kRegion = TERMS * kTile;       // halves of a wave's LDS region
    constexpr int NV = 4 * MT;                   // 16-byte loads per lane, tile and term
    static_assert(MT * NT * 256 * 4 <= kRegion * 2, "the sums fit the staging region");
    extern __shared__ __attribute__((aligned(16))) _Float16 lds_all[];

    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t c = lane & 15u, kb = lane >> 4;
    _Float16 *region = lds_all + wave * kRegion;

    // The row blocks of a column group run next to each other on one XCD (workgroups reach the eight XCDs in turn), so
    // that the weights come from HBM once.
    uint32_t group = blockIdx.x, m0 = 0;
    if (row_blocks > 1u) {
        const uint32_t q = blockIdx.x >> 3;
        group = (q / row_blocks) * 8u + (blockIdx.x & 7u);
        m0 = (q % row_blocks) * (16u * MT);
        if (group * NT >= n_tiles) return;
    }
    const uint32_t m_rows = m_total - m0 < 16u * MT ? m_total - m0 : 16u * MT;
    const uint32_t kc0 = blockIdx.y * chunks_per_split;
    const uint32_t nchunks = k_chunks - kc0 < chunks_per_split ? k_chunks - kc0 : chunks_per_split;
    const uint32_t count = nchunks > wave ? (nchunks - wave + W - 1u) / W : 0u;  // this wave's chunks: wave, wave + W, ...

    // this group's tiles; with the gated store on two tiles, a gate tile and the up tile of the same features
    const bool gated = out.swiglu != nullptr && partials == nullptr;
    uint32_t tile_of[NT];
#pragma unroll
    for (int i = 0; i < NT; i++)
        tile_of[i] = NT == 2 && gated ? (group >> 1) * 4u + (group & 1u) + 2u * i : group * NT + i;

    WvConsts dq = {0x000F000Fu, 0x00F000F0u, 0x64006400u, 0x54005400u};
    asm volatile("" : "+s"(dq.mask_lo), "+s"(dq.mask_hi), "+v"(dq.magic_lo), "+v"(dq.magic_hi));

    float4v acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int i = 0; i < NT; i++) acc[mt][i] = float4v{0.f, 0.f, 0.f, 0.f};

    // Load j of the tile takes rows 4 j .. 4 j + 3: lane L row 4 j + L / 16, vector (L % 16) ^ (row % 16) of its sixteen,
    // and writes it to slot L % 16 of that row.  Rows past m_rows replay the last row and are never stored; vectors past K
    // replay the row's first vector of the chunk, where the padded weights are zero -- and, up to sixteen f16 rows, are staged
    // as zeros: an infinity in that vector times a zero weight would make the row's sums NaN.  (Above that k_batch and
    // k_prefill, which take these rows on other shapes, replay it as well; there the masks cost 1 % of the launch.)
    const char *a_blk = (const char *)a_any + (size_t)m0 * k * 2u;
    uint32_t a_off[NV], a_vec[4];
#pragma unroll
    for (int j = 0; j < 4; j++) a_vec[j] = (lane & 15u) ^ (4u * j + (lane >> 4));
#pragma unroll
    for (int j = 0; j < NV; j++) {
        uint32_t row = 4u * j + (lane >> 4);
        const bool second = stacked && row >= 8u;   // (row r + 8 holds the second term of row r)
        if (second) row -= 8u;
        row = row < m_rows ? row : m_rows - 1;
        a_off[j] = (row * k + a_vec[j & 3] * 8u) * 2u + (second ? lo_offset : 0u);
    }
    const uint32_t q_off = lane * 16u, s_off = c * 8u;
    uint4v ar[TERMS][NV];
    uint4v wq[2][NT];
    uint2v ws[2][NT];
    // Chunk i of this wave.  Past the end every lane reads the first bytes of the wave's first chunk instead (one line per
    // load, never used): the loads are unconditional, so the compiler's count of loads in flight stays exact.
    auto chunk_at = [&](uint32_t i) { return kc0 + wave + (i < count ? i : 0u) * (uint32_t)W; };
    auto load_a = [&](uint32_t i) {
        const uint32_t kg = chunk_at(i), on = i < count ? 0xFFFFFFFFu : 0u;
#pragma unroll
        for (int t = 0; t < TERMS; t++) {
            const TWM_GLOBAL char *src = wv_scalar_base(a_blk, (size_t)t * lo_offset + (size_t)kg * 256u);
#pragma unroll
            for (int j = 0; j < NV; j++) {
                const uint32_t back = kg * 128u + a_vec[j & 3] * 8u < k ? 0u : a_vec[j & 3] * 16u;
                ar[t][j] = *(const TWM_GLOBAL uint4v *)(src + ((a_off[j] - back) & on));
            }
        }
    };
    auto load_b = [&](int slot, uint32_t i) {
        const uint32_t kg = chunk_at(i), on = i < count ? 0xFFFFFFFFu : 0u;
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const size_t tile = (size_t)kg * n_tiles + tile_of[t];
            wq[slot][t] = __builtin_nontemporal_load((const TWM_GLOBAL uint4v *)(wv_scalar_base(qw, tile * 1024u) + (q_off & on)));
            ws[slot][t] = __builtin_nontemporal_load((const TWM_GLOBAL uint2v *)(wv_scalar_base(sc, tile * 128u) + (s_off & on)));
        }
    };
    auto stage_a = [&](uint32_t i) {
        if constexpr (MT == 1 && TERMS == 1) {
            const uint32_t left = k - chunk_at(i) * 128u;  // the row's values from this chunk on
            if (left < 128u) {
#pragma unroll
                for (int j = 0; j < NV; j++) ar[0][j] = a_vec[j & 3] * 8u < left ? ar[0][j] : uint4v{0u, 0u, 0u, 0u};
            }
        }
#pragma unroll
        for (int t = 0; t < TERMS; t++)
#pragma unroll
            for (int j = 0; j < NV; j++) *(uint4v *)(region + t * kTile + j * 512 + lane * 8u) = ar[t][j];
    };
    uint32_t rd_off[4];  // row c of a row block, vector 4 g + kb of the chunk -> slot (4 g + kb) ^ c
#pragma unroll
    for (int g = 0; g < 4; g++) rd_off[g] = c * kWvRow + (((4u * g + kb) ^ c) * 8u);

    // The chunk's 4 NT (group, tile) units in turn: a unit's MFMAs are followed by the next unit's unpack and then by its own
    // scaling, so that the matrix pipe's latency passes under the unpack; the next group's operands are read one unit ahead.
    auto scale_of = [&](int slot, int u) {
        union { uint32_t u32; half2v h; } pair;
        pair.u32 = ws[slot][u % NT][(u / NT) >> 1];
        return pair.h[(u / NT) & 1];
    };
    auto operand = [&](int slot, int u) {
        half8 bf = wv_unpack(wq[slot][u % NT][u / NT], dq);
        if constexpr (RND) {
            union { half8 h; half2v h2[4]; } bw;
            bw.h = bf;
            const _Float16 sc16 = scale_of(slot, u);
            const half2v s2 = {sc16, sc16};
#pragma unroll
            for (int j = 0; j < 4; j++) bw.h2[j] *= s2;
            bf = bw.h;
        }
        return bf;
    };
    auto compute = [&](int slot) {
        half8 af[2][TERMS][MT];
        auto read_a = [&](int g) {
#pragma unroll
            for (int t = 0; t < TERMS; t++)
#pragma unroll
                for (int mt = 0; mt < MT; mt++) af[g & 1][t][mt] = *(const half8 *)(region + t * kTile + mt * 16 * kWvRow + rd_off[g]);
        };
        read_a(0);
        half8 bf = operand(slot, 0);
#pragma unroll
        for (int u = 0; u < 4 * NT; u++) {
            const int g = u / NT, i = u % NT;
            if (i == 0 && g < 3) read_a(g + 1);
            float4v d[MT];
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                if constexpr (RND) acc[mt][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[g & 1][0][mt], bf, acc[mt][i], 0, 0, 0);
                else d[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[g & 1][0][mt], bf, float4v{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            }
            if constexpr (TERMS == 2) {
#pragma unroll
                for (int mt = 0; mt < MT; mt++) d[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[g & 1][1][mt], bf, d[mt], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            half8 bn = bf;
            if (u + 1 < 4 * NT) bn = operand(slot, u + 1);
            if constexpr (!RND) {
                const float scale = (float)scale_of(slot, u);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[mt][i][r] += d[mt][r] * scale;
            }
            __builtin_amdgcn_sched_barrier(0);
            bf = bn;
        }
    };

    // Chunk i: its tile goes from the registers to LDS, the registers take the loads of tile i + 1; the chunk is computed
    // from LDS and weight slot i % 2, which then takes the loads of chunk i + 2.
    if (count) {
        load_a(0);
        load_b(0, 0);
        load_b(1, 1);
        __builtin_amdgcn_sched_barrier(0);
        auto step = [&](int slot, uint32_t i) {
            stage_a(i);
            __builtin_amdgcn_sched_barrier(0);
            load_a(i + 1u);
            __builtin_amdgcn_sched_barrier(0);
            compute(slot);
            __builtin_amdgcn_sched_barrier(0);
            load_b(slot, i + 2u);
            __builtin_amdgcn_sched_barrier(0);
        };
        for (uint32_t i = 0;; i += 2u) {
            step(0, i);
            if (i + 1u >= count) break;
            step(1, i + 1u);
            if (i + 2u >= count) break;
        }
    }

    // ---- the W waves' sums: register (mt, i, r) of lane (c, kb) is row 16 mt + 4 kb + r, column 16 i + c of the group
    float *red = (float *)lds_all;
    constexpr uint32_t kWaveFloats = kRegion / 2;   // (a wave writes its sums over its own tile)
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int i = 0; i < NT; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) red[wave * kWaveFloats + ((mt * NT + i) * 4 + r) * 64u + lane] = acc[mt][i][r];
    __syncthreads();
    constexpr uint32_t kCols = 16u * NT;
    const uint32_t n_ld = n_tiles * 16u;
    auto second_term = [&](uint32_t src) {  // of f32 rows in one block: rows 8 .. 15 hold the second terms, two row groups (32 lanes) further
        float s = red[src + 32u];
#pragma unroll
        for (int w = 1; w < W; w++) s += red[w * kWaveFloats + src + 32u];
        return s;
    };
    for (uint32_t idx = threadIdx.x; idx < 16u * MT * kCols; idx += 64u * W) {
        const uint32_t row = idx / kCols, col = idx % kCols, t = col >> 4;
        if (row >= m_rows) continue;
        const uint32_t reg = ((row >> 4) * NT + t) * 4u + (row & 3u), src = reg * 64u + ((row & 15u) >> 2) * 16u + (col & 15u);
        float s = red[src];
#pragma unroll
        for (int w = 1; w < W; w++) s += red[w * kWaveFloats + src];
        if (stacked) s += second_term(src);
        const uint32_t tile = NT == 2 && gated ? (group >> 1) * 4u + (group & 1u) + 2u * t : group * NT + t;
        const uint32_t on = tile * 16u + (col & 15u), om = m0 + row;
        if (partials) {
            partials[((size_t)blockIdx.y * m_total + om) * n_ld + on] = s;
            continue;
        }
        const float rs = out.row_scale ? out.row_scale[om] : 1.f;  // (f32 rows scaled into the f16 range)
        s *= rs;
        if (gated) {
            // the group's first half holds gate columns, its second half the up columns of the same features
            if (NT > 1 && t < NT / 2) {
                constexpr uint32_t kUp = NT / 2 * 4u * 64u;
                float u = red[src + kUp];
#pragma unroll
                for (int w = 1; w < W; w++) u += red[w * kWaveFloats + src + kUp];
                if (stacked) u += second_term(src + kUp);
                const uint32_t ffn = n >> 1, feat = paired_feature(on);
                if (feat < ffn) out.swiglu[(size_t)om * ffn + feat] = gated_mul(out.gate_act, s, u * rs);
            }
        } else if (on < n) {
#pragma unroll
            for (uint32_t sg = 0; sg < kMaxSegs; sg++) {
                if (sg < out.count) {
                    const uint32_t rel = on - out.seg[sg].start;
                    if (rel < out.seg[sg].width) out.seg[sg].ptr[(size_t)om * out.seg[sg].width + rel] = out.seg[sg].bias ? s + out.seg[sg].bias[rel] : s;
                }
            }
        }
    }
}

namespace {

template <int MT, int NT, int TERMS, int W, bool RND> struct Waves {
    static constexpr size_t lds = (size_t)W * TERMS * 16 * MT * kWvRow * sizeof(_Float16);
    static_assert(lds <= 160 * 1024 && !(RND && TERMS == 2), "");
    static hipError_t init()
    {
        if (lds <= 64 * 1024) return hipSuccess;
        return hipFuncSetAttribute((const void *)k_waves<MT, NT, TERMS, W, RND>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    }
    static hipError_t launch(hipStream_t s, const WeightView &w, const void *a, uint32_t m, const OutSpec &out, uint32_t splits,
                             float *partials, uint32_t lo_offset, bool stacked)
    {
        const uint32_t cps = (w.k_chunks + splits - 1) / splits;
        splits = (w.k_chunks + cps - 1) / cps;  // no empty split
        const uint32_t groups = w.n_tiles / NT, row_blocks = (m + 16 * MT - 1) / (16 * MT);
        const uint32_t gx = row_blocks > 1 ? (groups + 7) / 8 * 8 * row_blocks : groups;
        hipLaunchKernelGGL((k_waves<MT, NT, TERMS, W, RND>), dim3(gx, splits), dim3(64 * W), lds, s, (const uint4v *)w.qw, (const uint2v *)w.sc,
                           a, m, w.k, w.n, w.n_tiles, w.k_chunks, cps, row_blocks, lo_offset, stacked ? 1u : 0u,
                           splits > 1 ? partials : nullptr, out);
        if (splits > 1) return launch_splitk_reduce(s, partials, out, m, w.n, w.n_tiles * 16, splits);
        return hipGetLastError();
    }
};

// The forms that exist: eight waves; 64 f32 rows' worth of registers end at two tiles per workgroup.  fn gets the one of
// the runtime parameters (false: there is none), or every one in turn (mt = 0, until fn fails).
template <typename F> bool waves_form(uint32_t mt, uint32_t nt, uint32_t terms, uint32_t waves, hipError_t &e, F &&fn)
{
    bool found = false;
    e = hipSuccess;
#define TWM_WAVES(MT, NT, T, W, R)                                                                     \
    if (e == hipSuccess && (mt == 0 || (mt == MT && nt == NT && terms == T && waves == W))) {         \
        found = true;                                                                                  \
        e = fn(Waves<MT, NT, T, W, R>{});                                                              \
    }
    TWM_WAVES(1, 1, 1, 8, false) TWM_WAVES(1, 2, 1, 8, false) TWM_WAVES(1, 4, 1, 8, false)
    TWM_WAVES(2, 1, 1, 8, false) TWM_WAVES(2, 2, 1, 8, false) TWM_WAVES(2, 4, 1, 8, false)
    TWM_WAVES(1, 1, 2, 8, false) TWM_WAVES(1, 2, 2, 8, false) TWM_WAVES(1, 4, 2, 8, false)
    TWM_WAVES(2, 1, 2, 8, false) TWM_WAVES(2, 2, 2, 8, false)
    TWM_WAVES(3, 1, 1, 8, true) TWM_WAVES(3, 2, 1, 8, true) TWM_WAVES(3, 2, 1, 4, true)
    TWM_WAVES(4, 1, 1, 8, true) TWM_WAVES(4, 2, 1, 8, true) TWM_WAVES(4, 2, 1, 4, true)
#undef TWM_WAVES
    return found;
}

// 16-row blocks per workgroup: one or two up to 32 rows, above that three or four, whichever pads less
uint32_t waves_mt(uint32_t m)
{
    if (m <= 32) return m <= 16 ? 1u : 2u;
    return (m + 47) / 48 * 48 < (m + 63) / 64 * 64 ? 3u : 4u;
}

}  // namespace

uint32_t waves_block_rows(uint32_t m) { return 16u * waves_mt(m); }

// Once per device, outside any stream capture: the forms that ask for more than 64 KB of LDS.
hipError_t init_waves()
{
    hipError_t e;
    waves_form(0, 0, 0, 0, e, [](auto form) { return decltype(form)::init(); });
    return e;
}

// Where this kernel takes a GEMM, and in which form; nt = 0: it does not.  Lines fitted to forced sweeps on twenty projection
// shapes and redrawn after a comparison with the forms of before on 3000 random ones, 5 .. 192 rows, f16 and f32 rows (us, this
// kernel against the best other form):
// * one round of workgroups on 256 CUs: one tile each up to 4096 columns, two up to 8192, four up to 16384 (beyond, the
//   forms that share the activation tile among more columns are level or ahead: 4096 -> 22016 gated at 32 rows 22.8 / 21.0);
//   four tiles only from K = 3072 on (4096 -> 12288 at 32 rows 14.0 / 15.6, but 2048 -> 11264 gated at 16 7.9 / 7.4) -- except
//   up to eight f32 rows (2048 -> 11264 gated 10.2 / 11.1), and not for 17 .. 32 f32 rows (25.2 / 23.6);
// * deep K: up to 8192 with f16 rows and 16 of them (11008 -> 4096 level), 6144 with more or with f32 rows (11008 -> 4096 at
//   32 rows 15.0 / 14.5), 4608 with 17 .. 32 f32 rows on two tiles (5120 -> 5120 18.9 / 18.2), any depth with up to eight f32 rows (18944 -> 3584 20.2 / 20.7, 11008 -> 4096 14.4 / 15.5);
// * up to six f16 rows, seven up to K = 4096, or eight on more than one tile, the lane-per-column sub-tiles are ahead from
//   K = 2048 on (3584 -> 3584 at 5 rows 5.3 / 4.8, 4096 -> 4096 at 7 rows 6.2 / 5.9, at 8 rows 6.2 / 6.1, 4224 -> 896 at 7
//   rows 5.7 / 6.2); up to eight f16 rows on more than one tile the streaming kernel is on K of 800 .. 1024 (896 -> 8192 at 5
//   rows 4.8 / 4.6, 1024 -> 6144 gated at 7 rows 5.1 / 4.7; 640 -> 5120 4.2 / 4.4, 1536 -> 8192 5.6 / 5.7) and on more than
//   6144 gated columns of a shallower K (512 -> 8192 gated at 8 rows 4.4 / 4.2);
// * K is cut only where few workgroups would run, each range keeping eight chunks and more: four ways up to 64 of them
//   (4864 -> 896 at 32 rows 6.9 on four, 8.3 the other form), two ways up to 128 with up to eight f32 rows on K above 12288
//   and up to 112 above 32 rows;
// * above 32 rows: while one or two tiles make one round (3584 -> 3584 at 128 rows 12.0 / 17.4, at 192 18.8 / 17.6), which
//   with several row blocks is 32 workgroups on each XCD, column groups being dealt eight at a time: 2656 -> 2656 at 192 rows
//   is 252 workgroups, but 33 of them on four of the XCDs (20.2 / 13.1), and 5120 -> 320 at 160 rows on four K-ranges 36 on
//   each (13.3, on two 10.5).  K up to 6144, above 4096 only with most CUs busy (5632 -> 2048 at 64 rows 11.7 / 11.1, at 128
//   13.4 / 17.0); 33 .. 64 rows on a shallow K also two rounds of four-wave workgroups (2048 -> 11264 gated at 64 rows 15.8 /
//   17.9).  The lower line, K of about 1024, is where the sweep above 32 rows began and not where the other forms get ahead:
//   896 -> 1152 at 64 rows takes 5.4 here and 9.7 on the prefill GEMM's blocks, where it still runs.
WavesPlan plan_waves(uint32_t n_tiles, uint32_t k_chunks, uint32_t m, bool a_f32, bool gated)
{
    const WavesPlan none = {0, 0, 0};
    if (m < 5 || m > 192) return none;
    if (m <= 32) {
        const bool few_f32 = a_f32 && m <= 8;
        uint32_t nt = n_tiles <= 256 ? 1u : n_tiles <= 512 ? 2u : n_tiles <= 1024 ? 4u : 0u;
        if (gated && nt == 1) nt = 2;
        if (nt == 0 || (nt == 4 && !few_f32 && (k_chunks < 24 || (a_f32 && m > 16)))) return none;
        if (!a_f32 && m <= 8) {
            if (k_chunks >= 16 && (m <= 6 || nt > 1 || (m == 7 && k_chunks <= 32))) return none;
            if (k_chunks <= 8 && nt > 1 && (k_chunks >= 7 || (gated && n_tiles > 384))) return none;
        }
        if (!few_f32 && k_chunks > (!a_f32 && m <= 16 ? 64u : a_f32 && m > 16 && nt == 2 ? 36u : 48u)) return none;
        const uint32_t groups = n_tiles / nt;
        uint32_t splits = 1;
        if (groups <= 64 && k_chunks >= 32 && (m > 16 || (a_f32 && m > 8))) splits = 4;
        if (few_f32 && groups <= 128 && k_chunks > 96) splits = 2;
        return WavesPlan{nt, 8, splits};
    }
    if (k_chunks < 8 || k_chunks > 48) return none;
    const uint32_t blocks = (m + 16 * waves_mt(m) - 1) / (16 * waves_mt(m));
    for (uint32_t nt = gated ? 2 : 1; nt <= 2; nt++) {
        const uint32_t groups = n_tiles / nt * blocks, on_xcd = (n_tiles / nt + 7) / 8 * blocks;
        if (on_xcd > 32) continue;
        const uint32_t splits = k_chunks < 32 ? 1u : on_xcd <= 8 ? 4u : groups <= 112 ? 2u : 1u;
        if (k_chunks > 32 && splits == 1 && groups < 160) return none;
        return WavesPlan{nt, 8, splits};
    }
    if (m <= 64 && k_chunks <= 16 && n_tiles <= 768) return WavesPlan{2, 4, 1};
    return none;
}

// nt: 16-column tiles per workgroup (1, 2, 4; a gated store without a K-split needs 2 or 4), waves per workgroup (8; 4 with
// more than 32 rows on two tiles).  Up to 32 rows exact weights, f32 rows as two f16 terms; above that f16-rounded weights
// and one term.  `scratch` holds the row factors and f16 terms of f32 rows and behind them the split-K sums; the split
// factor is cut to what fits.
hipError_t launch_waves(hipStream_t s, const WeightView &w, const void *a, bool a_f32, uint32_t m, const OutSpec &out_in, uint32_t nt,
                        uint32_t waves, uint32_t splits, void *scratch, size_t scratch_bytes)
{
    if (m == 0 || w.n == 0) return hipSuccess;
    if (w.k_chunks == 0 || w.n_tiles % 4 != 0) return hipErrorInvalidValue;
    uint32_t terms = a_f32 && m <= 32 ? 2u : 1u;
    OutSpec out = out_in;
    uint32_t lo_offset = 0;
    char *free_at = (char *)scratch;
    size_t left = scratch ? scratch_bytes : 0;
    if (a_f32) {
        const size_t term_bytes = (((size_t)m * w.k * 2) + 255) & ~(size_t)255, factors = ((size_t)m * 4 + 255) & ~(size_t)255;
        if (left < factors + terms * term_bytes || term_bytes > 0x7FFFFFFFu) return hipErrorInvalidValue;
        float *row_scale = (float *)free_at;
        _Float16 *hi = (_Float16 *)(free_at + factors), *lo = terms == 2 ? (_Float16 *)(free_at + factors + term_bytes) : nullptr;
        hipError_t e = launch_f32_rows_to_f16(s, (const float *)a, hi, lo, row_scale, m, w.k);
        if (e != hipSuccess) return e;
        a = hi;
        out.row_scale = row_scale;
        lo_offset = (uint32_t)term_bytes;
        free_at += factors + terms * term_bytes;
        left -= factors + terms * term_bytes;
    }
    const bool stacked = terms == 2 && m <= 8;
    if (stacked) terms = 1;
    const size_t per_split = (size_t)m * w.n_tiles * 16 * 4;
    if (splits > left / per_split) splits = (uint32_t)(left / per_split);
    if (splits > w.k_chunks) splits = w.k_chunks;
    if (splits < 1) splits = 1;
    if (out.swiglu && splits == 1 && nt == 1) nt = 2;
    hipError_t e;
    const bool found = waves_form(waves_mt(m), nt, terms, waves, e, [&](auto form) {
        return decltype(form)::launch(s, w, a, m, out, splits, (float *)free_at, lo_offset, stacked);
    });
    return found ? e : hipErrorInvalidValue;
}

}  // namespace twm
