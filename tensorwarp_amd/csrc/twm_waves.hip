// GEMM for 33 .. 192 rows on narrow matrices: waves that share nothing until the end, each on k-chunks of its own.
//
// Semantics: the B operand is f16_rne(f32(scale) * (q - 8)) and the MFMAs accumulate over K (the reference's
// dequant-then-FP16-GEMM route, quantize.rs:534-571, 1825-1858; the arithmetic of the prefill GEMM).  Up to 32 rows
// k_waves_exact (twm_waves_exact.hip) has the same structure with exact weights.
//
// What bounds these launches is latency: 4 .. 20 MB of weights are read in one to three microseconds, and the prefill GEMM
// spends longer on a chain of barriers, a K-split's partial sums and the launch that adds them.  So: a workgroup owns 16 NT
// columns for up to 16 MT rows and (nearly always) the whole K, with NT chosen so that one round of workgroups fills the
// CUs; its waves deal the 128-deep chunks among themselves.  A wave loads its chunk's activation tile (16 MT x 128 f16,
// sixteen lanes per row) into registers, writes it to an LDS region of its own (256-byte rows, XOR-swizzled 16-byte slots)
// and reads the MFMA operands back -- reading them from memory in operand order costs 3.5 times as much, 37 against 130
// bytes per ns and CU, because sixteen lanes of a load then touch sixteen lines.  No other wave reads that region, so the
// main loop has no barrier; one at the end, then all waves add the partial sums.
// Measured against the prefill GEMM, which ran before (f16 rows, us): 3584 -> 3584 at 64 rows 13.8 -> 10.3, 96 rows 16.1 ->
// 10.0; 2048 -> 2048 at 128 rows 13.1 -> 7.7.
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

template <int MT, int NT, int W>
__global__ __launch_bounds__(64 * W) void k_waves(const uint4v *__restrict__ qw, const uint2v *__restrict__ sc,
                                                  const void *__restrict__ a_any, uint32_t m_total, uint32_t k, uint32_t n,
                                                  uint32_t n_tiles, uint32_t k_chunks, uint32_t chunks_per_split,
                                                  uint32_t row_blocks, float *__restrict__ partials, OutSpec out)
{
    constexpr int kRegion = 16 * MT * kWvRow;    // halves of a wave's LDS region: its activation tile
    constexpr int NV = 4 * MT;                   // 16-byte loads per lane and tile
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
    // replay the row's first vector of the chunk, where the padded weights are zero (as k_prefill does, which takes these
    // rows on other shapes).
    const char *a_blk = (const char *)a_any + (size_t)m0 * k * 2u;
    uint32_t a_vec[4];
#pragma unroll
    for (int j = 0; j < 4; j++) a_vec[j] = (lane & 15u) ^ (4u * j + (lane >> 4));
    // (found from an opaque row for each chunk: with the sixteen offsets held by name the 64-row form spilled, 8.9 -> 9.9 us on
    // 1664 -> 1664 at 187 rows)
    uint32_t row_bytes = k * 2u, quad_row = (lane >> 4);
    asm volatile("" : "+v"(quad_row));
    const uint32_t q_off = lane * 16u, s_off = c * 8u;
    uint4v ar[NV];
    uint4v wq[2][NT];
    uint2v ws[2][NT];
    // Chunk i of this wave.  Past the end every lane reads the first bytes of the wave's first chunk instead (one line per
    // load, never used): the loads are unconditional, so the compiler's count of loads in flight stays exact.
    auto chunk_at = [&](uint32_t i) { return kc0 + wave + (i < count ? i : 0u) * (uint32_t)W; };
    auto load_a = [&](uint32_t i) {
        const uint32_t kg = chunk_at(i), on = i < count ? 0xFFFFFFFFu : 0u;
        const TWM_GLOBAL char *src = wv_scalar_base(a_blk, (size_t)kg * 256u);
#pragma unroll
        for (int j = 0; j < NV; j++) {
            const uint32_t vec = kg * 128u + a_vec[j & 3] * 8u < k ? a_vec[j & 3] * 16u : 0u;
            const uint32_t row = 4u * j + quad_row;
            ar[j] = *(const TWM_GLOBAL uint4v *)(src + (((row < m_rows ? row : m_rows - 1u) * row_bytes + vec) & on));
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
    auto stage_a = [&]() {
#pragma unroll
        for (int j = 0; j < NV; j++) *(uint4v *)(region + j * 512 + lane * 8u) = ar[j];
    };
    uint32_t rd_off[4];  // row c of a row block, vector 4 g + kb of the chunk -> slot (4 g + kb) ^ c
#pragma unroll
    for (int g = 0; g < 4; g++) rd_off[g] = c * kWvRow + (((4u * g + kb) ^ c) * 8u);

    // The chunk's 4 NT (group, tile) units in turn: a unit's MFMAs are followed by the next unit's unpack, so that the matrix
    // pipe's latency passes under it; the next group's operands are read one unit ahead.
    auto operand = [&](int slot, int u) {
        union { half8 h; half2v h2[4]; } bw;
        bw.h = wv_unpack(wq[slot][u % NT][u / NT], dq);
        union { uint32_t u32; half2v h; } pair;
        pair.u32 = ws[slot][u % NT][(u / NT) >> 1];
        const _Float16 sc16 = pair.h[(u / NT) & 1];
        const half2v s2 = {sc16, sc16};
#pragma unroll
        for (int j = 0; j < 4; j++) bw.h2[j] *= s2;
        return bw.h;
    };
    auto compute = [&](int slot) {
        half8 af[2][MT];
        auto read_a = [&](int g) {
#pragma unroll
            for (int mt = 0; mt < MT; mt++) af[g & 1][mt] = *(const half8 *)(region + mt * 16 * kWvRow + rd_off[g]);
        };
        read_a(0);
        half8 bf = operand(slot, 0);
#pragma unroll
        for (int u = 0; u < 4 * NT; u++) {
            const int g = u / NT, i = u % NT;
            if (i == 0 && g < 3) read_a(g + 1);
#pragma unroll
            for (int mt = 0; mt < MT; mt++) acc[mt][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[g & 1][mt], bf, acc[mt][i], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            half8 bn = bf;
            if (u + 1 < 4 * NT) bn = operand(slot, u + 1);
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
            stage_a();
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
    for (uint32_t idx = threadIdx.x; idx < 16u * MT * kCols; idx += 64u * W) {
        const uint32_t row = idx / kCols, col = idx % kCols, t = col >> 4;
        if (row >= m_rows) continue;
        const uint32_t reg = ((row >> 4) * NT + t) * 4u + (row & 3u), src = reg * 64u + ((row & 15u) >> 2) * 16u + (col & 15u);
        float s = red[src];
#pragma unroll
        for (int w = 1; w < W; w++) s += red[w * kWaveFloats + src];
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

template <int MT, int NT, int W> struct Waves {
    static constexpr size_t lds = (size_t)W * 16 * MT * kWvRow * sizeof(_Float16);
    static_assert(lds <= 160 * 1024, "");
    static hipError_t init()
    {
        if (lds <= 64 * 1024) return hipSuccess;
        return hipFuncSetAttribute((const void *)k_waves<MT, NT, W>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    }
    static hipError_t launch(hipStream_t s, const WeightView &w, const void *a, uint32_t m, const OutSpec &out, uint32_t splits,
                             float *partials)
    {
        const uint32_t cps = (w.k_chunks + splits - 1) / splits;
        splits = (w.k_chunks + cps - 1) / cps;  // no empty split
        const uint32_t groups = w.n_tiles / NT, row_blocks = (m + 16 * MT - 1) / (16 * MT);
        const uint32_t gx = row_blocks > 1 ? (groups + 7) / 8 * 8 * row_blocks : groups;
        hipLaunchKernelGGL((k_waves<MT, NT, W>), dim3(gx, splits), dim3(64 * W), lds, s, (const uint4v *)w.qw, (const uint2v *)w.sc,
                           a, m, w.k, w.n, w.n_tiles, w.k_chunks, cps, row_blocks, splits > 1 ? partials : nullptr, out);
        if (splits > 1) return launch_splitk_reduce(s, partials, out, m, w.n, w.n_tiles * 16, splits);
        return hipGetLastError();
    }
};

// The forms that exist.  fn gets the one of the runtime parameters (false: there is none), or every one in turn (mt = 0, until
// fn fails).
template <typename F> bool waves_form(uint32_t mt, uint32_t nt, uint32_t waves, hipError_t &e, F &&fn)
{
    bool found = false;
    e = hipSuccess;
#define TWM_WAVES(MT, NT, W)                                                                           \
    if (e == hipSuccess && (mt == 0 || (mt == MT && nt == NT && waves == W))) {                       \
        found = true;                                                                                  \
        e = fn(Waves<MT, NT, W>{});                                                                    \
    }
    TWM_WAVES(3, 1, 8) TWM_WAVES(3, 2, 8) TWM_WAVES(3, 2, 4)
    TWM_WAVES(4, 1, 8) TWM_WAVES(4, 2, 8) TWM_WAVES(4, 2, 4)
#undef TWM_WAVES
    return found;
}

// 16-row blocks per workgroup: three or four, whichever pads less (up to 32 rows, k_waves_exact's one or two)
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
    waves_form(0, 0, 0, e, [](auto form) { return decltype(form)::init(); });
    return e;
}

// Where this kernel takes a GEMM of more than 32 rows, and in which form; nt = 0: it does not.  Lines fitted to forced sweeps on
// twenty projection shapes and redrawn after a comparison with the forms of before on 3000 random ones (us, this kernel
// against the best other form):
// * while one or two tiles make one round of workgroups (3584 -> 3584 at 128 rows 12.0 / 17.4, at 192 18.8 / 17.6), which
//   with several row blocks is 32 workgroups on each XCD, column groups being dealt eight at a time: 2656 -> 2656 at 192 rows
//   is 252 workgroups, but 33 of them on four of the XCDs (20.2 / 13.1), and 5120 -> 320 at 160 rows on four K-ranges 36 on
//   each (13.3, on two 10.5);
// * K is cut only where few workgroups would run, each range keeping eight chunks and more: four ways up to eight workgroups
//   on an XCD, two ways up to 112 in all;
// * K up to 6144, above 4096 only with most CUs busy (5632 -> 2048 at 64 rows 11.7 / 11.1, at 128 13.4 / 17.0); 33 .. 64 rows
//   on a shallow K also two rounds of four-wave workgroups (2048 -> 11264 gated at 64 rows 15.8 / 17.9).  The lower line, K of
//   about 1024, is where the sweep began and not where the other forms get ahead: 896 -> 1152 at 64 rows takes 5.4 here and
//   9.7 on the prefill GEMM's blocks, where it still runs.
WavesPlan plan_waves(uint32_t n_tiles, uint32_t k_chunks, uint32_t m, bool gated)
{
    const WavesPlan none = {0, 0, 0};
    if (m <= 32 || m > 192) return none;
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

// More than 32 rows.  nt: 16-column tiles per workgroup (1, 2; a gated store without a K-split needs 2), waves per workgroup
// (8; 4 on two tiles).  `scratch` holds the row factors and f16 rows of f32 activations and behind them the split-K sums; the
// split factor is cut to what fits.
hipError_t launch_waves(hipStream_t s, const WeightView &w, const void *a, bool a_f32, uint32_t m, const OutSpec &out_in, uint32_t nt,
                        uint32_t waves, uint32_t splits, void *scratch, size_t scratch_bytes)
{
    if (m == 0 || w.n == 0) return hipSuccess;
    if (w.k_chunks == 0 || w.n_tiles % 4 != 0) return hipErrorInvalidValue;
    OutSpec out = out_in;
    char *free_at = (char *)scratch;
    size_t left = scratch ? scratch_bytes : 0;
    if (a_f32) {
        const size_t rows_bytes = (((size_t)m * w.k * 2) + 255) & ~(size_t)255, factors = ((size_t)m * 4 + 255) & ~(size_t)255;
        if (left < factors + rows_bytes || rows_bytes > 0x7FFFFFFFu) return hipErrorInvalidValue;
        float *row_scale = (float *)free_at;
        _Float16 *rows16 = (_Float16 *)(free_at + factors);
        hipError_t e = launch_f32_rows_to_f16(s, (const float *)a, rows16, nullptr, row_scale, m, w.k);
        if (e != hipSuccess) return e;
        a = rows16;
        out.row_scale = row_scale;
        free_at += factors + rows_bytes;
        left -= factors + rows_bytes;
    }
    const size_t per_split = (size_t)m * w.n_tiles * 16 * 4;
    if (splits > left / per_split) splits = (uint32_t)(left / per_split);
    if (splits > w.k_chunks) splits = w.k_chunks;
    if (splits < 1) splits = 1;
    if (out.swiglu && splits == 1 && nt == 1) nt = 2;
    hipError_t e;
    const bool found = waves_form(waves_mt(m), nt, waves, e, [&](auto form) {
        return decltype(form)::launch(s, w, a, m, out, splits, (float *)free_at);
    });
    return found ? e : hipErrorInvalidValue;
}

}  // namespace twm
