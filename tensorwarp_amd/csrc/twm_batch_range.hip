// GEMM for 5 .. 32 f32 rows on deep, narrow matrices: K cut into ranges whose rows a workgroup stages at once, exact weights.
//
// Semantics: those of k_waves_exact (twm_waves_exact.hip; crates/kernels/src/quantize.rs:1219-1238): per 32-deep group the
// products a * (q - 8) are summed in f32 by MFMA, the group sum is scaled once by f32(scale) and added to the running f32 sum; f32
// rows enter as two f16 terms, with a power of two per row and 128-deep chunk that brings the row's largest magnitude there to
// [2^13, 2^14), exactly undone on the chunk's sums.  (One per row and k-slice, up to nine chunks, was no faster -- 18944 -> 3584 at 8
// rows 13.8, now 13.9 us, at 32 23.2 and 23.0 -- and a value far above its neighbours took the bits of 1151 of them instead of 127: with
// one of 1e6 in each of 8 rows the columns where its weight is 0 were 2.87e-7 off the 64-bit product, now 1.38e-7, k_waves_exact 1.53e-7.)
//
// What bounds these launches: each workgroup of k_waves_exact converts every row of its K-range itself, for one to four column
// tiles, and fetches 4 bytes per value for them (18944 -> 3584 at 32 rows: 56 column groups, 136 MB from L2 for 38 MB of weights,
// the conversion longer than the products).  So:
// * a workgroup takes eight or sixteen tiles and a range just short enough to stage all its rows in LDS (up to 147 KB), so that
//   rows are fetched and converted 14 to 28 times instead of 56 and the grid is still one round of the CUs;
// * the rows' loads are issued first, by all waves, then the weights of eight (tile, chunk) units per wave; those arrive during the
//   conversion.  (All of a wave's weights at once filled the CU's queue of loads in flight: 18944 -> 3584 at 8 rows 16.0, at 32 25.2.)
// * two k-slices of four waves beside each other; per group the wave reads the rows' operands once for its two or four tiles;
//   a unit's scaling and the next one's unpack stand between its matrix instructions (a v_mfma_f32_16x16x32 leaves the vector unit
//   two of its four issue slots: four in a row with the seventeen vector instructions behind them take 114 cycles, spread 104).
// The rounding error of the sums is that of the kernels before or less (a chunk's four groups are summed first, the ranges by
// pairs: 18944 -> 3584 at 32 rows 1.14e-7 of the result against 64 bits, k_waves_exact 1.14e-7; at 8 rows 1.06e-7 and 1.23e-7; with one
// chain each 1.33e-7 and 1.36e-7).
// What is left: the partial sums (17 x 32 x 3584 floats in the example), written and read back by k_splitk_reduce, 4.7 of 22.7 us.
#include "twm_waves_core.h"

#include <type_traits>

namespace twm {

namespace {

constexpr uint32_t kRangeWaves = 8;
constexpr uint32_t KS = 2;                 // k-slices of a range, four waves each
constexpr uint32_t COLS = kRangeWaves / KS;

constexpr uint32_t range_slice(int nt) { return nt == 4 ? 5u : 9u; }

// the largest of m over each sixteen lanes, in each of them
__device__ __forceinline__ float row16_max(float m)
{
    asm("s_nop 1\n"
        "v_max_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf\n"
        "s_nop 1\n"
        "v_max_f32_dpp %0, %0, %0 row_ror:4 row_mask:0xf bank_mask:0xf\n"
        "s_nop 1\n"
        "v_max_f32_dpp %0, %0, %0 row_ror:2 row_mask:0xf bank_mask:0xf\n"
        "s_nop 1\n"
        "v_max_f32_dpp %0, %0, %0 row_ror:1 row_mask:0xf bank_mask:0xf\n"
        : "+v"(m));
    return m;
}

}  // namespace

// grid: `per_xcd` workgroups for each of the eight XCDs, which take runs of (range, column group) in turn: the workgroups of a
// range share its activations in one or two L2 caches.
template <int MT, int MODE, int NT>
__global__ __launch_bounds__(64 * kRangeWaves) void k_batch_range(const uint4v *__restrict__ qw, const uint2v *__restrict__ sc,
                                                 const float *__restrict__ a, uint32_t m_rows, uint32_t k, uint32_t n_tiles,
                                                 uint32_t k_chunks, uint32_t chunks_per_split, uint32_t groups, uint32_t per_xcd,
                                                 uint32_t items, float *__restrict__ partials)
{
    constexpr int TERMS = MODE == kRowsF32 ? 2 : 1;
    constexpr int SLOTS = 8 / NT;
    constexpr uint32_t kSlice = range_slice(NT);                 // most chunks of a k-slice
    constexpr int kTile = 16 * MT * kWeRow;                      // halves of one term's rows of a chunk
    constexpr int kChunk = TERMS * kTile;
    constexpr uint32_t QUADS = MODE == kRowsF32Few ? 2 : 4 * MT; // row quads that are staged
    constexpr uint32_t UNITS = (KS * QUADS + kRangeWaves - 1) / kRangeWaves;
    constexpr uint32_t kTiles = COLS * NT, kSumRow = kTiles * 16u + 4u;   // floats of a row of sums (rows four apart lie 16 banks apart)
    extern __shared__ __attribute__((aligned(16))) _Float16 lds_all[];

    const uint32_t item = (blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3);
    if (item >= items) return;
    const uint32_t split = item / groups, group = item - split * groups;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t c = lane & 15u, kb = lane >> 4;

    const uint32_t kc0 = split * chunks_per_split;
    const uint32_t nchunks = k_chunks - kc0 < chunks_per_split ? k_chunks - kc0 : chunks_per_split;
    const uint32_t first = (nchunks + 1u) / 2u;                  // chunks of k-slice 0
    const uint32_t slice = wave / COLS, base = slice ? first : 0u, tile0 = group * kTiles + (wave % COLS) * NT;
    const uint32_t count = tile0 >= n_tiles ? 0u : slice ? nchunks - first : first;

    WeConsts dq = {0x000F000Fu, 0x00F000F0u, 0x64006400u, 0x54005400u};
    asm volatile("" : "+s"(dq.mask_lo), "+s"(dq.mask_hi), "+v"(dq.magic_lo), "+v"(dq.magic_hi));

    // ---- the range's activations: a wave takes row quad u % QUADS of k-slice u / QUADS, sixteen lanes to a row
    const uint32_t p = lane & 15u, odd = (lane >> 4) & 1u;
    uint4v ar[UNITS][kSlice][2];
    auto unit_of = [&](uint32_t i, uint32_t &quad, uint32_t &of, uint32_t &at, uint32_t &n) {
        const uint32_t u = wave + kRangeWaves * i;
        quad = u % QUADS;
        of = u / QUADS;
        at = of ? first : 0u;
        n = of == 0 ? first : of == 1 ? nchunks - first : 0u;
    };
#pragma unroll
    for (uint32_t i = 0; i < UNITS; i++) {
        uint32_t quad, of, at, n;
        unit_of(i, quad, of, at, n);
        uint32_t row = 4u * quad + (lane >> 4);
        row = row < m_rows ? row : m_rows - 1u;                  // rows past the last replay it and are never stored
#pragma unroll
        for (uint32_t j = 0; j < kSlice; j++) {
            if (j < n) {
                const uint32_t kg = kc0 + at + j;
                const TWM_GLOBAL char *src = we_scalar_base(a, (size_t)kg * 512u);
                const uint32_t most = (k - kg * 128u) * 4u - 16u;   // the row's last 16 bytes, for places past its end (staged as zeros)
#pragma unroll
                for (int l = 0; l < 2; l++) {                    // (odd lane groups the second half first: the LDS writes of two
                    uint32_t col = 16u * p + (((uint32_t)l ^ odd) << 8);   // rows take different banks)
                    col = col < most ? col : most;
                    ar[i][j][l] = *(const TWM_GLOBAL uint4v *)(src + (row * k * 4u + col));
                }
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();   // (no wave's weights ahead of another's activations)
    __builtin_amdgcn_sched_barrier(0);

    // ---- this wave's weights: 8 / NT chunks of its NT tiles in flight.  Past the end every lane reads the first bytes of the wave's
    // first chunk instead (one line per load, never used).
    uint4v wq[SLOTS][NT];
    uint2v ws[SLOTS][NT];
    const uint32_t q_off = lane * 16u, s_off = c * 8u;
    auto load_b = [&](int slot, int t, uint32_t i) {
        const uint32_t on = i < count ? 0xFFFFFFFFu : 0u, kg = kc0 + (i < count ? base + i : 0u);
        const size_t tile = (size_t)kg * n_tiles + (count ? tile0 + (uint32_t)t : 0u);
        wq[slot][t] = __builtin_nontemporal_load((const TWM_GLOBAL uint4v *)(we_scalar_base(qw, tile * 1024u) + (q_off & on)));
        ws[slot][t] = __builtin_nontemporal_load((const TWM_GLOBAL uint2v *)(we_scalar_base(sc, tile * 128u) + (s_off & on)));
    };
#pragma unroll
    for (int s = 0; s < SLOTS; s++)
#pragma unroll
        for (int t = 0; t < NT; t++) load_b(s, t, (uint32_t)s);
    __builtin_amdgcn_sched_barrier(0);

    float *factors = (float *)(lds_all + chunks_per_split * kChunk);   // [chunk][16 MT]
#pragma unroll
    for (uint32_t i = 0; i < UNITS; i++) {
        uint32_t quad, of, at, n;
        unit_of(i, quad, of, at, n);
        const uint32_t row = 4u * quad + (lane >> 4);
        if (n != 0 && (kc0 + at + n) * 128u > k) {               // the chunk that K ends in: zeros behind it
#pragma unroll
            for (uint32_t j = 0; j < kSlice; j++) {
                if (j < n) {
                    const uint32_t left = k - (kc0 + at + j) * 128u;
#pragma unroll
                    for (int l = 0; l < 2; l++)
                        ar[i][j][l] = ((uint32_t)l ^ odd) * 64u + 4u * p < left ? ar[i][j][l] : uint4v{0u, 0u, 0u, 0u};
                }
            }
        }
#pragma unroll
        for (uint32_t j = 0; j < kSlice; j++) {
            if (j < n) {
                const WeFactor factor = we_factor(row16_max(we_max8(ar[i][j][0], ar[i][j][1])));
                _Float16 *dst = lds_all + (at + j) * kChunk;
#pragma unroll
                for (int l = 0; l < 2; l++) {
                    uint2v hi, lo;
                    we_terms(ar[i][j][l], factor.down, hi, lo);
                    const uint32_t vec = (((uint32_t)l ^ odd) << 3) + (p >> 1);
                    *(uint2v *)(dst + row * kWeRow + ((vec ^ (row & 15u)) * 8u) + (p & 1u) * 4u) = hi;
                    if constexpr (MODE == kRowsF32Few)
                        *(uint2v *)(dst + (row + 8u) * kWeRow + ((vec ^ (row + 8u)) * 8u) + (p & 1u) * 4u) = lo;
                    else
                        *(uint2v *)(dst + kTile + row * kWeRow + ((vec ^ (row & 15u)) * 8u) + (p & 1u) * 4u) = lo;
                }
                if (p == 0) {
                    float *f = factors + (at + j) * 16u * MT;
                    f[row] = factor.back;
                    if (MODE == kRowsF32Few) f[row + 8u] = factor.back;
                }
            }
        }
    }
    __syncthreads();

    // ---- the products: group after group of a chunk on the NT tiles, one read of the activations for all of them
    float4v acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[mt][t] = float4v{0.f, 0.f, 0.f, 0.f};
    uint32_t rd_off[4];  // row c of a row block, vector 4 g + kb of the chunk -> slot (4 g + kb) ^ c
#pragma unroll
    for (int g = 0; g < 4; g++) rd_off[g] = c * kWeRow + (((4u * g + kb) ^ c) * 8u);
    half8 af[2][TERMS][MT];
    auto load_a = [&](int to, uint32_t i, int g) {
        const _Float16 *src = lds_all + (base + (i < count ? i : 0u)) * kChunk + rd_off[g];
#pragma unroll
        for (int t = 0; t < TERMS; t++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++) af[to][t][mt] = *(const half8 *)(src + t * kTile + mt * 16 * kWeRow);
    };
    // A unit is a group of a tile.  Its MFMAs are followed by the scaling of the unit before and the unpack of the next one,
    // so that no vector instruction waits for the matrix pipe.
    // (a chunk's four groups are summed first, its factors taken back on their sum: one long chain of additions would double the
    // rounding error)
    float4v d[2][MT], sum[MT][NT], back[MT];
    float scale = 0.f;
    half8 bf;
    auto scaled = [&](int u, int t) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                sum[mt][t][r] = u < NT ? d[u & 1][mt][r] * scale : __builtin_fmaf(d[u & 1][mt][r], scale, sum[mt][t][r]);
                if (u >= 3 * NT) acc[mt][t][r] = __builtin_fmaf(sum[mt][t][r], back[mt][r], acc[mt][t][r]);
            }
    };
    auto step = [&](int slot, uint32_t i) {
        bf = we_unpack(wq[slot][0][0], dq);
#pragma unroll
        for (int u = 0; u < 4 * NT; u++) {
            const int g = u / NT, t = u % NT;
            if (t == 0) load_a((g + 1) & 1, g == 3 ? i + 1u : i, (g + 1) & 3);
            if (u == 2 * NT) {
#pragma unroll
                for (int mt = 0; mt < MT; mt++) back[mt] = *(const float4v *)(factors + (base + i) * 16u * MT + 16 * mt + 4u * kb);
            }
#pragma unroll
            for (int mt = 0; mt < MT; mt++) d[u & 1][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[g & 1][0][mt], bf, float4v{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            if constexpr (TERMS == 2) {
#pragma unroll
                for (int mt = 0; mt < MT; mt++) d[u & 1][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[g & 1][1][mt], bf, d[u & 1][mt], 0, 0, 0);
            }
            if (u != 0) scaled(u - 1, (u - 1) % NT);
            if (u + 1 < 4 * NT) bf = we_unpack(wq[slot][(u + 1) % NT][(u + 1) / NT], dq);
            union { uint32_t u32; half2v h; } pair;
            pair.u32 = ws[slot][t][g >> 1];
            scale = (float)pair.h[g & 1];
            asm("" : "+v"(scale));
            // (a matrix instruction keeps its pipe for the time of four vector instructions)
#pragma unroll
            for (int mt = 0; mt < MT * TERMS; mt++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (g == 3) {
                load_b(slot, t, i + SLOTS);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        scaled(4 * NT - 1, NT - 1);
    };
    if (count) {
        load_a(0, 0, 0);
        for (uint32_t i = 0; i < count; i += SLOTS) {
#pragma unroll
            for (int s = 0; s < SLOTS; s++)
                if (i + s < count) step(s, i + s);
        }
    }
    __syncthreads();

    // ---- the two k-slices' sums: [slice][row][column]
    float *sums = (float *)lds_all;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                sums[(slice * 16u * MT + 16 * mt + 4u * kb + r) * kSumRow + ((wave % COLS) * NT + t) * 16u + c] = acc[mt][t][r];
    __syncthreads();
    constexpr uint32_t PER_ROW = kTiles * 4u, ROWS = 64u * kRangeWaves / PER_ROW;   // sixteen-byte places of a row; rows at a time
    const uint32_t n_ld = n_tiles * 16u, place = threadIdx.x % PER_ROW * 4u, col = group * (kTiles * 16u) + place;
    if (col >= n_ld) return;
    float *dst = partials + (size_t)split * m_rows * n_ld + col;
    for (uint32_t row = threadIdx.x / PER_ROW; row < m_rows; row += ROWS) {
        const float *at = sums + row * kSumRow + place;
        float4v s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (uint32_t i = 0; i < KS; i++) {
            s += *(const float4v *)(at + i * 16u * MT * kSumRow);
            if constexpr (MODE == kRowsF32Few) s += *(const float4v *)(at + (i * 16u * MT + 8u) * kSumRow);   // rows 8 .. 15 hold the second terms
        }
        *(float4v *)(dst + (size_t)row * n_ld) = s;
    }
}

namespace {

template <int MT, int MODE, int NT> struct BatchRange {
    static constexpr uint32_t tiles = COLS * NT;   // 16-column tiles of a workgroup
    static constexpr size_t chunk = (MODE == kRowsF32 ? 2 : 1) * 16 * MT * kWeRow * sizeof(_Float16) + 16 * MT * sizeof(float);   // staged values and factors
    static constexpr size_t sums = (size_t)KS * 16 * MT * (tiles * 16 + 4) * sizeof(float);
    static constexpr size_t most = 160 * 1024;
    static constexpr uint32_t max_chunks = most / chunk < KS * range_slice(NT) ? (uint32_t)(most / chunk) : KS * range_slice(NT);
    static size_t lds(uint32_t cps) { return cps * chunk > sums ? cps * chunk : sums; }
    static hipError_t init()
    {
        return hipFuncSetAttribute((const void *)k_batch_range<MT, MODE, NT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds(max_chunks));
    }
    static hipError_t launch(hipStream_t s, const WeightView &w, const float *a, uint32_t m, const OutSpec &out, uint32_t splits, float *partials)
    {
        const uint32_t cps = (w.k_chunks + splits - 1) / splits;
        if (cps > max_chunks) return hipErrorInvalidValue;
        splits = (w.k_chunks + cps - 1) / cps;   // no empty range
        const uint32_t groups = (w.n_tiles + tiles - 1) / tiles, items = groups * splits, per_xcd = (items + 7) / 8;
        hipLaunchKernelGGL((k_batch_range<MT, MODE, NT>), dim3(per_xcd * 8), dim3(64 * kRangeWaves), lds(cps), s, (const uint4v *)w.qw, (const uint2v *)w.sc, a, m,
                           w.k, w.n_tiles, w.k_chunks, cps, groups, per_xcd, items, partials);
        return launch_splitk_reduce(s, partials, out, m, w.n, w.n_tiles * 16, splits);
    }
};

// fn gets the form of a row count
template <typename F> auto range_form(uint32_t m, F &&fn)
{
    return m <= 8 ? fn(BatchRange<1, kRowsF32Few, 2>{}) : m <= 16 ? fn(BatchRange<1, kRowsF32, 2>{}) : fn(BatchRange<2, kRowsF32, 4>{});
}

}  // namespace

// Once per device, outside any stream capture: more than 64 KB of LDS.
hipError_t init_batch_range()
{
    for (uint32_t m : {8u, 16u, 32u})
        if (hipError_t e = range_form(m, [](auto form) { return decltype(form)::init(); })) return e;
    return hipSuccess;
}

// How many K-ranges a GEMM is cut into (0: another form runs): one round of workgroups, each with as many chunks as its staging
// takes, or fewer where the round fills the CUs with them.  Lines from random calls, 5 .. 32 f32 rows on 60 .. 600 column tiles,
// K of 3000 .. 24000 (us, k_waves_exact or above 160 chunks k_batch / this kernel):
// * 17 .. 32 rows: from a work of 21500 tiles times chunks on, gated 26500 (18944 -> 3584 at 32 rows 26.6 / 22.7, 8192 -> 8192 at
//   17 21.6 / 19.1, 12672 -> 5824 at 17 25.6 / 20.5; below, 7296 -> 4608 at 28 rows gains 1 %, 4608 -> 5120 at 32 is 13.6 / 15.8),
//   and above 160 chunks, where k_waves_exact ends, from 72 tiles on (22656 -> 1344 at 32 rows 23.3 / 17.2);
// * up to sixteen rows: 108 .. 360 tiles and a work of 19000 (18944 -> 3584 at 8 rows 15.9 / 13.9, 11008 -> 4096 at 13 15.0 / 12.9,
//   14336 -> 4096 at 16 16.3 / 15.1; 84 tiles at a work of 13000 - 15000 8 % behind, 440 .. 520 tiles, where k_waves_exact does not
//   cut K, 0 - 25 %; 13824 -> 5120 at 16 rows, 320 tiles, level), and not gated: the kernel that adds the ranges reads twice the
//   sums per value (0.92 .. 1.13 of the time).
// Against the kernels of before over these lines, in the mean: 17 .. 32 rows 0.88, up to sixteen 0.95.
uint32_t plan_batch_range(uint32_t n_tiles, uint32_t k_chunks, uint32_t m, bool a_f32, bool gated, size_t scratch_bytes)
{
    if (!a_f32 || m < 5 || m > 32) return 0;
    const uint32_t tiles = range_form(m, [](auto form) { return decltype(form)::tiles; });
    const uint32_t most = range_form(m, [](auto form) { return decltype(form)::max_chunks; });
    const uint32_t groups = (n_tiles + tiles - 1) / tiles;
    if (groups == 0 || groups > 128) return 0;
    const uint32_t cps = (k_chunks * groups + 255) / 256;
    if (cps < 2 || cps > most) return 0;
    const uint32_t splits = (k_chunks + cps - 1) / cps, work = n_tiles * k_chunks;
    if (splits < 2 || groups * splits > 256 || work * 10 < 256 * tiles * cps * 7) return 0;   // (CUs at least 70 % busy)
    if ((size_t)splits * m * n_tiles * 64 > scratch_bytes) return 0;
    if (m > 16 ? (k_chunks > 160 ? n_tiles < 72 : work < (gated ? 26500u : 21500u)) : (gated || n_tiles < 108 || n_tiles > 360 || work < 19000)) return 0;
    return splits;
}

uint32_t batch_range_columns(uint32_t m)
{
    return 16 * range_form(m, [](auto form) { return decltype(form)::tiles; });
}

// 1 .. 32 rows; splits >= 1 K-ranges of at most BatchRange::max_chunks chunks, their sums in `scratch`.
hipError_t launch_batch_range(hipStream_t s, const WeightView &w, const float *a, uint32_t m, const OutSpec &out, uint32_t splits,
                              void *scratch, size_t scratch_bytes)
{
    if (m == 0 || w.n == 0) return hipSuccess;
    if (w.k_chunks == 0 || w.n_tiles % 4 != 0 || m > 32 || splits == 0 || splits > w.k_chunks) return hipErrorInvalidValue;
    if ((uint64_t)m * w.k * 2 > 0x7FFFFFFFu) return hipErrorInvalidValue;   // (32-bit offsets into the rows)
    if (!scratch || (size_t)splits * m * w.n_tiles * 64 > scratch_bytes) return hipErrorInvalidValue;
    return range_form(m, [&](auto form) { return decltype(form)::launch(s, w, a, m, out, splits, (float *)scratch); });
}

}  // namespace twm
