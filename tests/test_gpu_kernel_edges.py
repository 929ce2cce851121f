"""GPU tests of single kernels at the sizes where their tilings change: against the CPU oracle's f64 dequant-then-matmul or
its byte-exact format functions, through the C ABI."""
import ctypes as C
import re
import shutil
from types import SimpleNamespace

import numpy as np
import pytest

import tensorwarp_amd as T
from oracle import twm_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = T.WarpDevice(0)
    yield d
    d.close()


def weight(dev, k, n, seed):
    packed, scales = O.synth_packed(k, n, seed), O.synth_scales(k, n, seed + 1)
    return packed, scales, T.MarlinWeight.upload(dev, packed, scales, k, n)


def close_rows(got, truth, bar):
    """Every row of `got` within `bar` of the truth, relative to max(|t|, 1e-3 of the row's largest)."""
    assert np.isfinite(got).all()
    for r in range(len(truth)):
        floor = 1e-3 * np.abs(truth[r]).max() + 1e-300
        err = (np.abs(got[r].astype(np.float64) - truth[r]) / np.maximum(np.abs(truth[r]), floor)).max()
        assert err < bar, (r, err)


# f32 sums of K products: K * 2^-24 relative to the sum of magnitudes at worst, 2e-4 of the floor above in practice
F32_SUM = 2e-4


@pytest.mark.parametrize("k", [32, 4096, 4128, 12288, 12320, 20512, 32800])
def test_f32_row_conversion_at_the_edges_of_its_register_tiers(dev, k):
    # rows of 4096, 12288, 20480 and 32768 values are the most that one, three, five and eight pieces per thread hold
    m, n = 6, 24
    packed, scales, w = weight(dev, k, n, 77 + k)
    rows = O.synth_normal_f32(m * k, 7 + k).reshape(m, k).copy()
    rows[1] *= np.float32(1e7)
    rows[2, k - 1] = np.float32(3e6)      # the row's largest value is its last
    rows[3] *= np.float32(1e-8)
    c = T.GpuTensor.from_host(dev, np.full((m, n), np.nan, np.float32))
    T.gemm(dev, w, T.GpuTensor.from_host(dev, rows), m, c)
    close_rows(c.to_host(), O.gemm_f64(rows, packed, scales, m, k, n), F32_SUM)
    w.free()


@pytest.mark.parametrize("m,k", [(85, 12288), (86, 12288), (51, 20480), (52, 20480), (31, 32768), (32, 32768), (33, 32768), (1, 32768)])
def test_f32_rows_converted_by_one_or_several_workgroups(dev, m, k):
    # the stretches of a row run as workgroups of their own up to 85, 51 and 32 rows of these lengths: rows of f16 values
    # times powers of two, the row's largest value in its first and in its last stretch
    n = 24
    packed, scales, w = weight(dev, k, n, 300 + m)
    base = O.synth_act_f16(m, k, 301).view(np.float16).astype(np.float32).reshape(m, k).copy()
    base[0, k - 1], base[m - 1, 0] = 64.0, 64.0
    factor = np.ones(m, np.float32)
    factor[::3] = 2.0 ** 40
    rows = base * factor[:, None]
    if m <= 32:
        truth = O.gemm_f64(rows, packed, scales, m, k, n)
    else:
        truth = (base.astype(np.float64) @ O.dequant_f16(packed, scales, k, n).view(np.float16).astype(np.float64).reshape(k, n)) * factor[:, None]
    c = T.GpuTensor.from_host(dev, np.full((m, n), np.nan, np.float32))
    a = T.GpuTensor.from_host(dev, rows)
    T.gemm(dev, w, a, m, c)
    close_rows(c.to_host(), truth, F32_SUM if m <= 32 else 1e-3)   # above 32 rows the prefill GEMM's bar
    for t in (a, c):
        t.free()
    w.free()


@pytest.mark.parametrize("m,k", [(33, 64), (65, 64), (160, 4128), (3600, 18944)])
def test_scaled_f32_rows_of_a_prompt_in_one_and_two_slabs(dev, m, k):
    # prompt rows outside the f16 range: the factors go back onto the sums 32 rows at a time (first, last and 32nd row of
    # such a group among them); 3600 x 18944 rows do not fit the half of the scratch that holds their f16 terms
    n, distinct = 72, 48
    packed, scales, w = weight(dev, k, n, 500 + k)
    base = O.synth_act_f16(distinct, k, 501).view(np.float16).astype(np.float32).reshape(distinct, k)
    factor = np.ones(m, np.float32)
    factor[[0, 31, 32, m // 2, m - 1]] = [2.0 ** 20, 2.0 ** -20, 2.0 ** 90, 2.0 ** 17, 2.0 ** -90]
    rows = base[np.arange(m) % distinct] * factor[:, None]   # f16 values times powers of two: the f16 terms are exact
    w16 = O.dequant_f16(packed, scales, k, n).view(np.float16).astype(np.float64).reshape(k, n)
    truth = (base.astype(np.float64) @ w16)[np.arange(m) % distinct] * factor[:, None].astype(np.float64)
    c = T.GpuTensor.from_host(dev, np.full((m, n), np.nan, np.float32))
    a = T.GpuTensor.from_host(dev, np.ascontiguousarray(rows))
    T.gemm(dev, w, a, m, c)
    close_rows(c.to_host(), truth, 1e-3)      # the prefill GEMM's bar: f32 sums over all of K inside the MFMAs
    for t in (a, c):
        t.free()
    w.free()


@pytest.mark.parametrize("m", [130, 160, 255, 400])
@pytest.mark.parametrize("gated", [False, True])
def test_f32_prompt_rows_that_fit_run_as_the_f16_rows_do(dev, m, gated):
    # f16 values as f32 rows, all of them in the scratch at once: one launch under the f16 rows' plan, so the same sums in the
    # same order (a gated launch goes through the K-split's buffer: the same products of the same sums)
    k, n = 2720, 1088
    packed, scales = O.synth_packed(k, n, 611), O.synth_scales(k, n, 612)
    if gated:
        half = n // 2
        p, s = packed.reshape(k // 32, n, 16), scales.reshape(k // 32, n)
        pair = [(T.GpuTensor.from_host(dev, np.ascontiguousarray(p[:, c])), T.GpuTensor.from_host(dev, np.ascontiguousarray(s[:, c]), "f16"))
                for c in (slice(0, half), slice(half, n))]
        w = T.MarlinWeight.gate_up(dev, *pair, k, half)
    else:
        half, w = n, T.MarlinWeight.upload(dev, packed, scales, k, n)
    a16 = O.synth_act_f16(m, k, 613)
    got = []
    dev.set_option("prefill_bm", 64)     # (the prefill GEMM at every one of these row counts)
    try:
        for rows in (T.GpuTensor.from_host(dev, a16, "f16"), T.GpuTensor.from_host(dev, a16.view(np.float16).astype(np.float32))):
            out = T.GpuTensor.from_host(dev, np.full((m, half), np.nan, np.float32))
            (T.gemm_swiglu if gated else T.gemm)(dev, w, rows, m, out)
            got.append(out.to_host())
    finally:
        dev.set_option("prefill_bm", 0)
    assert np.isfinite(got[0]).all() and np.array_equal(got[0], got[1])
    w.free()


@pytest.mark.parametrize("m", [130, 160, 200])
def test_f16_result_rows_are_the_f32_ones_rounded(dev, m):
    # rows that fit the staging part are one launch: the last ones, few enough for the exact decode arithmetic by themselves,
    # run as the others do
    k, n = 1088, 1024
    packed, scales, w = weight(dev, k, n, 621)
    a = T.GpuTensor.from_host(dev, O.synth_act_f16(m, k, 623), "f16")
    c, c16 = T.GpuTensor.from_host(dev, np.full((m, n), np.nan, np.float32)), T.GpuTensor(dev, (m, n), "f16")
    T.gemm(dev, w, a, m, c)
    T.gemm_f16out(dev, w, a, m, c16)
    assert np.array_equal(c16.to_host().view(np.float16), c.to_host().astype(np.float16))
    w.free()


@pytest.mark.parametrize("m", [9, 16, 17, 32])
@pytest.mark.parametrize("ffn,nt,waves", [(32, 0, 0), (96, 3, 0), (160, 3, 0), (96, 4, 8), (64, 1, 16)])
def test_batched_gate_through_lds(dev, m, ffn, nt, waves):
    # one tile per wave: the up tiles' sums reach the gate tiles' waves through LDS; one to five quads on workgroups of one,
    # two and three (the last one part empty), alone and with k-slices
    k = 544                                          # 17 groups: four chunks and a quarter
    gate, up = [(O.synth_packed(k, ffn, s), O.synth_scales(k, ffn, s + 1)) for s in (811, 813)]
    pair = [tuple(T.GpuTensor.from_host(dev, x, t) for x, t in zip(w, ("u8", "f16"))) for w in (gate, up)]
    w = T.MarlinWeight.gate_up(dev, *pair, k, ffn)
    a16 = O.synth_act_f16(m, k, 815)
    a = a16.view(np.float16).astype(np.float32).reshape(m, k)
    g, u = (O.gemm_f64(a, *x, m, k, ffn) for x in (gate, up))
    out = T.GpuTensor.from_host(dev, np.full((m, ffn), np.nan, np.float32))
    try:
        for key, v in (("kernel", 4 if nt else 0), ("nt", nt), ("waves", waves)):
            dev.set_option(key, v)
        T.gemm_swiglu(dev, w, T.GpuTensor.from_host(dev, a16, "f16"), m, out)
    finally:
        for key in ("kernel", "nt", "waves"):
            dev.set_option(key, 0)
    close_rows(out.to_host(), g / (1.0 + np.exp(-g)) * u, F32_SUM)
    w.free()


@pytest.mark.parametrize("splits", [2, 3, 4, 5, 6, 8, 9])
@pytest.mark.parametrize("m,n", [(5, 68), (40, 68), (24, 65), (40, 130)])
def test_split_sums_of_every_count(dev, m, n, splits):
    # the sum kernel takes four, two and one partial sums at a time; 16-byte stores where N is a multiple of four
    k = 9 * 128
    packed, scales, w = weight(dev, k, n, 900 + n)
    a16 = O.synth_act_f16(m, k, 903 + m)
    c = T.GpuTensor.from_host(dev, np.full((m, n), np.nan, np.float32))
    dev.set_option("kernel", 4 if m <= 32 else 0)
    try:
        T.gemm(dev, w, T.GpuTensor.from_host(dev, a16, "f16"), m, c, splits)
    finally:
        dev.set_option("kernel", 0)
    a = a16.view(np.float16).astype(np.float64).reshape(m, k)
    w16 = O.dequant_f16(packed, scales, k, n).view(np.float16).astype(np.float64).reshape(k, n)
    truth = O.gemm_f64(a.astype(np.float32), packed, scales, m, k, n) if m <= 32 else a @ w16
    close_rows(c.to_host(), truth, F32_SUM if m <= 32 else 1e-3)
    w.free()


@pytest.mark.parametrize("m,splits", [(24, 10), (24, 18), (40, 17), (65576, 2)])
def test_split_sums_past_eight_in_flight_and_of_many_rows(dev, m, splits):
    # the sum kernel has eight loads in flight behind the first, then what is left; one-wave and four-wave workgroups, rows of 32 quads
    k, n = splits * 128, 72
    packed, scales, w = weight(dev, k, n, 930 + splits)
    a16 = O.synth_act_f16(m, k, 931 + splits)
    c = T.GpuTensor.from_host(dev, np.full((m, n), np.nan, np.float32))
    dev.set_option("kernel", 4 if m <= 32 else 0)
    try:
        T.gemm(dev, w, T.GpuTensor.from_host(dev, a16, "f16"), m, c, splits)
    finally:
        dev.set_option("kernel", 0)
    truth = gemm_truth(a16.view(np.float16).astype(np.float32).reshape(m, k), packed, scales, m, k, n)
    err = np.abs(c.to_host() - truth) / np.maximum(np.abs(truth), 1e-3 * np.abs(truth).max(1, keepdims=True))
    assert err.max() < (F32_SUM if m <= 32 else 1e-3)     # (NaN where a row was not stored)
    w.free()


def gemm_truth(a, packed, scales, m, k, n):
    """Exact weights up to 32 rows, the FP16 Q4 unpack above (the library's default arithmetic), f64 sums."""
    if m <= 32:
        return O.gemm_f64(a, packed, scales, m, k, n)
    w16 = O.dequant_f16(packed, scales, k, n).view(np.float16).astype(np.float64).reshape(k, n)
    return a.astype(np.float64) @ w16


@pytest.mark.parametrize("nt,waves,splits", [(1, 8, 1), (2, 8, 1), (4, 8, 1), (2, 4, 1), (1, 8, 4)])
@pytest.mark.parametrize("m", [5, 8, 9, 16, 17, 32, 33, 48, 49, 64, 65, 96, 97, 129, 192])
def test_waves_on_their_own_k_ranges(dev, m, nt, waves, splits):
    # row blocks of 16, 32, 48 and 64 rows and their remainders; K of one group, fewer chunks than waves, and more than one
    # chunk per wave with a ragged end; N ragged; f16 rows, and f32 rows some of which leave the f16 range
    for k, n in ((32, 9), (416, 65), (1312, 131)):
        packed, scales, w = weight(dev, k, n, 1200 + k + m)
        a16 = O.synth_act_f16(m, k, 1203 + m)
        a = a16.view(np.float16).astype(np.float32).reshape(m, k).copy()
        big = a.copy()
        big[0] *= np.float32(2.0 ** 18)
        big[m - 1] *= np.float32(2.0 ** -22)
        bias = T.GpuTensor.from_host(dev, O.synth_normal_f32(n, 1207))
        for rows, dt in ((a16, "f16"), (big, "f32")):
            c = T.GpuTensor.from_host(dev, np.full((m, n), np.nan, np.float32))
            ad = T.GpuTensor.from_host(dev, rows, dt)
            try:
                for key, v in (("kernel", 5), ("nt", nt), ("waves", waves)):
                    dev.set_option(key, v)
                T.gemm_split(dev, w, ad, m, [c], [n], splits, biases=[bias] if dt == "f16" else None)
            finally:
                for key in ("kernel", "nt", "waves"):
                    dev.set_option(key, 0)
            truth = gemm_truth(a if dt == "f16" else big, packed, scales, m, k, n)
            if dt == "f16":
                truth = truth + bias.to_host().astype(np.float64)
            close_rows(c.to_host(), truth, F32_SUM if m <= 32 else 1e-3)
        w.free()


# Matrices on which the planner takes column groups of several tiles, or a kernel that is ahead there (each form of k_waves_exact
# by itself: the test behind these): a ragged last group, K one group past whole chunks and fewer chunks than two per
# wave; one and two row blocks, f16 rows, f32 rows in one block and in two tiles with rows outside the f16 range
@pytest.mark.parametrize("n", [12001, 17001, 22016, 30016, 40001])
@pytest.mark.parametrize("m,dtype", [(9, "f16"), (16, "f32"), (20, "f16"), (7, "f32"), (32, "f32")])
def test_waves_on_many_column_tiles(dev, m, dtype, n):
    k = 1312 if n < 40000 else 1056
    packed, scales, w = weight(dev, k, n, 1401 + m)
    a16 = O.synth_act_f16(m, k, 1403 + m)
    a = a16.view(np.float16).astype(np.float32).reshape(m, k).copy()
    if dtype == "f32":
        a[0] *= np.float32(2.0 ** 60)
        a[1, 128:256] *= np.float32(2.0 ** -30)      # a stretch of a row far below the rest of it
        a[m - 1] *= np.float32(2.0 ** -40)
    third = n // 3
    parts = [third, third + 1, n - 2 * third - 1]
    outs = [T.GpuTensor.from_host(dev, np.full((m, x), np.nan, np.float32)) for x in parts]
    bias = [T.GpuTensor.from_host(dev, np.zeros(x, np.float32)) for x in parts]
    T.gemm_split(dev, w, T.GpuTensor.from_host(dev, a16, "f16") if dtype == "f16" else T.GpuTensor.from_host(dev, a), m, outs, parts, biases=bias)
    close_rows(np.concatenate([o.to_host() for o in outs], axis=1), O.gemm_f64(a, packed, scales, m, k, n), F32_SUM)
    w.free()


# the gated store of whichever form the planner takes there, the last group ragged
@pytest.mark.parametrize("ffn", [6176, 10016, 14112, 18464])
@pytest.mark.parametrize("m,dtype", [(9, "f16"), (13, "f32"), (8, "f32"), (32, "f16")])
def test_waves_gated_store_on_many_column_tiles(dev, m, dtype, ffn):
    k = 1056
    gate, up = [(O.synth_packed(k, ffn, s), O.synth_scales(k, ffn, s + 1)) for s in (1511, 1513)]
    pair = [tuple(T.GpuTensor.from_host(dev, x, t) for x, t in zip(w, ("u8", "f16"))) for w in (gate, up)]
    w = T.MarlinWeight.gate_up(dev, *pair, k, ffn)
    a16 = O.synth_act_f16(m, k, 1515)
    a = a16.view(np.float16).astype(np.float32).reshape(m, k).copy()
    if dtype == "f32":
        a[1] *= np.float32(2.0 ** -21)
    g, u = (O.gemm_f64(a, *x, m, k, ffn) for x in (gate, up))
    out = T.GpuTensor.from_host(dev, np.full((m, ffn), np.nan, np.float32))
    T.gemm_swiglu(dev, w, T.GpuTensor.from_host(dev, a16, "f16") if dtype == "f16" else T.GpuTensor.from_host(dev, a), m, out)
    close_rows(out.to_host(), g / (1.0 + np.exp(-g)) * u, F32_SUM)
    w.free()


# Every form of k_waves_exact: one and two row blocks, f16 rows, up to eight f32 rows in one block and more in two tiles; two column
# groups of which the last has one whole tile and a ragged one, K one group past whole chunks on a wave or two more than once
@pytest.mark.parametrize("m,dtype,most", [(9, "f16", 10), (17, "f16", 10), (32, "f16", 10), (6, "f32", 10), (13, "f32", 8), (29, "f32", 4)])
@pytest.mark.parametrize("nt", [1, 2, 3, 4, 5, 6, 8, 10])
@pytest.mark.parametrize("splits", [1, 3])
def test_every_form_of_waves_on_exact_weights(dev, m, dtype, most, nt, splits):
    k, ffn = 1312, 96
    n = 16 * nt + 21
    packed, scales, w = weight(dev, k, n, 1601 + nt)
    gate, up = [(O.synth_packed(k, ffn, s), O.synth_scales(k, ffn, s + 1)) for s in (1611, 1613)]
    pair = [tuple(T.GpuTensor.from_host(dev, x, t) for x, t in zip(p, ("u8", "f16"))) for p in (gate, up)]
    wgu = T.MarlinWeight.gate_up(dev, *pair, k, ffn)
    a16 = O.synth_act_f16(m, k, 1615 + m)
    a = a16.view(np.float16).astype(np.float32).reshape(m, k).copy()
    if dtype == "f32":
        a[1] *= np.float32(2.0 ** -21)
        a[2, 128:256] *= np.float32(2.0 ** -30)
    rows = T.GpuTensor.from_host(dev, a16, "f16") if dtype == "f16" else T.GpuTensor.from_host(dev, a)
    c, out = (T.GpuTensor.from_host(dev, np.full((m, x), np.nan, np.float32)) for x in (n, ffn))
    runs = min(nt, most)
    dev.set_option("kernel", 5)
    try:
        dev.set_option("nt", nt)
        plans = [dev.plan(k, x, m, dtype=dtype, gated=g) for x, g in ((n, False), (2 * ffn, True))]
        T.gemm(dev, w, rows, m, c, splits)
        T.gemm_swiglu(dev, wgu, rows, m, out, splits)
    finally:
        dev.set_option("nt", 0)
        dev.set_option("kernel", 0)
    assert re.match(r"k_waves_exact: \d+-row x %d-column" % (16 * runs), plans[0]), plans
    assert re.match(r"k_waves_exact: \d+-row x %d-column" % (16 * (runs + runs % 2)), plans[1]), plans
    close_rows(c.to_host(), O.gemm_f64(a, packed, scales, m, k, n), F32_SUM)
    g, u = (O.gemm_f64(a, *x, m, k, ffn) for x in (gate, up))
    close_rows(out.to_host(), g / (1.0 + np.exp(-g)) * u, F32_SUM)
    w.free()
    wgu.free()


# few features of a deep matrix: K in ranges whose sums the reduction gates
@pytest.mark.parametrize("k,ffn,m,dtype", [(9344, 32, 9, "f16"), (9344, 96, 24, "f16"), (9376, 96, 25, "f32"), (12320, 160, 13, "f32"), (12288, 64, 8, "f32")])
def test_waves_gated_store_with_a_planned_k_split(dev, k, ffn, m, dtype):
    assert "k_splitk_reduce" in dev.plan(k, 2 * ffn, m, dtype=dtype, gated=True)
    gate, up = [(O.synth_packed(k, ffn, s), O.synth_scales(k, ffn, s + 1)) for s in (1521, 1523)]
    pair = [tuple(T.GpuTensor.from_host(dev, x, t) for x, t in zip(w, ("u8", "f16"))) for w in (gate, up)]
    w = T.MarlinWeight.gate_up(dev, *pair, k, ffn)
    a16 = O.synth_act_f16(m, k, 1525)
    a = a16.view(np.float16).astype(np.float32).reshape(m, k).copy()
    if dtype == "f32":
        a[1] *= np.float32(2.0 ** -21)
    g, u = (O.gemm_f64(a, *x, m, k, ffn) for x in (gate, up))
    out = T.GpuTensor.from_host(dev, np.full((m, ffn), np.nan, np.float32))
    T.gemm_swiglu(dev, w, T.GpuTensor.from_host(dev, a16, "f16") if dtype == "f16" else T.GpuTensor.from_host(dev, a), m, out)
    close_rows(out.to_host(), g / (1.0 + np.exp(-g)) * u, F32_SUM)
    w.free()


@pytest.mark.parametrize("m,dtype", [(5, "f32"), (8, "f32"), (9, "f16"), (13, "f32"), (32, "f16"), (40, "f16"), (64, "f32"), (96, "f16")])
def test_waves_gated_store(dev, m, dtype):
    k, ffn = 1056, 96                                # 33 groups; three quads of gate and up tiles
    gate, up = [(O.synth_packed(k, ffn, s), O.synth_scales(k, ffn, s + 1)) for s in (1311, 1313)]
    pair = [tuple(T.GpuTensor.from_host(dev, x, t) for x, t in zip(w, ("u8", "f16"))) for w in (gate, up)]
    w = T.MarlinWeight.gate_up(dev, *pair, k, ffn)
    a16 = O.synth_act_f16(m, k, 1315)
    a = a16.view(np.float16).astype(np.float32).reshape(m, k).copy()
    if dtype == "f32":
        a[1] *= np.float32(2.0 ** -21)
    g, u = (gemm_truth(a, *x, m, k, ffn) for x in (gate, up))
    truth = g / (1.0 + np.exp(-g)) * u
    ad = T.GpuTensor.from_host(dev, a16, "f16") if dtype == "f16" else T.GpuTensor.from_host(dev, a)
    for nt, splits in ((0, 0), (2, 1), (4, 1), (1, 3)):
        out = T.GpuTensor.from_host(dev, np.full((m, ffn), np.nan, np.float32))
        try:
            dev.set_option("kernel", 5 if nt else 0)
            dev.set_option("nt", nt)
            T.gemm_swiglu(dev, w, ad, m, out, splits)
        finally:
            dev.set_option("kernel", 0)
            dev.set_option("nt", 0)
        close_rows(out.to_host(), truth, F32_SUM if m <= 32 else 2e-3)   # (a product of two sums at 1e-3 each)
    w.free()


# one group and one column; column and group tiles of the [N,K] form (64 x 4) with a remainder; more groups than a grid's
# y dimension counts (65535), in both forms
@pytest.mark.parametrize("k,n", [(32, 1), (96, 63), (128, 64), (160, 65), (288, 258), (2097184, 2), (8388704, 1)])
def test_one_pass_quantizer_both_layouts(dev, k, n):
    rng = np.random.default_rng(k + n)
    w = rng.standard_normal((n, k), dtype=np.float32)
    w[0, :9] = [0.5, -0.5, 1.5, -2.5, 7.0, -7.0, 0.49999997, 3.4999998, -6.5]  # ties and their neighbours: factor 1
    w[0, 9:32] = 0.25
    if k > 32:
        w[0, 32:64] = 0.0
        w[-1, 64:96] *= np.float32(1e-39)   # the factor overflows
        w[-1, 40], w[-1, 41] = np.nan, np.inf
    want_p, want_s = O.quantize_tw_marlin_nk(w, k, n)
    for nk in (True, False):
        x = w if nk else np.ascontiguousarray(w.T)
        p, s = T.quantize_f32_to_tw_marlin(dev, T.GpuTensor.from_host(dev, x), k, n, weights_are_nk=nk)
        assert np.array_equal(p.to_host(), want_p) and np.array_equal(s.to_host().view(np.uint16), want_s.view(np.uint16)), nk


@pytest.mark.parametrize("k,n", [(32, 1), (64, 3), (64, 512), (96, 514), (32, 257), (2097184, 2)])
@pytest.mark.parametrize("offset", [0, 4])
def test_unpack_columns_and_alignments(dev, k, n, offset):
    # pairs of columns, single ones, records that start off a 16-byte line, and more groups than a grid's y counts
    packed, scales = O.synth_packed(k, n, 5), O.synth_scales(k, n, 6)
    raw = T.GpuTensor.from_host(dev, np.concatenate([np.zeros(offset, np.uint8), packed.reshape(-1)]))
    sc = T.GpuTensor.from_host(dev, scales)
    for f16, want in ((True, O.dequant_f16(packed, scales, k, n)), (False, O.dequant_f32(packed, scales, k, n).view(np.uint32))):
        out = T.GpuTensor(dev, (k, n), "f16" if f16 else "f32")
        call = dev._l.twm_dequant_to_f16 if f16 else dev._l.twm_dequant_to_f32
        assert call(dev.handle, raw.ptr + offset, sc.ptr, k, n, out.ptr) == 0
        assert np.array_equal(out.to_host().view(want.dtype), want), f16


# [N,K] tiles of 2 .. 64 columns, of which 67 groups leave a remainder; rows of a workgroup's 256 places that end anywhere
@pytest.mark.parametrize("n", [2, 5, 16, 31, 64, 100, 130, 250, 260, 512])
def test_format_kernels_on_narrow_matrices(dev, n):
    k = 67 * 32
    w = np.random.default_rng(n).standard_normal((n, k), dtype=np.float32)
    kn = np.ascontiguousarray(w.T)
    want_p, want_s = O.quantize_tw_marlin_nk(w, k, n)
    for x, nk in ((w, True), (kn, False)):
        p, s = T.quantize_f32_to_tw_marlin(dev, T.GpuTensor.from_host(dev, x), k, n, weights_are_nk=nk)
        assert np.array_equal(p.to_host(), want_p) and np.array_equal(s.to_host().view(np.uint16), want_s.view(np.uint16)), nk
    q4 = T.quantize_weights_q4_0(dev, T.GpuTensor.from_host(dev, kn), k, n)
    assert np.array_equal(q4.to_host().reshape(-1), O.quantize_weights_q4_0_kn(kn, k, n).reshape(-1))
    fp, fs = T.fuse_tw_marlin_n(dev, [(p, s), (p, s)], k, [n, n])
    wp, ws = O.fuse_tw_marlin_n([(want_p, want_s)] * 2, k, [n, n])
    assert np.array_equal(fp.to_host(), wp) and np.array_equal(fs.to_host(), ws)
    assert np.array_equal(T.dequant_to_f16(dev, p, s, k, n).to_host().view(np.uint16), O.dequant_f16(want_p, want_s, k, n))
    assert np.array_equal(T.dequant_to_f32(dev, p, s, k, n).to_host().view(np.uint32), O.dequant_f32(want_p, want_s, k, n).view(np.uint32))


# from 32768 records and 17 columns on a thread unpacks whole records, two of them where columns and output allow it; more
# groups than a grid's y dimension counts
@pytest.mark.parametrize("k,n", [(4096, 256), (4096, 257), (4096, 514), (61728, 17), (63552, 18), (4096, 255), (65568, 16), (2097184, 18)])
@pytest.mark.parametrize("out_offset", [0, 1])
def test_unpack_of_whole_records(dev, k, n, out_offset):
    packed, scales = O.synth_packed(k, n, 5), O.synth_scales(k, n, 6)
    raw, sc = T.GpuTensor.from_host(dev, packed), T.GpuTensor.from_host(dev, scales)
    for f16, want in ((True, O.dequant_f16(packed, scales, k, n)), (False, O.dequant_f32(packed, scales, k, n).view(np.uint32))):
        out = T.GpuTensor.from_host(dev, np.full(k * n + 2, 7, want.dtype if f16 else np.int32))
        call = dev._l.twm_dequant_to_f16 if f16 else dev._l.twm_dequant_to_f32
        assert call(dev.handle, raw.ptr, sc.ptr, k, n, out.ptr + out_offset * (2 if f16 else 4)) == 0
        got = out.to_host().view(want.dtype)
        assert np.array_equal(got[out_offset:out_offset + k * n], want.reshape(-1)), f16
        assert (got[:out_offset] == 7).all() and (got[out_offset + k * n:] == 7).all()


@pytest.mark.parametrize("k,ns", [(32, [1]), (64, [255, 1, 257]), (2097184, [2, 1])])
def test_fuse_of_ragged_parts(dev, k, ns):
    parts = [(O.synth_packed(k, n, 7 + i), O.synth_scales(k, n, 8 + i)) for i, n in enumerate(ns)]
    fp, fs = T.fuse_tw_marlin_n(dev, [tuple(T.GpuTensor.from_host(dev, x) for x in p) for p in parts], k, ns)
    wp, ws = O.fuse_tw_marlin_n(parts, k, ns)
    assert np.array_equal(fp.to_host(), wp) and np.array_equal(fs.to_host(), ws)


def test_saved_plans_of_every_kernel_come_back(dev):
    # a plan that the tuner keeps (valid, kernel, nt, waves, sub, sub_waves, splits, prefill_bm) is in an exported blob's last
    # 96 bytes, eight per bucket of row counts; import drops only values that no option takes
    k, n = 256, 128
    packed, scales, w = weight(dev, k, n, 1701)
    blob = w.export_blob()
    kept = [1, 5, 2, 0, 0, 0, 1, 0]
    blob[-96 + 8 * 5:-96 + 8 * 6] = np.array(kept, np.uint8)              # 17 .. 32 rows
    blob[-96 + 8 * 6:-96 + 8 * 7] = np.array([1, 6, 0, 0, 0, 0, 0, 0], np.uint8)
    back = T.MarlinWeight.import_blob(dev, blob)
    assert back.tuned_plan(64) is None and list(back.tuned_plan(20).values())[-7:] == kept[1:]
    a16 = O.synth_act_f16(20, k, 1703)
    c = T.GpuTensor.from_host(dev, np.full((20, n), np.nan, np.float32))
    T.gemm(dev, back, T.GpuTensor.from_host(dev, a16, "f16"), 20, c)
    close_rows(c.to_host(), gemm_truth(a16.view(np.float16).astype(np.float32).reshape(20, k), packed, scales, 20, k, n), F32_SUM)
    back.free()
    w.free()


@pytest.mark.parametrize("nt,taken", [(5, True), (10, True), (7, False), (9, False), (11, False)])
def test_column_tile_counts_of_saved_plans_and_of_the_option(dev, nt, taken):
    w = weight(dev, 256, 128, 1711)[2]
    blob = w.export_blob()
    blob[-96 + 8 * 5:-96 + 8 * 6] = np.array([1, 5, nt, 0, 0, 0, 1, 0], np.uint8)
    back = T.MarlinWeight.import_blob(dev, blob)
    assert (back.tuned_plan(20) is not None) == taken
    try:
        if taken:
            dev.set_option("nt", nt)
        else:
            with pytest.raises(T.DeviceError):
                dev.set_option("nt", nt)
    finally:
        dev.set_option("nt", 0)
    back.free()
    w.free()


# 48 .. 128-row blocks of 128 columns: a block's last row and the next one's first, K of one group, of two chunks and of an
# odd number with a ragged end, N ragged below and above a block; K-split and plain stores, f16 rows and scaled f32 rows
@pytest.mark.parametrize("form", [49, 65, 97, 129])
@pytest.mark.parametrize("m", [33, 48, 49, 64, 65, 96, 97, 128, 129, 193])
def test_prefill_blocks_of_128_columns(dev, m, form):
    for k, n, splits in ((32, 9, 1), (256, 132, 1), (672, 257, 1), (1312, 260, 3)):
        packed, scales, w = weight(dev, k, n, 1500 + k + m)
        a16 = O.synth_act_f16(m, k, 1503 + m)
        a = a16.view(np.float16).astype(np.float32).reshape(m, k).copy()
        big = a.copy()
        big[0] *= np.float32(2.0 ** 18)
        for rows, dt, vals in ((a16, "f16", a), (big, "f32", big)):
            c = T.GpuTensor.from_host(dev, np.full((m, n), np.nan, np.float32))
            ad = T.GpuTensor.from_host(dev, rows, dt)
            try:
                dev.set_option("prefill_bm", form)
                T.gemm(dev, w, ad, m, c, splits=splits)
            finally:
                dev.set_option("prefill_bm", 0)
            close_rows(c.to_host(), gemm_truth(vals, packed, scales, m, k, n), 1e-3)
        w.free()


@pytest.mark.parametrize("form", [0, 49, 65, 97, 129])
@pytest.mark.parametrize("m,ffn,dtype", [(33, 32, "f16"), (48, 96, "f32"), (65, 160, "f16"), (96, 288, "f16"), (129, 96, "f32")])
def test_prefill_gate_on_128_columns(dev, m, ffn, dtype, form):
    k = 416
    gate, up = [(O.synth_packed(k, ffn, s), O.synth_scales(k, ffn, s + 1)) for s in (1611, 1613)]
    pair = [tuple(T.GpuTensor.from_host(dev, x, t) for x, t in zip(w, ("u8", "f16"))) for w in (gate, up)]
    w = T.MarlinWeight.gate_up(dev, *pair, k, ffn)
    a16 = O.synth_act_f16(m, k, 1615)
    a = a16.view(np.float16).astype(np.float32).reshape(m, k).copy()
    if dtype == "f32":
        a[1] *= np.float32(2.0 ** -21)
    g, u = (gemm_truth(a, *x, m, k, ffn) for x in (gate, up))
    truth = g / (1.0 + np.exp(-g)) * u
    ad = T.GpuTensor.from_host(dev, a16, "f16") if dtype == "f16" else T.GpuTensor.from_host(dev, a)
    for splits in (1, 3):
        out = T.GpuTensor.from_host(dev, np.full((m, ffn), np.nan, np.float32))
        try:
            dev.set_option("prefill_bm", form)
            T.gemm_swiglu(dev, w, ad, m, out, splits)
        finally:
            dev.set_option("prefill_bm", 0)
        close_rows(out.to_host(), truth, 2e-3)   # (a product of two sums at 1e-3 each)
    w.free()


@pytest.mark.parametrize("m,option,value,exact", [(40, "prefill_min_m", 1 << 30, True), (24, "prefill_min_m", 8, False), (24, "batch_rounded", 1, False),
                                                  (40, None, 0, False), (24, None, 0, True)])
def test_measured_plans_keep_the_arithmetic_that_the_options_ask_for(dev, m, option, value, exact):
    # a measured plan of kernel 5 (exact weights up to 32 rows, f16-rounded ones above) on a context whose options ask for the
    # other arithmetic at that row count: the planners' choice runs.  At 2e-4 and 1e-3 of the floor in close_rows the two
    # arithmetics, 2^-12 of each weight apart, are told apart by the outputs that nearly cancel.
    k, n = 256, 128
    packed, scales, w = weight(dev, k, n, 1801)
    blob = w.export_blob()
    for bucket in (5, 6):                                                  # 17 .. 32 and 33 .. 64 rows
        blob[-96 + 8 * bucket:-96 + 8 * (bucket + 1)] = np.array([1, 5, 2, 0, 0, 0, 1, 0], np.uint8)
    back = T.MarlinWeight.import_blob(dev, blob)
    a16 = O.synth_act_f16(m, k, 1803)
    a = a16.view(np.float16).astype(np.float32).reshape(m, k)
    c = T.GpuTensor.from_host(dev, np.full((m, n), np.nan, np.float32))
    try:
        if option:
            dev.set_option(option, value)
        T.gemm(dev, back, T.GpuTensor.from_host(dev, a16, "f16"), m, c)
    finally:
        dev.set_option("prefill_min_m", 33)
        dev.set_option("batch_rounded", 0)
    w16 = O.dequant_f16(packed, scales, k, n).view(np.float16).astype(np.float64).reshape(k, n)
    truths = {True: O.gemm_f64(a, packed, scales, m, k, n), False: a.astype(np.float64) @ w16}
    close_rows(c.to_host(), truths[exact], F32_SUM if exact else 1e-3)
    with pytest.raises(AssertionError):
        close_rows(c.to_host(), truths[not exact], 1e-3)
    back.free()
    w.free()


@pytest.mark.parametrize("m", [7, 9, 16])
def test_a_column_lane_handle_keeps_its_one_copy_on_narrow_matrices(dev, m):
    # the documented range of the column-lane copy: captured without a second copy, and run eagerly without building one
    k, n = 2048, 2048
    dev.set_option("weight_copies", T.MarlinWeight.COPY_COLUMN_LANE)
    packed, scales, w = weight(dev, k, n, 1901)
    dev.set_option("weight_copies", 0)
    a16 = O.synth_act_f16(m, k, 1903 + m)
    a = T.GpuTensor.from_host(dev, a16, "f16")
    truth = O.gemm_f64(a16.view(np.float16).astype(np.float32).reshape(m, k), packed, scales, m, k, n)
    c = T.GpuTensor.from_host(dev, np.full((m, n), np.nan, np.float32))
    graph = T.GraphCapture.record_with_device(dev, lambda: T.gemm(dev, w, a, m, c))
    graph.replay()
    dev.synchronize()
    close_rows(c.to_host(), truth, F32_SUM)
    c.copy_from_host(np.full((m, n), np.nan, np.float32))
    T.gemm(dev, w, a, m, c)
    close_rows(c.to_host(), truth, F32_SUM)
    assert w.copies == T.MarlinWeight.COPY_COLUMN_LANE
    graph.destroy()
    w.free()


def test_a_measured_plan_does_not_ask_for_a_dropped_copy(dev):
    # a plan of kernel 5 (16-column tiles) on a handle that holds the column lanes: the planners' choice from what is held,
    # inside a capture too; with the copy back, the plan
    m, k, n = 16, 2048, 1024
    dev.set_option("weight_copies", T.MarlinWeight.COPY_COLUMN_LANE)
    packed, scales, w = weight(dev, k, n, 1951)
    dev.set_option("weight_copies", 0)
    blob = w.export_blob()
    blob[-96 + 8 * 4:-96 + 8 * 5] = np.array([1, 5, 1, 0, 0, 0, 1, 0], np.uint8)       # 9 .. 16 rows
    back = T.MarlinWeight.import_blob(dev, blob)
    a16 = O.synth_act_f16(m, k, 1953)
    a = T.GpuTensor.from_host(dev, a16, "f16")
    truth = O.gemm_f64(a16.view(np.float16).astype(np.float32).reshape(m, k), packed, scales, m, k, n)
    c = T.GpuTensor.from_host(dev, np.full((m, n), np.nan, np.float32))
    graph = T.GraphCapture.record_with_device(dev, lambda: T.gemm(dev, back, a, m, c))
    graph.replay()
    dev.synchronize()
    close_rows(c.to_host(), truth, F32_SUM)
    assert back.copies == T.MarlinWeight.COPY_COLUMN_LANE
    back.ensure(3)
    c.copy_from_host(np.full((m, n), np.nan, np.float32))
    T.gemm(dev, back, a, m, c)
    close_rows(c.to_host(), truth, F32_SUM)
    graph.destroy()
    back.free()
    w.free()


@pytest.mark.parametrize("k,m", [(416, 9), (416, 16), (992, 5), (2080, 8), (2080, 16)])
def test_an_infinite_activation_reaches_every_column_as_itself(dev, k, m):
    # K one group past a 128-deep chunk: the padded part of the last chunk must not multiply an infinity by its zero weights.
    # The infinity stands in the first and last piece of that chunk, and in the first of the row.  (Row counts and depths
    # that k_waves takes.)
    n = 96
    packed, scales, w = weight(dev, k, n, 2001)
    dense = O.dequant_f32(packed, scales, k, n).reshape(k, n)
    a16 = O.synth_act_f16(m, k, 2003)
    rows = a16.view(np.float16).reshape(m, k).copy()
    places = {1: k // 128 * 128, 3: k - 1, m - 1: 0}
    for r, p in places.items():
        rows[r, p] = np.inf
    c = T.GpuTensor.from_host(dev, np.full((m, n), -1.0, np.float32))
    T.gemm(dev, w, T.GpuTensor.from_host(dev, rows.view(np.uint16), "f16"), m, c)
    got = c.to_host()
    for r, p in places.items():
        want = np.where(dense[p] == 0, np.nan, np.copysign(np.inf, dense[p])).astype(np.float32)
        assert np.array_equal(got[r], want, equal_nan=True), (r, p)
    others = [r for r in range(m) if r not in places]
    truth = O.gemm_f64(rows[others].astype(np.float32), packed, scales, len(others), k, n)
    close_rows(got[others], truth, F32_SUM)
    w.free()


# One to four rows on a lane per column and group: whole chunks that leave slots of a wave without one (28 chunks on eight waves
# of four), chunks that each wave has one of, a padded last chunk, and both
@pytest.mark.parametrize("k,m", [(3584, 1), (3584, 2), (3584, 4), (256, 1), (1920, 1), (1440, 1), (1440, 3), (2592, 2), (3616, 4), (96, 1)])
def test_an_infinite_activation_of_a_few_rows_reaches_every_column_as_itself(dev, k, m):
    n = 96
    packed, scales, w = weight(dev, k, n, 2011)
    dense = O.dequant_f32(packed, scales, k, n).reshape(k, n)
    a16 = O.synth_act_f16(m, k, 2013)
    for p in (0, k // 128 * 128 if k % 128 else k - 128, k - 1):
        rows = a16.view(np.float16).reshape(m, k).copy()
        rows[m - 1, p] = np.inf
        c = T.GpuTensor.from_host(dev, np.full((m, n), -1.0, np.float32))
        T.gemm(dev, w, T.GpuTensor.from_host(dev, rows.view(np.uint16), "f16"), m, c)
        got = c.to_host()
        want = np.where(dense[p] == 0, np.nan, np.copysign(np.inf, dense[p])).astype(np.float32)
        assert np.array_equal(got[m - 1], want, equal_nan=True), p
        if m > 1:
            close_rows(got[:m - 1], O.gemm_f64(rows[:m - 1].astype(np.float32), packed, scales, m - 1, k, n), F32_SUM)
    w.free()


# 256 and 768 values are two and six chunks: the last pass of a wave has lane groups without one; four waves, of which all but
# one or two have no pass; a shape whose every lane group has a chunk of its own
@pytest.mark.parametrize("k,waves", [(256, 0), (768, 0), (768, 4), (512, 0), (512, 4), (2816, 0)])
def test_an_infinite_activation_of_a_bank_row_reaches_every_column_as_itself(dev, k, waves):
    n, experts, ids_h = 192, 3, np.array([2, 0], np.float32)
    raw = [(O.synth_packed(k, n, 2021 + e), O.synth_scales(k, n, 2031 + e)) for e in range(experts)]
    p, s = (T.GpuTensor.from_host(dev, np.concatenate([x[i].reshape(-1) for x in raw])) for i in (0, 1))
    bank = T.ExpertBank.from_device(dev, p, s, raw[0][0].size, raw[0][1].size, k, n, experts)
    dense = [O.dequant_f32(*raw[int(e)], k, n).reshape(k, n) for e in ids_h]
    ids, wts = T.GpuTensor.from_host(dev, ids_h), T.GpuTensor.from_host(dev, np.array([0.5, 0.25], np.float32))
    a16 = O.synth_act_f16(2, k, 2041)
    for at in (0, k - 128, k - 1):
        rows = a16.view(np.float16).reshape(2, k).copy()
        rows[:, at] = np.inf
        each = np.stack([np.where(d[at] == 0, np.nan, np.copysign(np.inf, d[at])) for d in dense]).astype(np.float32)
        a = T.GpuTensor.from_host(dev, rows.view(np.uint16), "f16")
        out = T.GpuTensor.from_host(dev, np.full((2, n), -1.0, np.float32))
        acc = T.GpuTensor.zeros(dev, (n,), "f32")
        dev.set_option("waves", waves)
        try:
            T.batched_marlin_gate_up(dev, a, bank, ids, out, 2, per_slot_rows=True)
            T.batched_marlin_down_axpy(dev, a, bank, ids, wts, acc, 2)
        finally:
            dev.set_option("waves", 0)
        assert np.array_equal(out.to_host(), each, equal_nan=True), at
        with np.errstate(invalid="ignore"):
            both = each[0] + each[1]
        assert np.array_equal(acc.to_host(), both, equal_nan=True), at
    bank.free()


@pytest.mark.parametrize("k,slots", [(1184, 4), (9344, 1)])
def test_bank_kernels_take_the_sub_tile_width_asked_for(dev, k, slots):
    # the widths add a pass's chunks in another order, which shows in the last bits of some column
    n, experts, ids_h = 192, 3, np.array([2, 0, 1, 1], np.float32)[:slots]
    raw = [(O.synth_packed(k, n, 2051 + e), O.synth_scales(k, n, 2061 + e)) for e in range(experts)]
    p, s = (T.GpuTensor.from_host(dev, np.concatenate([x[i].reshape(-1) for x in raw])) for i in (0, 1))
    bank = T.ExpertBank.from_device(dev, p, s, raw[0][0].size, raw[0][1].size, k, n, experts)
    ids, wts_h = T.GpuTensor.from_host(dev, ids_h), np.array([0.5, 0.25, 0.125, 1.0], np.float32)[:slots]
    a16 = O.synth_act_f16(slots, k, 2071)
    rows, a, wts = a16.view(np.float16).astype(np.float32).reshape(slots, k), T.GpuTensor.from_host(dev, a16, "f16"), T.GpuTensor.from_host(dev, wts_h)
    truth = np.concatenate([O.gemm_f64(rows[i:i + 1], *raw[int(ids_h[i])], 1, k, n) for i in range(slots)])
    got = {}
    for width in (16, 32):
        dev.set_option("sub", width)
        try:
            out, acc = T.GpuTensor.from_host(dev, np.full((slots, n), np.nan, np.float32)), T.GpuTensor.zeros(dev, (n,), "f32")
            T.batched_marlin_gate_up(dev, a, bank, ids, out, slots, per_slot_rows=True)
            T.batched_marlin_down_axpy(dev, a, bank, ids, wts, acc, slots)
        finally:
            dev.set_option("sub", 0)
        got[width] = out.to_host(), acc.to_host()
        close_rows(got[width][0], truth, F32_SUM)
        close_rows(got[width][1].reshape(1, n), (wts_h.astype(np.float64)[:, None] * truth).sum(0, keepdims=True), F32_SUM)
    assert not np.array_equal(got[16][0], got[32][0]) and not np.array_equal(got[16][1], got[32][1])
    bank.free()


# one chunk in part, the most chunks with one each per wave and one more, K one group past whole chunks, four chunks per wave of
# sixteen waves; a column and a sub-tile more than whole tiles
@pytest.mark.parametrize("k,n", [(32, 1), (96, 17), (1408, 81), (1440, 64), (2592, 130), (3616, 33), (8192, 65)])
@pytest.mark.parametrize("m,dtype", [(1, "f16"), (2, "f16"), (3, "f16"), (4, "f16"), (1, "f32")])
def test_up_to_four_rows_on_small_matrices(dev, k, n, m, dtype):
    packed, scales, w = weight(dev, k, n, 2101)
    a16 = O.synth_act_f16(m, k, 2103)
    a = a16.view(np.float16).astype(np.float32).reshape(m, k).copy()
    if dtype == "f32":
        a[0, : k // 2] *= np.float32(2.0 ** 20)      # half of the row outside the f16 range
    parts = [n] if n < 3 else [n // 2, n - n // 2]
    outs = [T.GpuTensor.from_host(dev, np.full((m, x), np.nan, np.float32)) for x in parts]
    b = O.synth_normal_f32(n, 2105)
    bias = [T.GpuTensor.from_host(dev, x) for x in np.split(b, np.cumsum(parts)[:-1])]
    T.gemm_split(dev, w, T.GpuTensor.from_host(dev, a16, "f16") if dtype == "f16" else T.GpuTensor.from_host(dev, a), m, outs, parts, biases=bias)
    truth = O.gemm_f64(a, packed, scales, m, k, n)
    got = np.concatenate([o.to_host() for o in outs], axis=1)
    floor = np.maximum(np.abs(truth), 1e-3 * np.abs(truth).max(axis=1, keepdims=True))
    assert (np.abs(got - (truth + b)) <= F32_SUM * floor + 2.0 ** -23 * np.abs(truth + b)).all()
    w.free()


@pytest.mark.parametrize("k,ffn", [(32, 32), (1440, 96), (2720, 32), (8192, 64)])
@pytest.mark.parametrize("m,dtype", [(1, "f16"), (2, "f16"), (4, "f16"), (1, "f32")])
def test_up_to_four_rows_gated_on_small_matrices(dev, k, ffn, m, dtype):
    gate, up = [(O.synth_packed(k, ffn, s), O.synth_scales(k, ffn, s + 1)) for s in (2111, 2113)]
    pair = [tuple(T.GpuTensor.from_host(dev, x, t) for x, t in zip(w, ("u8", "f16"))) for w in (gate, up)]
    w = T.MarlinWeight.gate_up(dev, *pair, k, ffn)
    a16 = O.synth_act_f16(m, k, 2115)
    a = a16.view(np.float16).astype(np.float32).reshape(m, k)
    g, u = (O.gemm_f64(a, *x, m, k, ffn) for x in (gate, up))
    out = T.GpuTensor.from_host(dev, np.full((m, ffn), np.nan, np.float32))
    T.gemm_swiglu(dev, w, T.GpuTensor.from_host(dev, a16, "f16") if dtype == "f16" else T.GpuTensor.from_host(dev, a), m, out)
    close_rows(out.to_host(), g / (1.0 + np.exp(-g)) * u, F32_SUM)
    w.free()


@pytest.mark.parametrize("copies,gemms", [(1, 0), (1, 1), (3, 17), (4, 16), (5, 16), (2, 30)])
def test_graphs_about_the_longest_that_replays_launch_by_launch(dev, copies, gemms):
    # one node to 46, copies between the launches, replays with new inputs and eager work between them
    k, n = 256, 64
    packed, scales, w = weight(dev, k, n, 2201)
    a = T.GpuTensor.zeros(dev, (1, k), "f16")
    src = [T.GpuTensor.zeros(dev, (n,), "f32") for _ in range(copies)]
    dst = [T.GpuTensor.zeros(dev, (n,), "f32") for _ in range(copies)]
    outs = [T.GpuTensor.zeros(dev, (1, n), "f32") for _ in range(gemms)]

    def work():
        for i in range(max(copies, gemms)):
            if i < copies:
                T.quantize._check(T._lib.load().twm_memcpy_d2d(dev.handle, dst[i].ptr, src[i].ptr, 4 * n))
            if i < gemms:
                T.gemm(dev, w, a, 1, outs[i])

    graph = T.GraphCapture.record_with_device(dev, work)
    for rep in range(3):
        rows = O.synth_act_f16(1, k, 2203 + rep)
        a.copy_from_host(rows.reshape(1, k))
        for i, s in enumerate(src):
            s.copy_from_host(np.full(n, 10 * rep + i, np.float32))
        graph.replay()
        dev.synchronize()
        truth = O.gemm_f64(rows.view(np.float16).astype(np.float32).reshape(1, k), packed, scales, 1, k, n)
        for o in outs:
            close_rows(o.to_host(), truth, F32_SUM)
        for i, d in enumerate(dst):
            assert (d.to_host() == 10 * rep + i).all()
        eager = T.GpuTensor.zeros(dev, (1, n), "f32")
        T.gemm(dev, w, a, 1, eager)
        assert all(np.array_equal(eager.to_host(), o.to_host()) for o in outs)
    graph.destroy()
    w.free()


# one pass per wave and the loop over passes, with and without a K-split, on both widths
@pytest.mark.parametrize("k,n,sub,splits", [(3584, 200, 16, 0), (3584, 200, 32, 0), (9344, 128, 16, 0), (9344, 128, 32, 3), (3584, 200, 16, 2)])
def test_traced_sub_tiles_compute_what_the_untraced_do(dev, k, n, sub, splits):
    packed, scales, w = weight(dev, k, n, 2501)
    a16 = O.synth_act_f16(1, k, 2503)
    a = T.GpuTensor.from_host(dev, a16, "f16")
    trace = T.GpuTensor.zeros(dev, (4 * 64,), "i32")
    got = []
    dev.set_option("sub", sub)
    try:
        for on in (False, True):
            if on:
                T.quantize._check(T._lib.load().twm_debug_trace(dev.handle, trace.ptr, 64))
            c = T.GpuTensor.from_host(dev, np.full((1, n), np.nan, np.float32))
            T.gemm(dev, w, a, 1, c, splits=splits)
            got.append(c.to_host())
            assert trace.to_host().any() == on
    finally:
        dev.set_option("sub", 0)
        T.quantize._check(T._lib.load().twm_debug_trace(dev.handle, None, 0))
    close_rows(got[0], O.gemm_f64(a16.view(np.float16).astype(np.float32).reshape(1, k), packed, scales, 1, k, n), F32_SUM)
    assert np.array_equal(got[0], got[1])
    w.free()


def replays_as_launches(graph):
    # (the second pointer of the handle is the instantiated graph; null: the nodes are launched)
    return C.c_void_p.from_address(graph.handle + 8).value is None


# small launches up to five nodes, those that give every SIMD a wave up to seven, copies counted as nodes without a wave
@pytest.mark.parametrize("k,n,gemms,copies,launched", [(128, 512, 5, 0, True), (128, 512, 6, 0, False), (128, 512, 1, 4, True), (128, 512, 1, 5, False),
                                                       (3584, 3584, 7, 0, True), (3584, 3584, 8, 0, False), (3584, 3584, 5, 1, True),
                                                       (3584, 3584, 3, 3, False)])
def test_which_graphs_replay_launch_by_launch(dev, k, n, gemms, copies, launched):
    w = T.MarlinWeight.upload(dev, O.synth_packed(k, n, 2401), O.synth_scales(k, n, 2402), k, n)
    a = T.GpuTensor.from_host(dev, O.synth_act_f16(1, k, 2403), "f16")
    outs = [T.GpuTensor.zeros(dev, (1, n), "f32") for _ in range(gemms + copies)]

    def work():
        for o in outs[:gemms]:
            T.gemm(dev, w, a, 1, o)
        for o in outs[gemms:]:
            T.quantize._check(T._lib.load().twm_memcpy_d2d(dev.handle, o.ptr, outs[0].ptr, 4 * n))

    graph = T.GraphCapture.record_with_device(dev, work)
    assert replays_as_launches(graph) == launched
    eager = T.GpuTensor.zeros(dev, (1, n), "f32")
    T.gemm(dev, w, a, 1, eager)
    for _ in range(3):
        for o in outs:
            o.copy_from_host(np.full(n, np.nan, np.float32))
        graph.replay()
        dev.synchronize()
        assert all(np.array_equal(o.to_host(), eager.to_host()) for o in outs)
    graph.destroy()
    w.free()


def test_a_graph_with_a_kernel_of_the_callers_own_stays_one(dev, tmp_path):
    # a second copy of the library stands for the caller's own code: its fill kernel, launched on the context's stream
    class Dim3(C.Structure):
        _fields_ = [(c, C.c_uint32) for c in "xyz"]

    other = C.CDLL(shutil.copy(T._lib.LIB_PATH, tmp_path / "other.so"))
    hip = C.CDLL("libamdhip64.so.7")
    hip.hipLaunchKernel.argtypes = [C.c_void_p, Dim3, Dim3, C.POINTER(C.c_void_p), C.c_size_t, C.c_void_p]
    words = 64
    buf = T.GpuTensor.from_host(dev, np.full(words, 7, np.int32))
    ptr, count = C.c_void_p(buf.ptr), C.c_size_t(words)
    args = (C.c_void_p * 2)(C.addressof(ptr), C.addressof(count))

    def work(lib):
        kernel = C.addressof(C.c_char.in_dll(lib, "_ZN3twm11k_fill_zeroEPjm"))
        assert hip.hipLaunchKernel(kernel, Dim3(1, 1, 1), Dim3(64, 1, 1), args, 0, T._lib.load().twm_ctx_stream(dev.handle)) == 0

    for lib, launched in ((T._lib.load(), True), (other, False)):
        graph = T.GraphCapture.record_with_device(dev, lambda: work(lib))
        assert replays_as_launches(graph) == launched
        for _ in range(2):
            buf.copy_from_host(np.full(words, 7, np.int32))
            graph.replay()
            dev.synchronize()
            assert not buf.to_host().any()
        graph.destroy()


# 64- and 96-row blocks of 192 columns, and the 128-row ones with the gated store: a block's last row and the next one's first,
# K of one group and with a ragged end, columns a quad below and above a block's three
@pytest.mark.parametrize("form", [66, 98])
@pytest.mark.parametrize("m", [33, 64, 65, 96, 97, 193])
def test_prefill_blocks_of_192_columns(dev, m, form):
    for k, n, splits in ((32, 9, 1), (672, 193, 1), (1312, 388, 3)):
        packed, scales, w = weight(dev, k, n, 2300 + k + m)
        a16 = O.synth_act_f16(m, k, 2303 + m)
        a = a16.view(np.float16).astype(np.float32).reshape(m, k).copy()
        big = a.copy()
        big[m - 1] *= np.float32(2.0 ** 18)
        for rows, dt, vals in ((a16, "f16", a), (big, "f32", big)):
            c = T.GpuTensor.from_host(dev, np.full((m, n), np.nan, np.float32))
            try:
                dev.set_option("prefill_bm", form)
                T.gemm(dev, w, T.GpuTensor.from_host(dev, rows, dt), m, c, splits=splits)
            finally:
                dev.set_option("prefill_bm", 0)
            close_rows(c.to_host(), gemm_truth(vals, packed, scales, m, k, n), 1e-3)
        w.free()


# Row stores of split outputs: segments that start on every fourth column and one that does not, across blocks' columns, with
# and without biases and K-splits, at an output address that is not 16-byte aligned
@pytest.mark.parametrize("widths", [(8, 200, 4), (184, 8, 200), (192, 192, 192), (201, 7, 60)])
@pytest.mark.parametrize("form,splits", [(98, 1), (192, 1), (66, 3), (128, 1), (65, 2)])
def test_prefill_rows_into_segments(dev, widths, form, splits):
    m, k, n = 99, 672, sum(widths)
    packed, scales, w = weight(dev, k, n, 2330)
    a16 = O.synth_act_f16(m, k, 2333)
    truth = gemm_truth(a16.view(np.float16).astype(np.float32).reshape(m, k), packed, scales, m, k, n)
    a = T.GpuTensor.from_host(dev, a16, "f16")
    biases = [np.linspace(-1, 1, x, dtype=np.float32) for x in widths]
    for shift in (0, 1):
        full = [T.GpuTensor.from_host(dev, b) for b in biases]
        for bias in (None, full, [full[0], None, full[2]]):
            outs = [T.GpuTensor.from_host(dev, np.full(m * x + shift, np.nan, np.float32)) for x in widths]
            places = [SimpleNamespace(ptr=o.ptr + 4 * shift) for o in outs]
            try:
                dev.set_option("prefill_bm", form)
                T.gemm_split(dev, w, a, m, places, list(widths), biases=bias, splits=splits)
            finally:
                dev.set_option("prefill_bm", 0)
            got = np.concatenate([o.to_host()[shift:].reshape(m, -1) for o in outs], 1)
            added = [b if t is not None else 0 * b for b, t in zip(biases, bias or [None] * 3)]
            close_rows(got, truth + np.concatenate(added), 1e-3)
    w.free()


@pytest.mark.parametrize("form", [66, 98, 192])
@pytest.mark.parametrize("m,ffn", [(33, 32), (65, 96), (97, 128), (129, 288), (260, 6304)])
def test_prefill_gate_on_192_columns(dev, m, ffn, form):
    # (260 rows x 6304 features: more workgroups of 128 x 192 than CUs, the form of which two share one)
    k = 416
    gate, up = [(O.synth_packed(k, ffn, s), O.synth_scales(k, ffn, s + 1)) for s in (2311, 2313)]
    pair = [tuple(T.GpuTensor.from_host(dev, x, t) for x, t in zip(w, ("u8", "f16"))) for w in (gate, up)]
    w = T.MarlinWeight.gate_up(dev, *pair, k, ffn)
    a16 = O.synth_act_f16(m, k, 2315)
    a = a16.view(np.float16).astype(np.float32).reshape(m, k)
    g, u = (gemm_truth(a, *x, m, k, ffn) for x in (gate, up))
    out = T.GpuTensor.from_host(dev, np.full((m, ffn), np.nan, np.float32))
    try:
        dev.set_option("prefill_bm", form)
        T.gemm_swiglu(dev, w, T.GpuTensor.from_host(dev, a16, "f16"), m, out, 1)
    finally:
        dev.set_option("prefill_bm", 0)
    close_rows(out.to_host(), g / (1.0 + np.exp(-g)) * u, 2e-3)   # (a product of two sums at 1e-3 each)
    w.free()


@pytest.mark.parametrize("m", [5, 8, 9, 16, 17, 31, 32])
def test_ranges_staged_at_once(dev, m):
    # k_batch_range: row blocks of 8, 16 and 32 rows and their remainders; ranges of an uneven number of chunks and a shorter last
    # one; K that ends inside a chunk, N inside a workgroup's columns; rows beyond the f16 range on both sides, one infinite row;
    # segments with biases
    k, n = (20512, 1157) if m > 16 else (22624, 1725)
    assert "k_batch_range" in dev.plan(k, n, m, dtype="f32")
    packed, scales, w = weight(dev, k, n, 1700 + m)
    a = O.synth_normal_f32(m * k, 1703 + m).reshape(m, k).copy()
    a[0] *= np.float32(3e7)
    a[1] *= np.float32(1e-9)
    a[m - 1, k - 1] = np.float32(4e5)
    a[2, ::3] *= np.float32(2.0 ** -20)
    truth = O.gemm_f64(a, packed, scales, m, k, n)
    a[3, k // 2] = np.inf
    ns = [n - 500, 499, 1]
    biases = [O.synth_normal_f32(x, 1709 + x) for x in ns]
    outs = [T.GpuTensor.from_host(dev, np.full((m, x), np.nan, np.float32)) for x in ns]
    T.gemm_split(dev, w, T.GpuTensor.from_host(dev, a), m, outs, ns, biases=[T.GpuTensor.from_host(dev, b) for b in biases])
    got = np.concatenate([o.to_host() - b for o, b in zip(outs, biases)], 1).astype(np.float64)
    keep = [r for r in range(m) if r not in (1, 3)]
    assert not np.isfinite(got[3]).any()
    close_rows(got[keep], truth[keep], F32_SUM)
    c = T.GpuTensor.from_host(dev, np.full((m, n), np.nan, np.float32))
    T.gemm(dev, w, T.GpuTensor.from_host(dev, a), m, c)          # (without a bias the row of 1e-9 is seen to its last digits)
    close_rows(c.to_host()[[1] + keep], truth[[1] + keep], F32_SUM)
    w.free()


@pytest.mark.parametrize("m", [5, 8, 16, 17, 32])
def test_large_values_of_other_chunks_take_no_bits_in_ranges_staged_at_once(dev, m):
    # f32 rows of k_batch_range: every fourth chunk holds a 2^40 alone, on weights of 0 in the first half of the columns; there the
    # results are the other chunks' sums, whose values keep their bits
    k, n = (20512, 1157) if m > 16 else (22624, 1725)
    assert "k_batch_range" in dev.plan(k, n, m, dtype="f32")
    half, packed, scales = n // 2, O.synth_packed(k, n, 1721).reshape(k // 32, n, 16), O.synth_scales(k, n, 1722)
    a = O.synth_normal_f32(m * k, 1723 + m).reshape(m, k).copy()
    for c in range(1, k // 128, 4):
        a[:, 128 * c: 128 * (c + 1)] = 0
        a[:, 128 * c + 32 + c % 32] = np.float32(2.0 ** 40)
        packed[4 * c + 1, :half] = 0x88                           # (the group that holds it)
    truth = O.gemm_f64(a, packed, scales, m, k, n)
    w = T.MarlinWeight.upload(dev, packed, scales, k, n)
    c = T.GpuTensor.from_host(dev, np.full((m, n), np.nan, np.float32))
    T.gemm(dev, w, T.GpuTensor.from_host(dev, a), m, c)
    close_rows(c.to_host()[:, :half], truth[:, :half], F32_SUM)
    w.free()


@pytest.mark.parametrize("m,k,n,gated,chunks,splits", [(8, 39712, 1707, False, 18, 18), (5, 32800, 1835, False, 16, 17), (16, 39712, 1707, False, 18, 18),
                                                       (13, 32800, 1835, False, 16, 17), (32, 43936, 1323, False, 9, 39), (20, 43808, 1323, False, 9, 39),
                                                       (17, 43680, 1323, False, 9, 38), (27, 43808, 1344, True, 9, 39)])
def test_ranges_of_as_many_chunks_as_a_workgroup_stages(dev, m, k, n, gated, chunks, splits):
    # k_batch_range: the longest ranges, 147 KB of staged rows, and last ranges of all chunks, two and one (whose second k-slice is
    # empty) with a K that ends inside them; f32 values with a second term.  The sums of a range's chunks are a chain of up to nine
    # additions, those of the ranges a tree: 1.0 - 1.3e-7 of a row's norm (a lost second term would be 1e-4)
    assert dev.plan(k, n, m, dtype="f32", gated=gated).startswith("k_batch_range: ")
    assert "ranges of up to %d chunks staged at once, %d K-splits" % (chunks, splits) in dev.plan(k, n, m, dtype="f32", gated=gated)
    a = O.synth_normal_f32(m * k, 1803 + m).reshape(m, k) * np.float32(0.3)
    rows = T.GpuTensor.from_host(dev, a)
    if gated:
        ffn = n // 2
        parts = [(O.synth_packed(k, ffn, s), O.synth_scales(k, ffn, s + 1)) for s in (1811, 1821)]
        w = T.MarlinWeight.gate_up(dev, *([T.GpuTensor.from_host(dev, p), T.GpuTensor.from_host(dev, s, "f16")] for p, s in parts), k, ffn)
        g, u = (O.gemm_f64(a, *x, m, k, ffn) for x in parts)
        truth, c = g / (1.0 + np.exp(-g)) * u, T.GpuTensor.from_host(dev, np.full((m, ffn), np.nan, np.float32))
        T.gemm_swiglu(dev, w, rows, m, c)
    else:
        packed, scales, w = weight(dev, k, n, 1801)
        truth, c = O.gemm_f64(a, packed, scales, m, k, n), T.GpuTensor.from_host(dev, np.full((m, n), np.nan, np.float32))
        T.gemm(dev, w, rows, m, c)
    err = np.linalg.norm(c.to_host() - truth, axis=1) / np.linalg.norm(truth, axis=1)
    assert err.max() < (2e-6 if gated else 1e-6), err
    w.free()


def test_options_that_ask_for_other_forms_get_them(dev):
    # k_batch_range runs only where nothing is asked for
    k, n, m = 22624, 1725, 8
    for option, value in (("kernel", 4), ("kernel", 5), ("nt", 2), ("waves", 8), ("prefill_bm", 64)):
        assert dev.plan(k, n, m, dtype="f32").startswith("k_batch_range: ")
        dev.set_option(option, value)
        try:
            assert "k_batch_range" not in dev.plan(k, n, m, dtype="f32"), option
        finally:
            dev.set_option(option, 0)


@pytest.mark.parametrize("k,n,m", [(22624, 1725, 8), (22624, 1725, 16), (20512, 1157, 20)])
def test_f32_rows_run_alike_whichever_copy_a_handle_holds(dev, k, n, m):
    # k_batch_range on a handle of the column-lane copy alone: the first call, which builds the tile copy, is the launch of every
    # later one
    assert "k_batch_range" in dev.plan(k, n, m, dtype="f32")
    packed, scales, both = weight(dev, k, n, 1790)
    dev.set_option("weight_copies", T.MarlinWeight.COPY_COLUMN_LANE)
    one = T.MarlinWeight.upload(dev, packed, scales, k, n)
    dev.set_option("weight_copies", 0)
    a = T.GpuTensor.from_host(dev, O.synth_normal_f32(m * k, 1791).reshape(m, k))
    got = []
    for w in (both, one, one):
        c = T.GpuTensor.from_host(dev, np.full((m, n), np.nan, np.float32))
        T.gemm(dev, w, a, m, c)
        got.append(c.to_host().view(np.uint32))
    assert one.copies == 3
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    both.free()
    one.free()


def test_ranges_staged_at_once_under_a_gate(dev):
    m, k, ffn = 23, 20256, 1344
    assert "k_batch_range" in dev.plan(k, 2 * ffn, m, dtype="f32", gated=True)
    gate, up = ((O.synth_packed(k, ffn, s), O.synth_scales(k, ffn, s + 1)) for s in (1750, 1760))
    w = T.MarlinWeight.gate_up(dev, *([T.GpuTensor.from_host(dev, p), T.GpuTensor.from_host(dev, s, "f16")] for p, s in (gate, up)), k, ffn)
    a = 0.3 * O.synth_normal_f32(m * k, 1770).reshape(m, k)
    g, u = (O.gemm_f64(a, *x, m, k, ffn) for x in (gate, up))
    out = T.GpuTensor.from_host(dev, np.full((m, ffn), np.nan, np.float32))
    T.gemm_swiglu(dev, w, T.GpuTensor.from_host(dev, a), m, out)
    close_rows(out.to_host(), g / (1.0 + np.exp(-g)) * u, F32_SUM)
    w.free()


@pytest.mark.parametrize("m,dtype", [(1, "f16"), (4, "f16"), (5, "f16"), (8, "f16"), (9, "f16"), (12, "f16"), (13, "f16"), (16, "f16"), (17, "f16"), (24, "f16"),
                                     (25, "f16"), (9, "f32"), (12, "f32"), (13, "f32"), (17, "f32"), (24, "f32"), (25, "f32")])
@pytest.mark.parametrize("nt", [1, 3, 8])
def test_row_quads_of_waves_on_exact_weights(dev, m, dtype, nt):
    # k_waves_exact loads the rows by quads: the rows of a block behind them are whatever the LDS holds, here NaNs that a launch on
    # rows of them has left, and touch no other row
    k, n = 1312, 16 * nt + 21
    packed, scales, w = weight(dev, k, n, 1651 + nt)
    a16 = O.synth_act_f16(m, k, 1655 + m)
    a = a16.view(np.float16).astype(np.float32).reshape(m, k)
    rows = T.GpuTensor.from_host(dev, a16, "f16") if dtype == "f16" else T.GpuTensor.from_host(dev, a)
    nans = T.GpuTensor.from_host(dev, np.full((32, k), np.nan, np.float32))
    c, junk = T.GpuTensor.from_host(dev, np.full((m, n), np.nan, np.float32)), T.GpuTensor.zeros(dev, (32, n), "f32")
    dev.set_option("kernel", 5)
    try:
        dev.set_option("nt", nt)
        T.gemm(dev, w, nans, 32, junk)
        T.gemm(dev, w, rows, m, c)
    finally:
        dev.set_option("nt", 0)
        dev.set_option("kernel", 0)
    close_rows(c.to_host(), O.gemm_f64(a, packed, scales, m, k, n), F32_SUM)
    w.free()


@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 4095), (3, 4096), (3, 4097), (2, 8193), (1, 4096 * 65 + 1), (40, 4096 * 33), (1023, 8200), (1025, 4100), (2049, 70),
                                       (2, 8192), (512, 5000), (513, 5000), (3, 16383), (3, 16384), (2, 16385), (512, 8200), (513, 12300)])
def test_argmax_at_the_edges_of_its_spans(dev, rows, cols):
    # spans of 4096, 8192 and 16384 columns, one or several to a workgroup; more spans than lanes merge them; ties across spans and between
    # zeros of either sign, a largest value in the last column, rows without a candidate; a second call finds the counters clear
    x = np.round(O.synth_normal_f32(rows * cols, 1800 + cols).reshape(rows, cols) * 2).astype(np.float32)
    x[0, -1] = 1e9
    x[rows // 2] = -np.abs(x[rows // 2])
    x[rows // 2, cols // 3] = np.float32(-0.0)
    if rows > 1:
        x[rows - 1] = np.nan if cols % 2 else np.float32(-1e30)
    xd, out = T.GpuTensor.from_host(dev, x), T.GpuTensor.from_host(dev, np.full(rows, -7, np.int32))
    for _ in range(2):
        T.argmax(dev, xd, out, rows, cols)
        assert np.array_equal(out.to_host(), O.argmax(x, rows, cols))
