"""GPU tests of single kernels at the sizes where their tilings change: against the CPU oracle's f64 dequant-then-matmul or
its byte-exact format functions, through the C ABI."""
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
