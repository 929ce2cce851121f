"""The launch planners, through twm_plan_describe: no GPU is touched (the library is only loaded).

The plans of the benchmark shapes are held to what every good plan must keep (kernel family and repacked copy of a row
count, no K-split where the columns alone fill the CUs, enough workgroups otherwise), not to their text: a planner's
rule can be refitted without editing this file, and bench.py prints every plan line beside the time it led to.  The
same invariants are checked over a sweep of shapes."""
import ctypes
import re

import numpy as np
import pytest

from tensorwarp_amd import _lib


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


def describe(lib, k, n, m, dtype=None, gated=0):
    buf = ctypes.create_string_buffer(256)
    rc = lib.twm_plan_describe(None, k, n, m, _lib.F16 if dtype is None else dtype, gated, buf, 256)
    assert rc == 0, lib.twm_last_error().decode()
    return buf.value.decode()


QWEN7B = {"qkv": (3584, 4608), "o": (3584, 3584), "gate_up": (3584, 37888), "down": (18944, 3584)}


def parse(text):
    """The fields of a plan line."""
    f = {"kernel": text.split(":")[0], "copy": text.rsplit(";", 1)[1].strip(), "text": text}
    for key, pat in (("sub", r"(\d+)-column sub-tiles"), ("waves", r"(\d+) waves?"), ("chunks", r"of up to (\d+) chunk"), ("splits", r"(\d+) K-split"),
                     ("quads", r"(\d+) quads? per workgroup"), ("tiles_per_wave", r"(\d+) tiles? per wave"),
                     ("slices", r"(\d+) k-slice"), ("tiles64", r"(\d+) x 64-column tiles"),
                     ("block_rows", r"(\d+)-row x"), ("block_cols", r"x (\d+)-column blocks")):
        m = re.search(pat, text)
        if m:
            f[key] = int(m.group(1))
    return f


def workgroups(f, k, n, m):
    n_pad = (n + 63) // 64 * 64
    if f["kernel"] in ("k_gemv4s", "k_gemv4g"):
        return n_pad // f["sub"] * f["splits"]
    if f["kernel"] == "k_gemv4":
        return -(-(n_pad // 64) // f["tiles64"]) * f["splits"]
    if f["kernel"] == "k_batch":
        return -(-(n_pad // 64) // (f["quads"] * f["tiles_per_wave"])) * f["splits"]
    if f["kernel"] == "k_stream":
        return n_pad // 64 * f["splits"]
    if f["kernel"] in ("k_prefill", "k_waves", "k_waves_exact", "k_batch_range"):
        return -(-m // f["block_rows"]) * -(-n_pad // f["block_cols"]) * f["splits"]
    raise AssertionError(f["text"])


CUS = 256


@pytest.mark.parametrize("name", list(QWEN7B))
@pytest.mark.parametrize("m,dtype", [(1, "f16"), (1, "f32"), (2, "f16"), (4, "f16"), (8, "f16"), (16, "f16"), (32, "f16")])
def test_plans_of_the_qwen7b_projections(lib, name, m, dtype):
    # What every plan of the benchmark layer must keep, whatever rule of a planner produced it (the plan lines themselves
    # are printed by bench.py beside the times they led to): the kernel family of the row count, the repacked copy that
    # family reads, no K-split where the columns alone give a workgroup to at least half the CUs, enough workgroups
    # otherwise, and at one row the sub-tile kernel without a hand-over between workgroups.
    k, n = QWEN7B[name]
    f = parse(describe(lib, k, n, m, _lib.F32 if dtype == "f32" else _lib.F16))
    k_chunks, wgs = (k // 32 + 3) // 4, workgroups(f, k, n, m)
    if m <= 4:
        assert f["kernel"] in ("k_gemv4s", "k_gemv4g", "k_gemv4") and f["copy"] == "column-lane copy", f["text"]
        assert f["splits"] == 1, f["text"]                   # (a hand-over between workgroups costs over a microsecond)
    elif m <= 16:
        assert f["kernel"] in ("k_gemv4s", "k_gemv4", "k_stream", "k_batch", "k_waves_exact"), f["text"]
    else:
        assert f["kernel"] in ("k_batch", "k_waves_exact") and f["copy"] == "16-column tile copy", f["text"]
    if m == 1:
        assert f["kernel"] in ("k_gemv4s", "k_gemv4g") and wgs >= CUS // 2, f["text"]
        if f["kernel"] == "k_gemv4g":                         # a wave has up to four chunks, all of them in flight
            assert f["waves"] * f["chunks"] >= k_chunks and f["chunks"] <= 4, f["text"]
        elif k_chunks <= 32:                                  # K up to 4096: a wave makes one pass or two, no loop
            assert f["waves"] * (64 // f["sub"]) * 2 >= k_chunks, f["text"]
        else:                                                 # deep K: sixteen columns, few waves, the pass loop
            assert f["sub"] == 16 and f["waves"] in (4, 8, 16), f["text"]
    if f["kernel"] in ("k_stream", "k_batch", "k_waves_exact"):
        assert f["copy"] == "16-column tile copy" and 1 <= f["splits"] <= 16, f["text"]
        unsplit = wgs // f["splits"]
        if f["splits"] > 1:
            assert unsplit < CUS and "k_splitk_reduce" in f["text"], f["text"]   # only where the columns leave CUs idle
            assert k_chunks // f["splits"] >= 7, f["text"]                        # and every range keeps some depth
        if n >= 16384:
            assert f["splits"] == 1 and wgs >= 128, f["text"]                    # wide: the columns are enough


@pytest.mark.parametrize("k,n,m", [(4096, 11008, 2048), (11008, 4096, 2048), (4096, 11008, 512), (11008, 4096, 512),
                                   (3584, 4608, 2048), (3584, 37888, 128), (896, 1152, 64)])
def test_plans_of_prefill(lib, k, n, m):
    f = parse(describe(lib, k, n, m))
    assert f["kernel"] == "k_prefill" and f["copy"] == "16-column tile copy", f["text"]
    assert f["block_rows"] in (64, 128) and f["block_cols"] in (192, 256), f["text"]
    wgs, k_chunks = workgroups(f, k, n, m), (k // 32 + 3) // 4
    if f["splits"] > 1:
        assert wgs // f["splits"] < CUS // 2 and "k_splitk_reduce" in f["text"], f["text"]   # K is cut only to fill idle CUs
        assert k_chunks // f["splits"] >= 2, f["text"]
    if m >= 2048 and n >= 4096:
        assert f["block_rows"] == 128 and f["splits"] == 1 and wgs >= CUS, f["text"]        # enough tiles: the cheapest form per row


@pytest.mark.parametrize("k,n,m", [(15360, 64, 525), (13056, 64, 929), (11136, 320, 579), (16640, 320, 446), (13344, 128, 992), (384, 18624, 205), (128, 23232, 833),
                                   (160, 39552, 75)])
def test_gated_prompts_where_192_column_blocks_are_behind(lib, k, n, m):
    # under a K-split, which they make of many parts, and on a few chunks: 7 - 27 % behind the forms that run
    f = parse(describe(lib, k, n, m, gated=1))
    assert f["kernel"] == "k_prefill" and (f["block_cols"] != 192 or f["block_rows"] < (128 if k > 256 else 96)), f["text"]


def test_plans_of_lm_head_and_small_shapes(lib):
    lm = parse(describe(lib, 3584, 152064, 1))
    assert lm["kernel"] in ("k_gemv4", "k_gemv4s") and lm["splits"] == 1 and workgroups(lm, 3584, 152064, 1) >= 8 * CUS, lm["text"]
    small = parse(describe(lib, 896, 1152, 1))
    assert small["kernel"] == "k_gemv4g" and small["splits"] == 1, small["text"]            # small matrix, one row: a lane per column and group


def test_the_gated_store_takes_32_column_sub_tiles(lib):
    # 16 gate + 16 up columns per workgroup: with 8 + 8 the stores would be 128-byte runs
    assert describe(lib, 3584, 37888, 1, gated=1).startswith("k_gemv4s: 32-column sub-tiles")
    assert describe(lib, 3584, 37888, 1, gated=0).startswith("k_gemv4s: 16-column sub-tiles")


def test_pick_splits_agrees_with_the_described_plan(lib):
    rng = np.random.default_rng(7)
    for _ in range(400):
        k = 32 * int(rng.integers(1, 700))
        n = int(rng.integers(1, 60000))
        m = int(rng.choice([1, 2, 3, 4, 5, 8, 9, 16, 17, 32]))
        text = describe(lib, k, n, m)
        splits = int(re.search(r"(\d+) K-split", text).group(1))
        assert splits == lib.twm_pick_splits(k, n, m), (k, n, m, text)
        k_chunks = (k // 32 + 3) // 4
        assert 1 <= splits <= max(1, k_chunks), (k, n, m, text)
        # which rows go to which kernel family
        kernel = text.split(":")[0]
        if m <= 4:
            assert kernel in ("k_gemv4", "k_gemv4s", "k_gemv4g"), (k, n, m, text)
            assert "column-lane copy" in text
        if m > 16:
            assert kernel in ("k_batch", "k_waves_exact"), (k, n, m, text)
        if kernel == "k_gemv4s":
            sub, waves = map(int, re.search(r"(\d+)-column sub-tiles, (\d+) waves", text).groups())
            assert sub in (16, 32) and 1 <= waves <= 16
            if m > 4:   # rows beyond four repeat the MFMA chain: only in the one-pass form
                assert waves * (64 // sub) >= k_chunks, (k, n, m, text)


def test_plans_of_the_kernel_on_narrow_matrices(lib):
    # k_waves: blocks of whole tiles that divide the padded columns and whose rows pad less than a block, its arithmetic by
    # the row count, one round of workgroups on the CUs (two of the four-wave form), K cut only where that leaves CUs idle
    rng = np.random.default_rng(11)
    taken = set()
    for _ in range(6000):
        k, n = 32 * int(rng.integers(1, 200)), int(rng.choice([400, 3000, 20000]) * rng.random()) + 1
        m, gated = int(rng.integers(1, 260)), int(rng.integers(0, 2))
        n = n // 64 * 64 + 64 if gated else n
        dtype = _lib.F32 if rng.integers(0, 2) else _lib.F16
        f = parse(describe(lib, k, n, m, dtype, gated))
        if f["kernel"] != "k_waves":
            continue
        wgs, k_chunks = workgroups(f, k, n, m), (k // 32 + 3) // 4
        assert 33 <= m <= 192 and f["copy"] == "16-column tile copy" and "f16-rounded weights" in f["text"], f["text"]
        assert f["block_cols"] in ((32,) if gated else (16, 32)) and f["block_rows"] in (48, 64), f["text"]
        assert -(-m // f["block_rows"]) * f["block_rows"] - m < f["block_rows"], f["text"]
        assert wgs <= (CUS if f["waves"] == 8 else 2 * CUS) and (f["waves"] == 8 or 33 <= m <= 64), f["text"]
        blocks, groups = -(-m // f["block_rows"]), (n + 63) // 64 * 64 // f["block_cols"]
        if blocks > 1:  # the row blocks of a column group stay on one of the eight XCDs: one round on its 32 CUs
            assert -(-groups // 8) * blocks * f["splits"] <= CUS // 8, f["text"]
        if f["splits"] > 1:
            assert wgs // f["splits"] <= CUS // 2 and k_chunks // f["splits"] >= 8 and "k_splitk_reduce" in f["text"], f["text"]
        taken.add((f["block_rows"], f["block_cols"]))
    assert taken == {(48, 16), (48, 32), (64, 16), (64, 32)}, taken


def test_plans_of_the_few_row_kernels(lib):
    # k_gemv4g: up to four f16 rows or one f32 row, every wave's chunks in flight at once.  k_waves_exact: 5 .. 32 rows, blocks of
    # 16 or 32 rows x 1 .. 10 column tiles, a gate tile beside its up tile unless K is split, K split only into ranges of some
    # depth where the columns leave CUs idle
    rng = np.random.default_rng(13)
    seen = {"k_gemv4g": 0, "k_waves_exact": 0}
    for _ in range(6000):
        k, n = 32 * int(rng.integers(1, 600)), int(rng.choice([400, 3000, 40000]) * rng.random()) + 1
        m, gated = int(rng.integers(1, 5) if rng.integers(0, 2) else rng.integers(5, 34)), int(rng.integers(0, 2))
        n = n // 64 * 64 + 64 if gated else n
        f32 = bool(rng.integers(0, 2))
        f = parse(describe(lib, k, n, m, _lib.F32 if f32 else _lib.F16, gated))
        k_chunks, wgs = (k // 32 + 3) // 4, workgroups(f, k, n, m)
        if f["kernel"] == "k_gemv4g":
            assert m <= (1 if f32 else 4) and f["copy"] == "column-lane copy" and f["sub"] == 16, f["text"]
            assert 1 <= f["waves"] <= 16 and f["chunks"] <= 4 and f["waves"] * f["chunks"] >= k_chunks, f["text"]
        elif f["kernel"] == "k_waves_exact":
            assert 5 <= m <= 32 and f["copy"] == "16-column tile copy" and "exact weights" in f["text"] and f["waves"] == 8, f["text"]
            assert f["block_rows"] == (16 if m <= 16 else 32) and f["block_cols"] % 16 == 0, f["text"]
            nt = f["block_cols"] // 16
            assert nt in (1, 2, 3, 4, 5, 6, 8, 10) and not (gated and f["splits"] == 1 and nt % 2), f["text"]
            assert not f32 or nt <= (10 if m <= 8 else 8 if m <= 16 else 4), f["text"]      # (where their registers end)
            if f["splits"] > 1:
                assert wgs <= CUS and k_chunks // f["splits"] >= 8 and "k_splitk_reduce" in f["text"], f["text"]
        else:
            continue
        seen[f["kernel"]] += 1
    assert min(seen.values()) >= 400, seen


def test_plans_of_ranges_staged_at_once(lib):
    # k_batch_range: 5 .. 32 f32 rows, one round of workgroups that keeps at least 70 % of the CUs busy, no more chunks than a
    # workgroup's LDS holds, the partial sums within the default scratch; gated only from 17 rows on
    rng = np.random.default_rng(17)
    seen = {8: 0, 16: 0, 32: 0}
    for _ in range(6000):
        k, n = 32 * int(rng.integers(100, 900)), int(rng.integers(900, 10000))
        m, gated = int(rng.integers(4, 35)), int(rng.integers(0, 2))
        n = n // 64 * 64 + 64 if gated else n
        assert not describe(lib, k, n, m, _lib.F16, gated).startswith("k_batch_range"), (k, n, m)
        f = parse(describe(lib, k, n, m, _lib.F32, gated))
        if f["kernel"] != "k_batch_range":
            continue
        rows, k_chunks, wgs = f["block_rows"], (k // 32 + 3) // 4, workgroups(f, k, n, m)
        assert 5 <= m <= 32 and rows == (8 if m <= 8 else 16 if m <= 16 else 32) and not (gated and m <= 16), f["text"]
        assert f["copy"] == "16-column tile copy" and "+ k_splitk_reduce" in f["text"], f["text"]
        assert f["block_cols"] == (128 if m <= 16 else 256) and f["chunks"] <= (18 if m <= 16 else 9), f["text"]
        assert f["splits"] >= 2 and (f["splits"] - 1) * f["chunks"] < k_chunks <= f["splits"] * f["chunks"], f["text"]
        assert wgs <= CUS and 10 * k_chunks * ((n + 63) // 64 * 64) >= 7 * CUS * f["chunks"] * f["block_cols"], f["text"]
        assert f["splits"] * m * ((n + 63) // 64 * 64) * 4 <= 256 << 20, f["text"]
        seen[rows] += 1
    assert min(seen.values()) >= 25, seen


@pytest.mark.parametrize("k,n,m,dtype,gated", [(1152, 33728, 19, "f16", 0), (1664, 24966, 9, "f16", 0), (1152, 38272, 9, "f16", 0), (1792, 26560, 14, "f16", 0),
                                               (128, 39553, 16, "f32", 0), (17536, 5504, 25, "f32", 0), (8064, 9792, 23, "f32", 0),
                                               (7296, 10560, 27, "f32", 1), (3072, 192, 8, "f16", 1), (9216, 4352, 11, "f16", 0), (13600, 5440, 7, "f16", 1), (10848, 5696, 31, "f16", 1),
                                               (2592, 51736, 28, "f16", 0), (3840, 52422, 17, "f16", 0), (2496, 64331, 10, "f16", 0), (2592, 57664, 5, "f16", 1),
                                               (64, 84583, 6, "f32", 0), (2400, 82295, 5, "f32", 0), (2080, 104768, 6, "f32", 1), (896, 98304, 8, "f32", 0), (576, 49216, 10, "f32", 1), (1984, 59058, 12, "f32", 0),
                                               (160, 12385, 24, "f16", 0), (192, 13060, 9, "f16", 0), (160, 12160, 17, "f16", 1), (1600, 12768, 9, "f16", 0),
                                               (2784, 4611, 5, "f16", 0), (2848, 4968, 5, "f16", 0), (3392, 5083, 5, "f16", 0), (4640, 12716, 5, "f16", 0)])
def test_shapes_on_which_the_other_kernels_stay_ahead(lib, k, n, m, dtype, gated):
    # uneven chunks on many tiles, groups that leave CUs idle, gated pairs on few columns: measured 8 - 19 % slower on k_waves_exact;
    # more tiles than one round of workgroups takes: 7 - 90 %; the last eight 4 - 11 %
    f = parse(describe(lib, k, n, m, _lib.F32 if dtype == "f32" else _lib.F16, gated))
    assert f["kernel"] != "k_waves_exact", f["text"]


@pytest.mark.parametrize("k,n,m,dtype,gated", [(2592, 37888, 28, "f16", 0), (3584, 37888, 8, "f16", 1), (4096, 22016, 13, "f32", 1), (3584, 152064, 8, "f32", 0)])
def test_wide_shapes_that_one_round_of_workgroups_covers(lib, k, n, m, dtype, gated):
    # (or, with up to eight f32 rows, a K deep enough that the other forms' conversion launch costs more)
    f = parse(describe(lib, k, n, m, _lib.F32 if dtype == "f32" else _lib.F16, gated))
    assert f["kernel"] == "k_waves_exact", f["text"]


@pytest.mark.parametrize("k,n,m,gated,group_lane", [(256, 14656, 3, 1, False), (544, 28096, 1, 1, False), (544, 25088, 4, 1, False), (576, 28479, 1, 0, False),
                                                    (1088, 26584, 1, 0, False), (1152, 30080, 2, 1, False), (1600, 30792, 1, 0, False),
                                                    (256, 14656, 3, 0, True), (384, 28096, 1, 1, True), (1024, 25088, 4, 1, True), (896, 1152, 1, 0, True)])
def test_chunks_that_do_not_come_out_even_on_many_tiles(lib, k, n, m, gated, group_lane):
    # where a wave of k_gemv4g has two to four chunks: 7 - 14 % behind the other kernels of up to four rows, or ahead of them
    f = parse(describe(lib, k, n, m, gated=gated))
    assert (f["kernel"] == "k_gemv4g") == group_lane, f["text"]


@pytest.mark.parametrize("k,n,m,dtype,gated", [(832, 19155, 107, "f16", 0), (768, 12111, 210, "f32", 0), (1056, 19537, 110, "f16", 0), (1248, 17344, 120, "f16", 1),
                                               (2336, 11008, 86, "f16", 1), (5856, 5632, 73, "f16", 1), (2528, 11456, 75, "f32", 1)])
def test_prompts_that_stay_off_low_blocks_of_192_columns(lib, k, n, m, dtype, gated):
    # rows that are no whole 16-byte places, the 64-row gate on up to twelve chunks, and K-splits of a few chunks: 5 - 23 % behind
    f = parse(describe(lib, k, n, m, _lib.F32 if dtype == "f32" else _lib.F16, gated))
    assert f["kernel"] == "k_prefill" and f["block_cols"] != 192, f["text"]


@pytest.mark.parametrize("k,n,m,dtype,gated,split", [(3072, 128, 25, "f16", 0, False), (3584, 467, 24, "f16", 0, False), (2336, 1216, 5, "f32", 1, False),
                                                     (3712, 448, 11, "f32", 0, True), (4096, 128, 25, "f16", 0, True)])
def test_a_shallow_matrix_is_not_split(lib, k, n, m, dtype, gated, split):
    # (the launch of the sum kernel costs more than a few chunks per wave)
    f = parse(describe(lib, k, n, m, _lib.F32 if dtype == "f32" else _lib.F16, gated))
    assert f["kernel"] == "k_waves_exact" and (f["splits"] > 1) == split, f["text"]


@pytest.mark.parametrize("k,n,m,dtype", [(17824, 256, 24, "f32"), (16000, 256, 29, "f16"), (14976, 1344, 23, "f32"), (18176, 128, 9, "f16"),
                                         (9344, 384, 25, "f32")])
def test_few_gated_columns_of_a_deep_matrix_have_their_k_split(lib, k, n, m, dtype):
    # (unsplit, the columns alone are a handful of workgroups that walk all of K)
    dt = _lib.F32 if dtype == "f32" else _lib.F16
    gated, plain = (parse(describe(lib, k, n, m, dt, g)) for g in (1, 0))
    assert gated["splits"] > 1 and 2 * workgroups(gated, k, n, m) >= workgroups(plain, k, n, m), (gated["text"], plain["text"])


def test_describe_rejects_what_twm_gemm_rejects(lib):
    buf = ctypes.create_string_buffer(64)
    assert lib.twm_plan_describe(None, 100, 64, 1, _lib.F16, 0, buf, 64) == _lib.SHAPE_ERROR       # K % 32
    assert lib.twm_plan_describe(None, 128, 64, 1, 7, 0, buf, 64) == _lib.UNSUPPORTED_OP           # dtype
    assert lib.twm_plan_describe(None, 128, 64, 1, _lib.F16, 0, None, 0) == _lib.INVALID_HANDLE
    assert lib.twm_plan_describe(None, 128, 64, 0, _lib.F16, 0, buf, 64) == 0 and buf.value == b"nothing to launch"


# ---------------------------------------------------------------- the drop-in on the reference's arrays

def describe_m1(lib, k, n):
    buf = ctypes.create_string_buffer(256)
    rc = lib.twm_plan_describe_m1(None, k, n, buf, 256)
    assert rc == 0, lib.twm_last_error().decode()
    return buf.value.decode()


@pytest.mark.parametrize("k,n", [(3584, 4608), (3584, 3584), (3584, 37888), (18944, 3584),     # the Qwen-7B layer
                                 (13824, 5120), (28672, 8192), (8192, 10240), (8192, 57344), (3584, 152064)])
def test_drop_in_plans_of_model_shapes(lib, k, n):
    # held to what a good plan keeps, not to its text: the MFMA kernels on the arrays as they are, one launch without a
    # hand-over between workgroups, a workgroup for at least half of the CUs, and up to K = 4096 one pass per wave
    f = parse(describe_m1(lib, k, n))
    assert f["kernel"] in ("k_gemv4s", "k_gemv4") and f["copy"] == "reference arrays" and f["splits"] == 1, f["text"]
    assert workgroups(f, k, n, 1) >= CUS // 2, f["text"]
    if k <= 4096:
        assert f["kernel"] == "k_gemv4s" and f["waves"] * (64 // f["sub"]) >= (k // 32 + 3) // 4, f["text"]


def test_drop_in_plan_invariants(lib):
    for k in (32, 64, 896, 2048, 3584, 4096, 5120, 8192, 11008, 16384, 18944, 28672, 32768, 65536):
        for n in (8, 64, 100, 256, 300, 1024, 1152, 4096, 4608, 6144, 8192, 16384, 22016, 57344):
            text = describe_m1(lib, k, n)
            kernel = text.split(":")[0]
            assert kernel in ("k_gemv4s", "k_gemv4"), text
            waves = int(re.search(r"(\d+) waves", text).group(1))
            splits = int(re.search(r"(\d+) K-split", text).group(1))
            k_chunks = (k // 32 + 3) // 4
            assert 1 <= waves <= 16 and 1 <= splits <= k_chunks, (k, n, text)
            if kernel == "k_gemv4s":
                assert int(re.search(r"(\d+)-column sub-tiles", text).group(1)) in (16, 32)
            # K is cut over workgroups only on a few 16-column sub-tiles with a very deep K each, within the CU count;
            # what the no-allocation entry point's static scratch (16 Ki floats, 256 counters) is sized by
            sub_tiles = (n + 63) // 64 * 4
            if splits > 1:
                assert kernel == "k_gemv4s" and sub_tiles <= 64 and k_chunks // splits >= 64 and sub_tiles * splits <= 256, (k, n, text)
                assert splits * ((n + 63) // 64 * 64) <= 16384 and sub_tiles <= 256
    assert "2 K-splits" in describe_m1(lib, 16384, 256) and "4 K-splits" in describe_m1(lib, 32768, 64)
    assert "1 K-split;" in describe_m1(lib, 8192, 200) and "1 K-split;" in describe_m1(lib, 18944, 3584)


def test_describe_m1_edges(lib):
    buf = ctypes.create_string_buffer(64)
    assert lib.twm_plan_describe_m1(None, 100, 64, buf, 64) == _lib.SHAPE_ERROR      # K % 32, as the call itself
    assert lib.twm_plan_describe_m1(None, 128, 64, None, 0) == _lib.INVALID_HANDLE
    assert lib.twm_plan_describe_m1(None, 128, 0, buf, 64) == 0 and buf.value == b"nothing to launch"
    assert lib.twm_plan_describe_m1(None, 0, 64, buf, 64) == 0 and buf.value == b"k_fill_zero"
