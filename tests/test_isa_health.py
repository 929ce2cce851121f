"""What the compiler made of the kernels whose speed hangs on its instruction scheduling and register allocation, checked
on the CPU from the gfx950 assembly: no register spills, and no prefetch moved down to its first use.

k_batch, k_batch_range and k_prefill keep several chunks of loads in flight; their source pins every prefetch in place, but the
compiler's choices move with unrelated code (a multiply added to k_batch's store loops once moved the main loop's weight
loads of one instantiation down to their use, each followed by a wait for everything in flight: 19.2 -> 22.3 us on
3584 -> 37888 at 16 rows; the same multiply in k_prefill's store made its 128 x 256 form spill and run six times
slower).  Neither shows in a parity test."""
import os
import re
import shutil
import subprocess
import tempfile
from concurrent.futures import ThreadPoolExecutor

import pytest

from tensorwarp_amd import build

CSRC = build.CSRC
FILES = ["twm_batch.hip", "twm_prefill.hip", "twm_gemv4s.hip", "twm_gemv4g.hip", "twm_moe.hip", "twm_waves.hip", "twm_waves_exact.hip", "twm_batch_range.hip",
         "twm_splitk.hip"]
# The sub-tile kernel's looping forms with many rows (and with four f32 rows on 16 columns) run out of registers with
# two register sets live.  No planner chooses them (five rows and up run only where one pass per wave covers K; f32
# rows on a deep K take 32 columns or whole tiles); only the option knobs reach them, and the parity tests do.
FORCED_ONLY_SPILLS = ("8k_gemv4sILi32ELi16ELb0ELb0ELb0E", "8k_gemv4sILi16ELi4ELb1ELb0ELb0E", "8k_gemv4sILi16ELi8ELb0ELb0ELb0E",
                      "8k_gemv4sILi16ELi16ELb0ELb0ELb0E")


def assembly_of(src, out_dir):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    out = os.path.join(out_dir, src.replace(".hip", ".s"))
    flags = [f for f in build.FLAGS if f not in ("-fPIC", "-Wall", "-Wno-unused-function")]
    cmd = [hipcc] + flags + build.PER_FILE_FLAGS.get(src, []) + ["--offload-device-only", "-S", os.path.join(CSRC, src), "-o", out]
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0, res.stdout[-2000:]
    return open(out).read()


@pytest.fixture(scope="module")
def kernels():
    with tempfile.TemporaryDirectory() as d:
        with ThreadPoolExecutor(max_workers=len(FILES)) as pool:
            texts = list(pool.map(lambda f: assembly_of(f, d), FILES))
    found = {}
    for text in texts:
        for m in re.finditer(r"\n(_ZN3twm\w+):[^\n]*\n(.*?)s_endpgm", text, re.S):
            name, body = m.group(1), m.group(2)
            spill = re.search(r"\.set " + re.escape(name) + r"\.private_seg_size, (\d+)", text)
            found[name] = (body, int(spill.group(1)) if spill else 0)
    return found


def test_no_kernel_spills(kernels):
    assert len(kernels) > 80
    # every file's kernels are among them: one that moves to another file takes its check along
    for kernel, forms in (("k_batch", 10), ("k_prefill", 10), ("k_prefill192", 4), ("k_gemv4s", 20), ("k_gemv4g", 4), ("k_bank_gemv", 20), ("k_bank_down_axpy", 2),
                          ("k_waves", 4), ("k_waves_exact", 60), ("k_batch_range", 3), ("k_splitk_reduce", 6), ("k_splitk_reduce_swiglu", 2)):
        assert sum("%d%sI" % (len(kernel), kernel) in name for name in kernels) >= forms, kernel
    spilled = {name: scratch for name, (body, scratch) in kernels.items() if scratch and not any(f in name for f in FORCED_ONLY_SPILLS)}
    assert not spilled, spilled


def test_no_prefetch_was_moved_down_to_its_use(kernels):
    # a load of weights or activations followed at once by a wait for every load in flight
    pattern = re.compile(r"(?:global_load_dwordx[24]|global_load_lds_dwordx4) [^\n]*\n\s*s_waitcnt vmcnt\(0\)")
    checked = 0
    for name, (body, _) in kernels.items():
        if "7k_batchI" in name or "9k_prefillILi8ELi4ELb0E" in name or "9k_prefillILi4E" in name or "12k_prefill192I" in name or "13k_batch_rangeI" in name:
            checked += 1
            assert not pattern.search(body), name
    assert checked >= 40


def test_counted_waits_match_the_loads_of_a_chunk(kernels):
    # k_prefill's forms with three or four chunks in flight wait for "all but the newest D - 2 chunks' loads" by number: every
    # chunk of the main loop has to issue that number of loads between two barriers, the start D chunks' worth
    checked = 0
    for name, (body, _) in kernels.items():
        form = re.search(r"9k_prefillILi(\d+)ELi(\d+)ELb0ELi(\d)E", name) or re.search(r"12k_prefill192ILi(\d+)E()()", name)
        if not form:
            continue
        mt, ntw, depth = (int(x) if x else 3 for x in form.groups())
        per_chunk = mt + 2 * ntw
        parts = re.split(r"s_waitcnt vmcnt\((\d+)\) lgkmcnt\(0\)\n\s*s_barrier", body)
        loads = [len(re.findall(r"\bglobal_load_(?:lds_)?dword", p)) for p in parts[0::2]]
        waits = [int(x) for x in parts[1::2]]
        assert waits[:depth + 1] == [(depth - 1) * per_chunk] + [(depth - 2) * per_chunk] * depth, (name, waits)
        assert loads[:depth + 1] == [depth * per_chunk, 0] + [per_chunk] * (depth - 1), (name, loads)
        checked += 1
    assert checked == 15


def test_unsplit_sub_tile_launches_hand_nothing_over(kernels):
    # k_gemv4s, its upfront form and the traced twin that stands for both: without a K-split no arrival counter is touched (there
    # may be fewer of them than sub-tiles) and no partial sum parked
    forms = [(name, body) for name, (body, _) in kernels.items() if re.search(r"\d+k_gemv4s(_upfront|_traced)?I", name)]
    unsplit = [(name, body) for name, body in forms if re.search(r"Lb0EEEvPKc", name)]
    assert len(unsplit) >= 20 and sum("k_gemv4s_traced" in name for name, _ in unsplit) == 4
    for name, body in unsplit:
        assert "global_atomic" not in body, name
    assert all("global_atomic" in body for name, body in forms if re.search(r"Lb1EEEvPKc", name))


def test_plain_stores_of_192_column_blocks_carry_no_other_store(kernels):
    # the search for a segment and the gate are instantiations of their own: compiled into the plain one they cost it 10 - 20 %
    # on a shallow K, also where they are skipped
    forms = {}
    for name, (body, _) in kernels.items():
        m = re.search(r"(9k_prefillILi8ELi3ELb\dELi\d|12k_prefill192ILi\d)ELNS_12PrefillStoreE(\d)E", name)
        if m:
            forms.setdefault(m.group(1), {})[int(m.group(2))] = body
    assert len(forms) == 4
    for which, by_store in forms.items():
        plain, segments, gate = (by_store[i] for i in range(3))
        assert "v_exp_f32" in gate and "v_exp_f32" not in plain + segments, which
        assert len(plain) < len(segments), which


def test_the_gated_sum_has_both_places_in_flight(kernels):
    # the gate's and the up projection's first partial sums are loaded before either is waited for, whatever the splits
    forms = [(name, body) for name, (body, _) in kernels.items() if "k_splitk_reduce_swiglu" in name]
    assert len(forms) == 2
    for name, body in forms:
        first, second = [m.start() for m in re.finditer(r"global_load_dwordx4", body)][:2]
        assert not re.search(r"vmcnt|branch|\n\.LBB", body[first:second]), name
