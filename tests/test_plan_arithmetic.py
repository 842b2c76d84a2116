"""Host check of the decode work-placement arithmetic (apertura_amd/csrc/esda_plan.h:
visibility, the prefix table, balanced shares and their segment walk, partial slots,
the merge's split owners, grid splits) -- the functions the attend and merge kernels
call -- over 3,000 random batches including 256-sequence batches, fewer rows than
workgroups, and 256 x 16 kv heads x 16,384 workgroups.  tests/plan_check.cpp is built
with g++; a variant with the batch-256 prefix-table bug planted must fail.  And the plans of
esda_prefill (apertura_amd/csrc/esda_prefill_plan.h, through tests/prefill_plan_check.cpp):
the kernel forms and key splits that the GPU tests' shapes rely on."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "plan_check.cpp")
INC = os.path.join(ROOT, "apertura_amd", "csrc")


def _build(tmp_path, *defines, src=SRC):
    cxx = os.environ.get("CXX", "g++")
    if not shutil.which(cxx):
        pytest.skip(f"{cxx} not found")
    exe = tmp_path / ("plan_check" + "".join(d.lower() for d in defines))
    cmd = [cxx, "-std=c++17", "-O2", "-Wall", "-Wextra", "-Werror", "-I", INC, "-I", os.path.join(ROOT, "include"),
           src, "-o", str(exe)]
    cmd += [f"-D{d}" for d in defines]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


def test_plan_arithmetic_over_random_batches(tmp_path):
    exe = _build(tmp_path)
    r = subprocess.run([str(exe), "3000"], capture_output=True, text=True, timeout=600)
    print(r.stdout[-2000:])
    assert r.returncode == 0 and r.stdout.strip().endswith("3000 batches, 0 failures"), r.stdout[-2000:]


def test_planted_prefix_table_bug_is_caught(tmp_path):
    exe = _build(tmp_path, "PLANT_TABLE_BUG")
    r = subprocess.run([str(exe), "64"], capture_output=True, text=True, timeout=600)
    assert r.returncode != 0 and "table[256] never written" in r.stdout, r.stdout[-2000:]


def _prefill_bytes(Hq, Hkv, D, Sq, Sk, q_pos0, k_pos0=0, window=0, split_keys=0):
    from apertura_amd.prefill import PrefillStep, prefill_workspace_bytes
    return prefill_workspace_bytes(PrefillStep(Hq, Hkv, D, Sq, Sk, q_pos0, k_pos0, window, split_keys=split_keys,
                                               kv_head_stride=Sk * D))


@pytest.mark.parametrize("Hq,Hkv,D,Sq,past,splits", [
    (32, 4, 512, 333, 5600, 3),    # 84 tiles of 4 heads: 252 workgroups, not 336
    (32, 4, 512, 200, 8056, 4),    # 52 tiles of 4 heads: 208
    (32, 4, 512, 512, 15872, 2),   # 128 tiles: 256
    (32, 4, 512, 770, 0, 1),       # 49 fresh tiles of 4 heads: unsplit
    (32, 4, 512, 4096, 0, 1),      # four rounds of tiles
    (8, 4, 256, 17, 10, 1),        # one stage
])
def test_prefill_plan_fills_whole_rounds(Hq, Hkv, D, Sq, past, splits):
    """Automatic key splits by the workspace they ask for (D fp32 and (m, l) per row and split)."""
    n = _prefill_bytes(Hq, Hkv, D, Sq, past + Sq, past)
    assert n == (0 if splits == 1 else splits * Sq * Hq * (D * 4 + 8) + 256)


def test_prefill_plan_of_extreme_forced_splits_is_quick():
    """Forced splits are planned without walking them: the largest accepted count, a count
    past the limit (refused), and one split longer than the keys."""
    import time

    from apertura_amd import EsdaError
    t0 = time.perf_counter()
    n = 65535 * 32
    assert _prefill_bytes(16, 8, 256, 64, n, n - 64, split_keys=32) == 65535 * 64 * 16 * (256 * 4 + 8) + 256
    with pytest.raises(EsdaError):
        _prefill_bytes(16, 8, 256, 64, 2 ** 30, 2 ** 30 - 64, split_keys=32)
    assert _prefill_bytes(16, 8, 256, 2 ** 20, 2 ** 20, 0, split_keys=2 ** 30) == 0
    assert time.perf_counter() - t0 < 2.0


def _plans(tmp_path, descs, gaps=False):
    """The plans of (Hq, Hkv, D, Sq, past, window, split_keys), the chunk's own keys and its past (on
    sliding layers the last window of it): (waves, rows per tile, splits) each, with gaps also whether
    the merge reads live splits only, or the refusal."""
    exe = _build(tmp_path, src=os.path.join(ROOT, "tests", "prefill_plan_check.cpp"))
    lines = []
    for Hq, Hkv, D, Sq, past, window, split in descs:
        Sk = min(past + Sq, window + Sq) if window else past + Sq
        lines.append(f"{Hq} {Hkv} {D} {Sq} {Sk} {past} {past + Sq - Sk} {window} {split}")
    r = subprocess.run([str(exe)], input="\n".join(lines) + "\n", capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    out = []
    for line in r.stdout.splitlines():
        if line.startswith("refused"):
            out.append(line)
        else:
            nw, qt, tiles, splits, kps, live_only, nbytes = map(int, line.split())
            out.append((nw, qt, splits, live_only) if gaps else (nw, qt, splits))
    return out


def test_prefill_forms_the_peak_tests_rely_on(tmp_path):
    from test_prefill_gpu import PEAKS_512
    plans = _plans(tmp_path, [(32, 4, 512, Sq, past, 0, 0) for Sq, past, _, _ in PEAKS_512])
    assert plans == [form for _, _, form, _ in PEAKS_512]


def test_prefill_forms_the_planned_tests_rely_on(tmp_path):
    """Forms and splits at the edges of the choice; among them chunks that the dispatch order
    decides (round-robin over the XCDs and their engines, whatever the workgroups' lengths)."""
    from test_prefill_gpu import PLANNED
    plans = _plans(tmp_path, [(Hq, Hkv, D, Sq, past, window, 0) for D, Hq, Hkv, Sq, past, window, _ in PLANNED])
    assert plans == [form for *_, form in PLANNED]
    # unsplit, though an even spread of two splits' work would end first
    assert _plans(tmp_path, [(32, 8, 128, 2043, 0, 0, 0), (16, 16, 512, 1364, 91, 0, 0)]) == [(8, 256, 1), (4, 64, 1)]


def test_forced_splits_of_many_workgroups_take_tall_tiles(tmp_path):
    """Forced splits past three workgroups a CU: every piece loads its queries and fills its pipeline
    anew, so the tall tiles, which have fewer pieces, are the cheap ones."""
    chunks = [(32, 16, 256, 3028, 759, 0, 1024), (16, 8, 256, 2005, 0, 0, 512), (8, 4, 256, 3163, 954, 0, 256),
              (8, 1, 256, 2091, 36, 1024, 128), (16, 2, 512, 969, 0, 0, 128)]
    assert _plans(tmp_path, chunks) == [(8, 256, 4), (8, 256, 4), (8, 256, 17), (8, 256, 9), (8, 128, 8)]


def test_merges_that_read_live_splits_only(tmp_path):
    """Where a large split plan leaves a quarter of the tiles without a key in the last split: fresh
    prompts, not small ones, nor a past or a window that fills all splits but the last."""
    from test_prefill_gpu import GAPS
    plans = _plans(tmp_path, [(Hq, Hkv, D, Sq, past, window, split) for D, Hq, Hkv, Sq, past, window, split, _ in GAPS], gaps=True)
    assert [(s, g) for _, _, s, g in plans] == [(s, 1) for *_, s in GAPS]
    same = [(32, 4, 512, 512, 8192, 0, 1088), (16, 8, 256, 256, 0, 0, 128), (16, 8, 256, 2048, 9000, 1024, 512)]
    assert [p[2:] for p in _plans(tmp_path, same, gaps=True)] == [(8, 0), (2, 0), (3, 0)]


def test_plans_follow_the_description_of_each_call(tmp_path):
    """The library keeps the calling thread's last plan: descriptions that differ in one field, taken
    in turn and from two threads at once, get their own workspace sizes, refused ones none."""
    import threading

    from apertura_amd import EsdaError
    base = dict(Hq=32, Hkv=4, D=512, Sq=200, Sk=8256, q_pos0=8056)
    descs = [base, dict(base, Sq=199, q_pos0=8057), dict(base, split_keys=512), dict(base, window=64),
             dict(base, D=256)]
    exe = _build(tmp_path, src=os.path.join(ROOT, "tests", "prefill_plan_check.cpp"))
    text = "".join(f"{d['Hq']} {d['Hkv']} {d['D']} {d['Sq']} {d['Sk']} {d['q_pos0']} 0 {d.get('window', 0)} "
                   f"{d.get('split_keys', 0)}\n" for d in descs)
    r = subprocess.run([str(exe)], input=text, capture_output=True, text=True, timeout=60)
    want = [int(line.split()[-1]) for line in r.stdout.splitlines()]
    assert len(set(want)) == len(want)
    wrong = []

    def walk(order):
        for i in order:
            if _prefill_bytes(**descs[i]) != want[i] or _prefill_bytes(**descs[i]) != want[i]:
                wrong.append(i)
            with pytest.raises(EsdaError):
                _prefill_bytes(**dict(descs[i], split_keys=33))
            if _prefill_bytes(**descs[i]) != want[i]:
                wrong.append(i)

    threads = [threading.Thread(target=walk, args=(list(range(len(descs)))[::s] * 50,)) for s in (1, -1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@pytest.mark.parametrize("name,merge,longest", [
    ("balanced_merge_4_pairs", "merge_kernel<16>", 117),
    ("balanced_merge_40_pairs", "merge_kernel<4>", 36),
    ("balanced_merge_42_pairs", "merge_kernel<4>", 13),
    ("balanced_merge_44_pairs", "merge_rows_kernel", 13),
    ("balanced_merge_loop_4", "merge_kernel<4>", 252),
    ("balanced_merge_loop_16", "merge_kernel<16>", 511),
])
def test_balanced_merges_the_edge_cases_rely_on(name, merge, longest):
    """The merge and the most partials of a pair for the GPU tests' balanced cases: the plan's shares
    from the workspace it asks for, the owners by esda_plan.h's rule, the merge by the launch's."""
    from apertura_amd.decode import DecodeStep, workspace_bytes
    from test_decode_gpu import EDGE
    c = next(c for c in EDGE if c["name"] == name)
    B, Hkv, D, cap = c["B"], c["Hkv"], c["D"], c["cap"]
    G = c["Hq"] // Hkv
    n = workspace_bytes(DecodeStep(batch=B, num_q_heads=c["Hq"], num_kv_heads=Hkv, head_dim=D, cap=cap,
                                   kv_shared=c.get("shared", False), scale=1.0))
    up = lambda x: (x + 255) // 256 * 256
    W = next(w for w in range(1, 20000) if 256 + up((B + 1) * 8) + up((B * Hkv + w) * G * 8) + (B * Hkv + w) * G * D * 4 == n)
    pairs, rows = B * Hkv, [p + 1 for p in c["pos"]]
    total = sum(rows) * Hkv
    Wr, first, most = min(W, total), 0, 0
    for r in rows:
        for _ in range(Hkv):
            owner = lambda x: ((x + 1) * Wr - 1) // total
            most = max(most, owner(first + r - 1) - owner(first) + 1)
            first += r
    kernel = "merge_rows_kernel" if W < 6 * pairs else "merge_kernel<4>" if 2 * W <= 64 * pairs else "merge_kernel<16>"
    assert (kernel, most) == (merge, longest)
    if "loop" in name:
        assert most > (64 if kernel == "merge_kernel<4>" else 256)
