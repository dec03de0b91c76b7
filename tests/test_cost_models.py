"""The cost models that choose between the GEMM kernels (csrc/gemm_model.h) cut decode attention into key ranges (csrc/attention_model.h) and choose stream_kernel
(csrc/stream_model.h) are host code: compiled into a small program and asked here."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "tensor_parallel_amd" / "csrc"


def ask(tmp_path, body, header="gemm_model.h"):
    """The program's output for a body that prints rows of numbers, as lists of floats."""
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    (tmp_path / "ask.cpp").write_text('#include <stdio.h>\n#include <initializer_list>\n#include "' + header + '"\nusing namespace tpamd;\nint main() {\n' + body + "\n}\n")
    subprocess.run(["g++", "-std=c++17", "-I", str(CSRC), str(tmp_path / "ask.cpp"), "-o", str(tmp_path / "ask")], check=True)
    out = subprocess.run([str(tmp_path / "ask")], check=True, capture_output=True, text=True, timeout=60).stdout
    return [[float(v) for v in line.split()] for line in out.splitlines()]


def test_no_mid_tile_is_predicted_faster_than_its_weights_stream(tmp_path):
    """Up to 128 rows of wide matrices: every tiling is floored at the same 5 TB/s, so a tie decides there, and not which model lacks the floor."""
    rows = ask(tmp_path, """
    const long long shapes[][2] = {{64128, 4096}, {32000, 4096}, {28672, 8192}, {28672, 4096}, {4096, 5504}, {260, 64}};
    for (auto &s : shapes) for (int swiglu = 0; swiglu < 2; ++swiglu) for (int m : {17, 40, 64, 100, 128}) {
        int tmx = 0, tnx = 0;
        printf("%d %lld %lld %d %.9g\\n", m, s[0], s[1], swiglu, estimate_mid(m, s[0], (int)(s[1] / 64), 256, swiglu != 0, &tmx, &tnx));
    }""")
    assert len(rows) == 6 * 2 * 5
    for m, n, k, swiglu, us in rows:
        assert us * 5e6 >= n * k * (4 if swiglu else 2) * (1 - 1e-6), (m, n, k, swiglu, us)


def test_a_forced_split_count_is_one_that_a_launch_takes(tmp_path):
    """TPAMD_W8_TILE_SPLITS is taken as it stands in the environment: 0 was a division by zero in the launch."""
    rows = ask(tmp_path, """
    for (int wanted : {-7, 0, 1, 3, 16, 17, 1 << 30}) for (int kt : {2, 5, 64}) printf("%d %d %d\\n", wanted, kt, forced_splits(wanted, kt, 16));""")
    assert [r[2] for r in rows] == [1, 1, 1, 1, 1, 1, 1, 1, 1, 2, 3, 3, 2, 5, 16, 2, 5, 16, 2, 5, 16]


def test_slabs_are_taken_without_scratch_memory_where_they_measured_faster(tmp_path):
    """Rows, columns, K, outliers, and which of the two was faster by 15 % or more on a stream without scratch memory."""
    cases = [(65, 4096, 5504, 0, 1), (65, 4096, 5504, 1, 1), (129, 4096, 5504, 0, 1), (257, 4096, 5504, 0, 0), (400, 4096, 5504, 1, 0), (65, 8192, 4096, 0, 1),
             (200, 8192, 4096, 1, 0), (65, 28672, 4096, 0, 0), (65, 28672, 4096, 1, 0), (256, 1024, 16384, 1, 1), (400, 1024, 16384, 0, 0), (100, 16384, 8192, 0, 0)]
    rows = ask(tmp_path, "".join(f'printf("%d\\n", w8_slabs_without_scratch({m}, {n}, {k}, {o}) ? 1 : 0);\n' for m, n, k, o, _ in cases))
    assert [r[0] for r in rows] == [c[4] for c in cases]


def test_sums_of_two_ranks_stay_in_two_launches_where_those_measured_faster(tmp_path):
    """Rows, columns and K, and whether one launch of both ranks took longer than two on 256 CUs (by 4 % or more; the others took at most 0.98 of two)."""
    cases = [(2, 1024, 8192, 1), (2, 2048, 16384, 1), (2, 2048, 5632, 0), (2, 2304, 8192, 0), (2, 5568, 4096, 1), (2, 4864, 4096, 1), (2, 5120, 4608, 0), (3, 5120, 2048, 1), (3, 10240, 2048, 1),
             (3, 4096, 2048, 0), (8, 5568, 4096, 1), (16, 6000, 8192, 1), (8, 5120, 8192, 0), (8, 7168, 4096, 1), (8, 6000, 3584, 0), (1, 4096, 8192, 1), (1, 4096, 4096, 0),
             (4, 14336, 2048, 1), (12, 9216, 1024, 1), (2, 9216, 2048, 0), (8, 12288, 4096, 0), (16, 20480, 6144, 1), (16, 32768, 4096, 1), (16, 16384, 2048, 0), (24, 18432, 4096, 1),
             (24, 10240, 8192, 1), (64, 9216, 4096, 1), (128, 9216, 8192, 1), (24, 20480, 1024, 1), (40, 12288, 2048, 0), (64, 16384, 1024, 0), (40, 8192, 14336, 0), (512, 4096, 5504, 0)]
    rows = ask(tmp_path, "".join(f'printf("%d\\n", sum_in_two_launches({m}, {n}, {k}, 256) ? 1 : 0);\n' for m, n, k, _ in cases))
    assert [r[0] for r in rows] == [c[3] for c in cases]


def test_key_ranges_of_a_decode_step_are_counts_that_measured_fast(tmp_path):
    """Heads, keys, head_dim, and the least and largest count of ranges that measured within 8 % of the best one on 256 CUs (every count between them did)."""
    cases = [(1, 131072, 128, 56, 64), (2, 131072, 64, 56, 64), (16, 131072, 128, 10, 16), (32, 32768, 128, 5, 8), (32, 20000, 64, 7, 8), (96, 2675, 128, 2, 2), (48, 6133, 64, 4, 5),
             (64, 8192, 64, 3, 4), (256, 4096, 128, 1, 1), (256, 500, 128, 1, 1), (128, 2048, 64, 1, 3), (32, 500, 64, 1, 1), (1, 64, 128, 1, 1), (4, 1000, 64, 4, 8)]
    rows = ask(tmp_path, "".join(f'printf("%d\\n", decode_splits({heads}, {keys}, {D}, 256));\n' for heads, keys, D, _, _ in cases), "attention_model.h")
    for case, (count,) in zip(cases, rows):
        assert case[3] <= count <= case[4], (case, count)


def test_stream_kernel_is_left_to_the_launches_that_it_measured_faster_on(tmp_path):
    """Ranks in the launch (sum: 0), gated pair, rows, columns, K, and whether stream_kernel takes it: differences of 7 % or more on 256 CUs, either way."""
    cases = [(2, 1, 64, 6144, 1408, 0), (1, 1, 40, 2048, 14336, 0), (1, 1, 28, 2048, 2944, 0), (1, 1, 24, 2048, 1408, 1), (2, 1, 40, 8192, 5120, 0), (2, 1, 36, 8192, 8192, 1),
             (1, 1, 36, 11008, 1024, 0), (2, 1, 24, 5504, 4096, 1), (1, 1, 40, 5504, 4096, 1), (2, 1, 28, 1024, 4416, 0), (1, 1, 36, 2048, 2048, 1),
             (1, 0, 3, 452, 8192, 0), (1, 0, 3, 1024, 4096, 0), (1, 0, 3, 11008, 2048, 0), (1, 0, 3, 5200, 1024, 1), (2, 0, 8, 4096, 1024, 0), (1, 0, 12, 2048, 8128, 0),
             (1, 0, 12, 4608, 14336, 1), (1, 0, 16, 4096, 2048, 1), (1, 0, 28, 3072, 5120, 0), (1, 0, 28, 5120, 2752, 1), (2, 0, 32, 16000, 2688, 0), (2, 0, 28, 16000, 4096, 1),
             (2, 0, 24, 6144, 4096, 1), (2, 0, 36, 2048, 1984, 1), (2, 0, 56, 1024, 2048, 0),
             (0, 0, 64, 16000, 1408, 0), (0, 0, 36, 16000, 4096, 1), (0, 0, 8, 4096, 5504, 1), (0, 0, 24, 4096, 2048, 1), (0, 0, 64, 4096, 5504, 0)]
    rows = ask(tmp_path, "".join(f'printf("%d\\n", stream_measured_faster({m}, {n}, {k}, {ranks or 2}, {"true" if pair else "false"}, {"false" if ranks else "true"}, 256) ? 1 : 0);\n'
                                 for ranks, pair, m, n, k, _ in cases), "stream_model.h")
    assert [(c[:5], r[0]) for c, r in zip(cases, rows)] == [(c[:5], c[5]) for c in cases]


def test_tiles_are_chosen_that_measured_fast(tmp_path):
    """Ranks, gated pair, rows, columns, K, and what measured within 5 % of the best on 256 CUs (a gemm_mid_kernel tile as 1000 * rows + columns, 256 or 128): shapes on which the models were 10 to 28 % off,
    and others of every kind."""
    cases = [(1, 1, 641, 2200, 5120, {128}), (1, 1, 1507, 1120, 5376, {128}), (2, 1, 727, 1024, 5184, {128}), (1, 1, 222, 7800, 5504, {128}), (2, 1, 776, 1596, 5120, {128192}),
             (2, 1, 5049, 3072, 11008, {256}), (2, 1, 3684, 4096, 8192, {256}), (1, 1, 384, 5120, 5120, {128}), (2, 0, 5429, 5504, 8192, {256}),
             (2, 1, 512, 5504, 4096, {256192}), (2, 0, 645, 16000, 4096, {224192}), (1, 0, 2103, 4096, 5504, {192192})]
    rows = ask(tmp_path, "TileChoice c;\n" + "".join(
        f'c = choose_tile({m}, {n}, {k // 64}, 256, {"true" if pair else "false"}, {ranks}); printf("%d\\n", c.tmx ? 32000 * c.tmx + 32 * c.tnx : c.big ? 256 : 128);\n' for ranks, pair, m, n, k, _ in cases))
    assert [(c[:5], int(r[0])) for c, r in zip(cases, rows) if int(r[0]) not in c[5]] == []


def test_sums_on_128_tiles_are_left_where_256_tiles_of_each_rank_measured_faster(tmp_path):
    """Rows, columns, K, and whether one launch of both ranks was the faster one."""
    cases = [(938, 4096, 14336, 0), (1464, 2416, 13440, 0), (1048, 1800, 4096, 0), (512, 4096, 5504, 1), (645, 4096, 5504, 0), (128, 4096, 4096, 1)]
    rows = ask(tmp_path, "".join(f'printf("%d\\n", sum_predicted_faster({m}, {n}, {k // 64}, 256) ? 1 : 0);\n' for m, n, k, _ in cases))
    assert [r[0] for r in rows] == [c[3] for c in cases]
