"""The rule that sends a grouped GEMM to the few-rows kernels
(``placemoe_amd/csrc/few_rows_rule.h``), compiled with the host compiler:
calls that measured slower on them than on the 256-row kernels stay off, calls
that gain stay on, and no call goes past the lines."""

import itertools
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from tests import test_gpu_few_rows, test_gpu_gemm_bounds

ROOT = Path(__file__).resolve().parents[1]
KINDS = ("fc1", "fc2", "fc1_dgrad", "fc2_dgrad")


@pytest.fixture(scope="module")
def tiling(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = tmp_path_factory.mktemp("rule") / "few_rows_rule"
    subprocess.run([cxx, "-O2", "-std=c++17", f"-I{ROOT / 'placemoe_amd' / 'csrc'}",
                    str(ROOT / "tests" / "few_rows_rule_main.cpp"), "-o", str(exe)], check=True)

    def ask(calls):
        """calls: (kind, rows, copies, H, I) -> tile heights, on 256 CUs."""
        lines = []
        for kind, rows, copies, H, I in calls:
            N, K = {"fc1": (2 * I, H), "fc2": (H, I), "fc1_dgrad": (H, 2 * I), "fc2_dgrad": (I, H)}[kind]
            lines.append(f"{KINDS.index(kind)} {rows} {copies} {N} {K} 256")
        out = subprocess.run([str(exe)], input="\n".join(lines), check=True, capture_output=True, text=True).stdout
        return [int(x) for x in out.split()]

    return ask


# (kind, rows per copy, copies, H, I): us few-rows / 256-row
SLOWER = [
    ("fc1", 72, 16, 7168, 2048),  # 254 / 213, log-normal counts
    ("fc1", 120, 16, 7168, 2048),  # 261 / 218, even
    ("fc1", 96, 32, 2048, 768),  # 85 / 66, Zipf(1.0)
    ("fc1", 120, 16, 4096, 1536),  # 143 / 117, Zipf(1.0)
    ("fc1", 56, 128, 1280, 768),  # 145 / 134, log-normal
    ("fc1", 120, 128, 1280, 768),  # 158 / 138, even
    ("fc2", 48, 160, 2048, 768),  # 118 / 108, log-normal
    ("fc2", 48, 48, 5120, 1536),  # 176 / 153, log-normal
    ("fc1_dgrad", 40, 16, 4096, 1536),  # 107 / 77, Zipf(1.0)
    ("fc1_dgrad", 24, 32, 2048, 768),  # 62 / 47, Zipf(1.0)
    ("fc2_dgrad", 24, 32, 7168, 2048),  # 253 / 197, Zipf(1.0)
    ("fc2_dgrad", 120, 160, 2048, 768),  # 184 / 147, even
    ("fc2_dgrad", 96, 128, 2048, 768),  # 156 / 142, Zipf(1.0)
    ("fc2_dgrad", 120, 40, 2048, 1408),  # 103 / 73, even
]
FASTER = [
    ("fc1", 5, 160, 2048, 768, 64),  # 177 / 256
    ("fc1", 12, 16, 7168, 2048, 64),  # 163 / 211
    ("fc1", 96, 128, 2048, 768, 128),  # 213 / 228
    ("fc2", 5, 160, 2048, 768, 64),  # 91 / 105
    ("fc2", 48, 12, 1024, 2816, 64),  # 31 / 63
    ("fc1_dgrad", 5, 160, 2048, 768, 128),  # 170 / 182
    ("fc1_dgrad", 40, 12, 1024, 2816, 64),  # 53 / 111
    ("fc2_dgrad", 25, 160, 2048, 768, 64),  # 113 / 139
    ("fc2_dgrad", 12, 16, 7168, 2048, 64),  # 90 / 177
    ("fc2_dgrad", 64, 128, 2048, 768, 128),  # 121 / 137
]


def test_calls_that_measured_slower_stay_on_the_256_row_kernels(tiling):
    calls = [(k, n * g, g, H, I) for k, n, g, H, I in SLOWER]
    assert dict(zip(calls, tiling(calls))) == dict.fromkeys(calls, 0)


def test_calls_that_gain_go_to_the_few_rows_kernels(tiling):
    calls = [(k, n * g, g, H, I) for k, n, g, H, I, _ in FASTER]
    assert tiling(calls) == [want for *_, want in FASTER]


def test_no_call_goes_past_the_lines(tiling):
    most64 = {"fc1": 56, "fc2": 48, "fc1_dgrad": 40, "fc2_dgrad": 56}
    most128 = {"fc1": 120, "fc2": 0, "fc1_dgrad": 40, "fc2_dgrad": 120}
    layers = [(1, 64, 8), (3, 1096, 776), (16, 7168, 2048), (128, 2048, 768), (1024, 128, 72), (160, 1024, 704)]
    calls = [(k, max(1, rows * g + d), g, H, I) for k, rows, (g, H, I), d in
             itertools.product(KINDS, (0, 1, 8, 40, 48, 56, 57, 120, 121, 500), layers, (-1, 0, 1))]
    for (kind, rows, g, H, I), bm in zip(calls, tiling(calls)):
        assert bm in (0, 64, 128)
        assert bm != 64 or rows <= most64[kind] * g
        assert bm != 128 or rows <= most128[kind] * g
        if rows <= 8 * g:  # one tile a copy on any kernel: always
            assert bm != 0, (kind, rows, g, H, I)


def _wgrad_line():
    src = (ROOT / "placemoe_amd" / "csrc" / "grouped_gemm.hip").read_text()
    return int(re.search(r"constexpr int64_t kFewRowsWgrad = (\d+);", src).group(1))


def test_gpu_cases_reach_every_few_rows_kernel(tiling):
    cases = [(int(sum(c)), len(c), H, I) for c, H, I in test_gpu_few_rows.CASES.values() if len(c) <= 1024]
    reached = {kind: set(tiling([(kind, *c) for c in cases])) for kind in KINDS}
    assert reached == {"fc1": {0, 64, 128}, "fc2": {0, 64}, "fc1_dgrad": {0, 64, 128}, "fc2_dgrad": {0, 64, 128}}
    line = _wgrad_line()
    assert all(sum(c) <= line * len(c) for c, _, _ in test_gpu_few_rows.WGRAD_CASES)
    assert all(sum(c) > line * len(c) for c, _, _ in test_gpu_few_rows.WGRAD_PAST_THE_LINE)


def test_gpu_cases_of_the_256_row_kernels_stay_on_them(tiling):
    for seed, cases in ((0, test_gpu_gemm_bounds.TILE_TABLE_CASES), (7, test_gpu_gemm_bounds.EIGHT_WAVE_CASES)):
        for G, A, H, I in cases:
            rows = int(test_gpu_gemm_bounds._copies(G, A, seed=G + seed)[-1])
            assert tiling([(kind, rows, G, H, I) for kind in KINDS]) == [0] * 4, (G, A)
            assert rows > _wgrad_line() * G, (G, A)
    assert max(G for G, *_ in test_gpu_gemm_bounds.TILE_TABLE_CASES) > 512  # the plain weight-gradient order
    assert max(G for G, *_ in test_gpu_gemm_bounds.EIGHT_WAVE_CASES) > 512
