"""The rule for the fp32 layers that run on the bf16 matrix cores
(plan_f32_split in ml-edsl_amd/csrc/plan_f32.cpp), on the CPU."""
from __future__ import annotations

import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "ml-edsl_amd", "csrc")

DRIVER = r"""
#include <cstdio>
#include "plan_f32.hpp"
int main() {
  long long M, N, K, ldc;
  int aligned, forced;
  while (scanf("%lld %lld %lld %d %d %lld", &M, &N, &K, &aligned, &forced, &ldc) == 6) {
    const edsl::F32TileQuery q{M, N, K, K, N, aligned != 0, 256, forced, ldc};
    const int cfg = edsl::plan_f32_tile(q), t = edsl::plan_f32_split(q, cfg);
    printf("%s %lld\n", edsl::f32_split_name(t), (long long)edsl::f32_split_grid(t, M, N));
  }
}
"""


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan_split")
    src, exe = d / "driver.cpp", d / "driver"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{CSRC}", "-o", str(exe), str(src),
                    os.path.join(CSRC, "plan_f32.cpp")], check=True)
    return str(exe)


# (M, K, N), aligned, forced configuration, ldc (0: N), split tile
CASES = [
    ((4096, 4096, 4096), 1, -1, 0, "256x128x16"), ((4096, 256, 4096), 1, -1, 0, "128x128x16"),
    ((4001, 4001, 4001), 0, -1, 0, "256x128x16"), ((4000, 1024, 4000), 1, -1, 0, "256x128x16"),
    ((2500, 2500, 2500), 1, -1, 0, "256x128x16"), ((2048, 4096, 4096), 1, -1, 0, "256x128x16"),
    ((2048, 2048, 2048), 1, -1, 0, "128x128x32_w8"), ((2001, 2001, 2001), 0, -1, 0, "128x128x32_w8"),
    ((10000, 500, 1000), 1, -1, 0, "128x128x16"), ((3333, 3333, 3333), 0, -1, 0, "128x128x16"),
    # K split over waves in even rounds
    ((1024, 1024, 1024), 1, -1, 0, "none"), ((3072, 3072, 3072), 1, -1, 0, "none"),
    ((1500, 1500, 1500), 1, -1, 0, "none"), ((1000, 1000, 1000), 1, -1, 0, "none"),
    # short K, small M, a forced configuration, rows of C past 31-bit offsets
    ((4096, 255, 4096), 1, -1, 0, "none"), ((64, 4096, 8192), 1, -1, 0, "none"),
    ((4096, 4096, 4096), 1, 16, 0, "none"), ((4096, 4096, 4096), 1, -1, 1 << 21, "none"),
    ((4096, 4096, 4096), 1, -1, (1 << 21) - 1, "256x128x16"),
]


def test_split_rule(driver):
    text = "".join(f"{M} {N} {K} {al} {f} {ldc or N}\n" for (M, K, N), al, f, ldc, _ in CASES)
    out = subprocess.run([driver], input=text, capture_output=True, text=True, check=True).stdout.split("\n")
    got = [line.split()[0] for line in out if line]
    assert got == [c[-1] for c in CASES], [(c, g) for c, g in zip(CASES, got) if c[-1] != g]
