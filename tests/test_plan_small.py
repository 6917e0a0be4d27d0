"""The rule for the 16x16 small-output tiles (plan_f32_small in
ml-edsl_amd/csrc/plan_f32.cpp), on the CPU."""
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
  long long M, N, K;
  int aligned, stream, forced;
  while (scanf("%lld %lld %lld %d %d %d", &M, &N, &K, &aligned, &stream, &forced) == 6)
    printf("%d\n", edsl::plan_f32_small(edsl::F32TileQuery{M, N, K, K, N, aligned != 0, 256, forced}, stream != 0));
}
"""


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan_small")
    src, exe = d / "driver.cpp", d / "driver"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{CSRC}", "-o", str(exe), str(src),
                    os.path.join(CSRC, "plan_f32.cpp")], check=True)
    return str(exe)


# (M, K, N), aligned, streamed rows, forced configuration, waves
CASES = [
    ((16, 512, 512), 1, 1, -1, 8), ((64, 256, 64), 1, 1, -1, 4), ((16, 1024, 8192), 1, 1, -1, 8),
    ((16, 1024, 8208), 1, 1, -1, 0),   # more than two tiles per CU
    ((16, 1025, 512), 1, 1, -1, 0), ((16, 2048, 1024), 1, 1, -1, 0),
    ((64, 448, 256), 1, 0, -1, 4), ((64, 449, 256), 0, 0, -1, 8), ((256, 1024, 256), 1, 0, -1, 8),
    ((256, 256, 256), 1, 0, -1, 0),    # the exact 16x16 tile
    ((512, 512, 512), 1, 0, -1, 0),    # R x C tiles
    ((64, 256, 4096), 1, 0, -1, 0),    # four tiles per CU
    ((401, 511, 399), 0, 0, -1, 8), ((528, 255, 528), 0, 0, -1, 4), ((600, 255, 600), 0, 0, -1, 0),
    ((256, 1024, 256), 1, 0, 3, 0),    # a forced configuration
    # any-shape layers past 2.5 tiles per CU: W rows of an even and an odd stride
    ((32, 323, 7146), 0, 0, -1, 4), ((32, 323, 7147), 0, 0, -1, 4),
    ((513, 1023, 512), 0, 0, -1, 8), ((64, 450, 2498), 0, 0, -1, 8),
    ((4, 0, 8), 1, 0, -1, 0), ((0, 4, 8), 1, 0, -1, 0), ((1, 1, 1), 0, 0, -1, 4),
    ((4096, 4096, 4096), 1, 0, -1, 0), ((2001, 2001, 2001), 0, 0, -1, 0),
]


def test_small_tile_rule(driver):
    text = "".join(f"{M} {N} {K} {al} {st} {f}\n" for (M, K, N), al, st, f, _ in CASES)
    got = [int(v) for v in subprocess.run([driver], input=text, capture_output=True, text=True, check=True).stdout.split()]
    assert got == [c[-1] for c in CASES], [(c, g) for c, g in zip(CASES, got) if c[-1] != g]
