"""The runtime's grow-only device buffers (ml-edsl_amd/csrc/dev_buf.hpp) on a
device that runs out of memory, on the CPU with stand-ins for the HIP calls."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

DRIVER = r"""
#include <cstdio>
#include <cstdlib>
#include <map>
#include "dev_buf.hpp"

static size_t g_left = 0;
static std::map<void*, size_t> g_live;
static hipError_t g_last = hipSuccess;
extern "C" hipError_t hipMalloc(void** p, size_t n) {
  if (n > g_left) return g_last = hipErrorOutOfMemory;
  g_left -= n;
  *p = malloc(16);
  g_live[*p] = n;
  return hipSuccess;
}
extern "C" hipError_t hipFree(void* p) {
  g_left += g_live.at(p);
  g_live.erase(p);
  free(p);
  return hipSuccess;
}
extern "C" hipError_t hipGetLastError() { const hipError_t e = g_last; g_last = hipSuccess; return e; }
extern "C" hipError_t hipDeviceSynchronize() { return hipSuccess; }
void edsl::rt::check_hip(hipError_t e, const char*) { if (e != hipSuccess) throw e; }

#define CHECK(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)

int main() {
  using edsl::rt::DevBuf;
  {  // kept: growth at least twofold, the outgrown buffer still allocated
    g_left = 1 << 20;
    DevBuf b(true);
    void* p = b.ensure(1000);
    CHECK(b.cap == 1024 && b.ensure(1024) == p);
    void* q = b.ensure(1025);
    CHECK(q != p && b.cap == 2048 && b.retired.size() == 1 && b.retired[0] == p && g_live.count(p));
    // no room for twice the size: the size itself
    g_left = 3072;
    CHECK(b.ensure(3000) && b.cap == 3072 && g_last == hipSuccess);
    // no room at all: null, no error left behind, and the buffer goes on
    void* last = b.p;
    g_left = 100;
    CHECK(b.try_ensure(4000) == nullptr && g_last == hipSuccess);
    CHECK(b.p == last && b.cap == 3072 && b.try_ensure(3072) == last && b.retired.size() == 2);
    bool thrown = false;
    try { b.ensure(4000); } catch (hipError_t e) { thrown = e == hipErrorOutOfMemory; }
    CHECK(thrown && b.ensure(64) == last);
  }
  {  // not kept: released first
    g_left = 4096;
    DevBuf b;
    b.ensure(4096);
    CHECK(b.ensure(4000) && b.cap == 4096);
    g_left = 1024;
    CHECK(b.ensure(5000) && b.cap == 5120 && b.retired.empty() && g_left == 0);
  }
  puts("ok");
}
"""


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir(os.path.join(ROCM, "include", "hip")),
                    reason="g++ or the HIP headers not available")
def test_buffers_on_a_full_device(tmp_path):
    src, exe = tmp_path / "driver.cpp", tmp_path / "driver"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROCM, "include"),
                    "-I" + os.path.join(ROOT, "ml-edsl_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0 and res.stdout == "ok\n", res.stdout
