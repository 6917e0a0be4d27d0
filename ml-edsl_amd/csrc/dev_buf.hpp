// The runtime's grow-only device buffers.
#pragma once

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstddef>
#include <vector>

namespace edsl {
namespace rt {

void check_hip(hipError_t e, const char* what);  // throws Failure (runtime.cpp)

struct DevBuf {
  void* p = nullptr;
  size_t cap = 0;
  // Workspaces of the device entry points may be baked into HIP graphs that
  // callers capture, so an outgrown one is kept (retired) rather than freed:
  // a replay still finds the buffer it was captured with. Growth is then at
  // least twofold while the device has the memory, which bounds the retired
  // total by the final capacity.
  bool keep_old = false;
  std::vector<void*> retired;

  DevBuf() = default;
  explicit DevBuf(bool keep) : keep_old(keep) {}

  // A buffer of at least `bytes`, or null where device memory does not suffice;
  // a kept buffer then stays in use for calls that fit it. A buffer that is
  // released may still be in use by queued work, so the device is drained first.
  void* try_ensure(size_t bytes) {
    if (bytes <= cap && p) return p;
    if (p && !keep_old) {
      check_hip(hipDeviceSynchronize(), "hipDeviceSynchronize");
      check_hip(hipFree(p), "hipFree");
      p = nullptr;
      cap = 0;
    }
    const size_t least = std::max<size_t>((bytes + 255) & ~size_t(255), 256);
    for (const size_t want : {std::max(least, 2 * cap), least}) {
      void* fresh = nullptr;
      const hipError_t e = hipMalloc(&fresh, want);
      if (e == hipSuccess) {
        if (p) retired.push_back(p);
        p = fresh;
        cap = want;
        return p;
      }
      (void)hipGetLastError();  // not for the next launch to report
      if (e != hipErrorOutOfMemory) check_hip(e, "hipMalloc");
    }
    return nullptr;
  }

  void* ensure(size_t bytes) {
    void* const q = try_ensure(bytes);
    if (!q) check_hip(hipErrorOutOfMemory, "hipMalloc");
    return q;
  }
};

}  // namespace rt
}  // namespace edsl
