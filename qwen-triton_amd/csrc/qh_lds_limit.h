// The limit of a kernel's dynamic LDS, host side.
#pragma once

#include <hip/hip_runtime_api.h>
#include <stdint.h>

#include <atomic>

#include "qwen_hip.h"

namespace qh {

void set_error(const char* fmt, ...);

// Raises one kernel's limit once per device: the attribute belongs to the current device, so a process that
// goes on to another one sets it there too, and a call that failed is made again. Not a stream operation
// (allowed under capture). One static instance per kernel; threads may share it.
class LdsLimit {
 public:
  int raise(const void* kern, int bytes, const char* name) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
      set_error("%s: no current device", name);
      return QH_E_HIP;
    }
    if (done_.load(std::memory_order_relaxed) >> dev & 1) return QH_OK;
    const hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) {
      set_error("%s: cannot raise the LDS limit to %d bytes: %s", name, bytes, hipGetErrorString(e));
      return QH_E_HIP;
    }
    done_.fetch_or(1ull << dev, std::memory_order_relaxed);
    return QH_OK;
  }

 private:
  std::atomic<uint64_t> done_{0};
};

}  // namespace qh
