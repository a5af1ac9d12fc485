// Dynamic LDS of a kernel beyond the default of 64 KiB a workgroup.
#pragma once

#include <atomic>
#include <cstdint>

#include "runtime.h"

namespace life {

// One kernel's allowance (gfx950 has 160 KiB), asked for once on each device
// that launches it: the attribute belongs to the device, and a launch that
// needs it fails without.
class LdsLimit {
  public:
    // bytes: of this launch; most: of any launch of the kernel.
    void allow(const void* kernel, size_t bytes, size_t most) {
        if (bytes <= 64 * 1024) return;
        int device = 0;
        LIFE_HIP(hipGetDevice(&device));
        const uint64_t bit = device < 64 ? uint64_t(1) << device : 0;
        if (allowed_.load(std::memory_order_relaxed) & bit) return;
        LIFE_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)most));
        allowed_.fetch_or(bit, std::memory_order_relaxed);
    }

  private:
    std::atomic<uint64_t> allowed_{0};  // devices, a bit each (past 64: asked for at every launch)
};

}  // namespace life
