// chronos_lds.h — dynamic LDS beyond a kernel's default, asked for on the host.
#pragma once
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <stdint.h>

namespace chronos {

// Lets Kern take up to `bytes` of dynamic LDS on the current device: once per kernel and device, to which the attribute belongs (a call costs 1 to 2 us).
template <auto* Kern> inline void lds_limit(int bytes) {
    static std::atomic<uint64_t> done{0};   // a bit per device; of those beyond 64, every time
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) dev = -1;
    const uint64_t bit = dev >= 0 && dev < 64 ? 1ull << dev : 0;
    if (bit != 0 && (done.load(std::memory_order_acquire) & bit) != 0) return;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(Kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess)
        done.fetch_or(bit, std::memory_order_release);
}

}  // namespace chronos
