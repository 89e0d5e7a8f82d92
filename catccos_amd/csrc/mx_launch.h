// Host-side launch state that the translation units with matmul kernels share.
#pragma once

#include <atomic>
#include <vector>

#include "mx_common.h"

namespace cmx {

// Launch state that belongs to a device, not to the process: the dynamic-LDS limit of a kernel has to be raised on
// every device that runs it, and the CU count differs between devices.  One slot per device ordinal; the flags are
// atomics so that concurrent first calls from several host threads are merely redundant.
constexpr int kMaxDevices = 64;

struct PerDeviceFlag {
    std::atomic<bool> done[kMaxDevices];
};

inline int current_device_slot(int* dev_out) {
    int dev = 0;
    CMX_HIP(hipGetDevice(&dev));
    CMX_REQUIRE(dev >= 0 && dev < kMaxDevices, "device ordinal out of range");
    *dev_out = dev;
    return CMX_OK;
}

// Every kernel that needs more dynamic LDS than the default limit is listed here at load time (one entry per
// instantiation that a launch function names), so that cmx_init can raise all the limits up front and no first
// call has to -- hipFuncSetAttribute is not allowed while a stream is being captured into a graph.
struct LdsKernel {
    const void* fn;
    int bytes;
    PerDeviceFlag* flag;
};
inline std::vector<LdsKernel>& lds_registry() {
    static std::vector<LdsKernel> v;
    return v;
}
template <auto KFN, size_t SMEM>
struct LdsSetup {
    static inline PerDeviceFlag flag{};
    static inline const bool registered = (lds_registry().push_back({reinterpret_cast<const void*>(KFN), (int)SMEM, &flag}), true);
};

inline int allow_dynamic_lds(const void* kfn, int bytes, PerDeviceFlag& flag) {
    int dev = 0;
    int rc = current_device_slot(&dev);
    if (rc != CMX_OK) return rc;
    if (!flag.done[dev].load(std::memory_order_acquire)) {
        CMX_HIP(hipFuncSetAttribute(kfn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
        flag.done[dev].store(true, std::memory_order_release);
    }
    return CMX_OK;
}
// raises the limit of KFN on the current device unless cmx_init or an earlier call has done so
template <auto KFN, size_t SMEM>
int allow_dynamic_lds() {
    (void)LdsSetup<KFN, SMEM>::registered;
    return allow_dynamic_lds(reinterpret_cast<const void*>(KFN), (int)SMEM, LdsSetup<KFN, SMEM>::flag);
}

inline int cu_count(int* out) {
    static std::atomic<int> cus[kMaxDevices];
    int dev = 0;
    int rc = current_device_slot(&dev);
    if (rc != CMX_OK) return rc;
    int n = cus[dev].load(std::memory_order_acquire);
    if (n == 0) {
        CMX_HIP(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev));
        n = n > 0 ? n : 256;
        cus[dev].store(n, std::memory_order_release);
    }
    *out = n;
    return CMX_OK;
}

}  // namespace cmx
