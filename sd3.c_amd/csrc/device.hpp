// What the host side keeps of a device. A process may use several, from several threads: nothing here holds for another device than the
// one it was asked on. Host code only (no device code, so that it also compiles without hipcc).
#pragma once
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <mutex>

#include "../../include/sd3_hip.h"

namespace sd3 {

int fail(int status, const char* fmt, ...);

constexpr int KNOWN_DEVICES = 64;  // devices whose answers are kept; those beyond are asked every time

// compute units of the current device (0 after a failed query, which has set the error message)
inline int compute_units() {
    static std::atomic<int> known[KNOWN_DEVICES];
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0) {
        fail(SD3_ERR_HIP, "cannot query the current device");
        return 0;
    }
    if (dev < KNOWN_DEVICES && (n = known[dev].load(std::memory_order_relaxed)) > 0) return n;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
        fail(SD3_ERR_HIP, "cannot query the number of compute units");
        return 0;
    }
    if (dev < KNOWN_DEVICES) known[dev].store(n, std::memory_order_relaxed);
    return n;
}

// One per kernel (a static of its launcher): allows it `bytes` of dynamic LDS on the current device, where a launch may otherwise have
// no more than 64 KiB. The setting belongs to the function on one device and replaces the one before, so what is set is the most that the
// kernel was ever asked to have, one thread at a time: a size that was allowed stays allowed.
class DynamicLds {
    std::atomic<int> allowed_[KNOWN_DEVICES] = {};  // bytes
    std::mutex setting_;
    int most_ = 0;

  public:
    int allow(const void* kernel, int bytes) {
        if (bytes <= 65536) return SD3_OK;
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || dev < 0) return fail(SD3_ERR_HIP, "cannot query the current device");
        if (dev < KNOWN_DEVICES && allowed_[dev].load(std::memory_order_acquire) >= bytes) return SD3_OK;
        std::lock_guard<std::mutex> one(setting_);
        const int size = most_ > bytes ? most_ : bytes;
        const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, size);
        if (e != hipSuccess) return fail(SD3_ERR_HIP, "cannot allow a kernel %d bytes of LDS: %s", size, hipGetErrorString(e));
        most_ = size;
        if (dev < KNOWN_DEVICES) allowed_[dev].store(size, std::memory_order_release);
        return SD3_OK;
    }
};

}  // namespace sd3
