// Scratch of an attention backward from torch's caching allocator: the largest of the three sizes that can be had.
#pragma once
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/util/Exception.h>
#include <hip/hip_runtime_api.h>

#include <stdint.h>

#include <algorithm>

namespace tyr_torch {

// Whether the allocator can be expected to have `bytes`: from its cache, or from the device.  A request that fails gives the whole
// cache back to the device and waits for it, each time, so one that the caller can do without is not made in vain.  Blocks of the
// cache may be too small one by one, hence "expected".  While the cache holds as much as is asked for (every call but the first
// ones) this copies 1.5 KB of counters; asking the device is not for a stream under capture.
inline bool can_have(size_t bytes, c10::DeviceIndex device) {
    namespace alloc = c10::hip::HIPCachingAllocator;
    try {
        const auto stats = alloc::getDeviceStats(device);
        using c10::CachingAllocator::StatType;
        constexpr size_t all = (size_t)StatType::AGGREGATE, large = (size_t)StatType::LARGE_POOL;
        const int64_t cached = stats.reserved_bytes[large].current - stats.active_bytes[large].current;
        if (cached >= (int64_t)bytes || c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) return true;
        size_t free = 0, total = 0;
        if (hipMemGetInfo(&free, &total) != hipSuccess) {
            (void)hipGetLastError();
            return true;
        }
        const int64_t allowed = (int64_t)(alloc::getMemoryFraction(device) * (double)total) - stats.reserved_bytes[all].current;
        return cached + std::min<int64_t>((int64_t)free, allowed) >= (int64_t)bytes;
    } catch (const c10::Error&) {                     // an allocator that does not tell
        return true;
    }
}

// `take` of the first of `full`, `parts` and `least` bytes that can be had.  (Up to 20 MB the allocator cuts requests from blocks that
// many share.)
template <class F>
auto take_largest(size_t full, size_t parts, size_t least, c10::DeviceIndex device, F take) {
    size_t above = SIZE_MAX;
    for (size_t bytes : {full, parts}) {
        if (bytes > least && bytes < above && (bytes <= (size_t)20 << 20 || can_have(bytes, device))) {
            try {
                return take(bytes);
            } catch (const c10::OutOfMemoryError&) {}
        }
        above = bytes;
    }
    return take(least);
}

}  // namespace tyr_torch
