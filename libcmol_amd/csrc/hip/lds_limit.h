// lds_limit.h — a kernel's dynamic LDS limit, raised once per device.
#pragma once
#include <atomic>
#include <cstdint>

// Kernels with more than 64 KiB of dynamic LDS need their limit raised on
// every device they run on.  One of these per kernel (static) remembers the
// devices that took it; a refusal (e.g. inside a stream capture) is reported
// and asked again on the next launch.  Several threads may get here at once:
// the call is idempotent.
struct LdsLimit {
    std::atomic<uint64_t> done{0};   // bit d: device d; devices past 63 are asked on every launch
    // device: the current device, negative if unknown; set(): raises it there
    template <typename Set>
    bool raise(int device, Set set)
    {
        const uint64_t bit = device >= 0 && device < 64 ? 1ull << device : 0;
        if (done.load(std::memory_order_relaxed) & bit) return true;
        if (!set()) return false;
        done.fetch_or(bit, std::memory_order_relaxed);
        return true;
    }
};
