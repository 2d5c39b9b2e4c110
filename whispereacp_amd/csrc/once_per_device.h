// What a process does once for each of its GPUs: no HIP here, so that it can be
// checked on the CPU.
#pragma once

#include <atomic>
#include <cstdint>

namespace wsp
{
// Calls `prepare` (0: success) for a device until it has succeeded there once;
// threads may race, so `prepare` has to bear being called twice.
class OncePerDevice
{
public:
    template <class Prepare>
    auto operator()(int device, Prepare prepare) -> decltype(prepare())
    {
        const bool kept = device >= 0 && device < 64;
        const std::uint64_t bit = kept ? std::uint64_t(1) << device : 0;
        if (done.load(std::memory_order_acquire) & bit)
            return {};
        const auto status = prepare();
        if (status == decltype(prepare()) {})
            done.fetch_or(bit, std::memory_order_release);
        return status;
    }

private:
    std::atomic<std::uint64_t> done {0};
};
} // namespace wsp
