// What has to be done once on every device a process uses, before a kernel's first launch there.  Plain C++, no HIP.
#pragma once
#include <atomic>
#include <cstdint>

namespace tsv {

// Threads may ask at once: both then do it, which does no harm, and neither goes on before it is done.
class OncePerDevice {
    std::atomic<uint64_t> done{0};

  public:
    bool needed(int device) const { return device < 0 || device > 63 || !((done.load(std::memory_order_acquire) >> device) & 1); }
    void note(int device) {
        if (device >= 0 && device <= 63) done.fetch_or(1ull << device, std::memory_order_release);
    }
};

}  // namespace tsv
