// More than 64 KB of dynamic LDS has to be asked for, once for a kernel and device and outside any stream capture a caller may open
// later.  The record is per device: a process that goes on to a second one asks again there.
#pragma once

#include <atomic>
#include <cstddef>
#include <cstdint>

namespace afhip {

class LdsLimit {
  public:
    // `device()` gives the current device or a negative number, `ask()` raises the kernel's limit there; what `ask` returns is
    // returned, `ok` where nothing had to be asked.  A failure is not remembered; two threads may both ask, which does no harm.
    template <typename Status, typename Device, typename Ask>
    Status raise(size_t lds, Status ok, Device device, Ask ask) {
        if (lds <= 64 * 1024) return ok;
        const int d = device();
        const uint64_t bit = d >= 0 && d < 64 ? uint64_t{1} << d : 0;  // (others ask every time)
        if (devices_.load(std::memory_order_acquire) & bit) return ok;
        const Status s = ask();
        if (s == ok) devices_.fetch_or(bit, std::memory_order_release);
        return s;
    }

  private:
    std::atomic<uint64_t> devices_{0};
};

}  // namespace afhip
