// How much dynamic LDS each kernel may have. hipFuncSetAttribute holds for the whole process, and a smaller request from one
// thread takes away what another has asked for: what is asked for is remembered process-wide and only rises.
#pragma once

#include <cstddef>
#include <map>
#include <mutex>
#include <utility>

namespace tnn {

class LdsReservations {
  public:
    /// Bytes the kernel may have on the device once this returns, at least `bytes`; 0 if `set` (called with the bytes, only where
    /// they are more than anyone has asked for) fails.
    template <typename Set> size_t at_least(const void *kernel, int device, size_t bytes, Set &&set) {
        const std::lock_guard<std::mutex> lock(mutex_);
        size_t &reserved = reserved_[{kernel, device}];
        if (reserved < bytes) {
            if (!set(bytes)) return 0;
            reserved = bytes;
        }
        return reserved;
    }

  private:
    std::mutex mutex_;
    std::map<std::pair<const void *, int>, size_t> reserved_;
};

} // namespace tnn
