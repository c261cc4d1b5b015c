// Errors of the host code (no device headers).
#pragma once

#include <cstdint>
#include <stdexcept>

namespace symhip {

struct Error : std::runtime_error {
  using std::runtime_error::runtime_error;
};

// The device has no room for an allocation. Of all errors the one that asking for less can mend.
struct OutOfMemory : Error {
  using Error::Error;
};

// reserve(m) for m = want, want / 2, .. 1 until the device has the room; returns that m. Every error
// but OutOfMemory passes through, and so does OutOfMemory at m = 1.
template <typename F>
int32_t reserve_at_most(int32_t want, F&& reserve) {
  for (int32_t m = want;; m /= 2) {
    try {
      reserve(m);
      return m;
    } catch (const OutOfMemory&) {
      if (m <= 1) throw;
    }
  }
}

}  // namespace symhip
