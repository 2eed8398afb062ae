// Host threads that only help: work that is done without them, later.
#pragma once

#include <cstddef>
#include <system_error>
#include <vector>

namespace vsplat {

// Adds up to `count` threads running `body`; fewer where the system refuses one
// (a limit on threads), which is not an error.
template <class Thread, class Body> void start_helpers(std::vector<Thread> &threads, size_t count, const Body &body) {
  threads.reserve(threads.size() + count);
  try {
    for (size_t k = 0; k < count; ++k) threads.emplace_back(body);
  } catch (const std::system_error &) {
  }
}

} // namespace vsplat
