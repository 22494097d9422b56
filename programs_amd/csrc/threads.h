// A few host threads for the length of one call.
#pragma once
#include <exception>
#include <thread>
#include <vector>

namespace fvk {

// part(t) for t in [0, n): part 0 on the calling thread, which also runs the
// parts whose threads cannot be started (an exception must not leave a C entry)
template <class F>
void on_threads(int n, F part) {
  std::vector<std::thread> th;
  int started = 1;
  try {
    th.reserve(n);
    for (; started < n; ++started) th.emplace_back(part, started);
  } catch (const std::exception &) {
  }
  part(0);
  for (int t = started; t < n; ++t) part(t);
  for (auto &t : th) t.join();
}

}  // namespace fvk
