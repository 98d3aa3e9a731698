// Host work over an index range on a few threads of its own.
#pragma once
#include <algorithm>
#include <cstddef>
#include <exception>
#include <thread>
#include <vector>

namespace gagp_amd {

constexpr std::size_t kHostThreads = 8;

// f(begin, end) over contiguous ranges of [0, n), at least `grain` long, the
// first on the calling thread. An exception leaves as a loop over [0, n) would
// have thrown it: the one of the lowest range, each range stopping at its first.
template <class F>
void parallel_ranges(std::size_t n, std::size_t grain, F f) {
  const std::size_t cores = std::max<std::size_t>(1, std::thread::hardware_concurrency());
  const std::size_t parts = std::max<std::size_t>(1, std::min({kHostThreads, cores, n / std::max<std::size_t>(1, grain)}));
  std::vector<std::exception_ptr> failed(parts);
  const auto run = [&](std::size_t k) {
    try {
      f(n * k / parts, n * (k + 1) / parts);
    } catch (...) {
      failed[k] = std::current_exception();
    }
  };
  std::vector<std::thread> threads;
  threads.reserve(parts);
  std::size_t inline_from = parts;  // ranges no thread could be started for
  for (std::size_t k = 1; k < parts; ++k) {
    try {
      threads.emplace_back(run, k);
    } catch (...) {  // no thread, or no memory for one; what is started has to be joined
      inline_from = k;
      break;
    }
  }
  run(0);
  for (std::size_t k = inline_from; k < parts; ++k) run(k);
  for (auto& t : threads) t.join();
  for (const auto& e : failed)
    if (e) std::rethrow_exception(e);
}

}  // namespace gagp_amd
