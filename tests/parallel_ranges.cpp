// Test driver (CPU only): parallel_ranges covers every index once and throws
// what a loop over the range would have thrown first.
#include <atomic>
#include <cstdio>
#include <stdexcept>
#include <string>

#include "parallel.hpp"

int main() {
  int wrong = 0;
  for (const std::size_t n : {std::size_t(0), std::size_t(1), std::size_t(7), std::size_t(8), std::size_t(511), std::size_t(4099)})
    for (const std::size_t grain : {std::size_t(1), std::size_t(512)}) {
      std::vector<std::atomic<int>> seen(n);
      gagp_amd::parallel_ranges(n, grain, [&](std::size_t begin, std::size_t end) {
        for (std::size_t i = begin; i < end; ++i) ++seen[i];
      });
      for (auto& x : seen) wrong += x != 1;
      if (n < 8) continue;
      std::string said;
      try {
        gagp_amd::parallel_ranges(n, grain, [&](std::size_t begin, std::size_t end) {
          for (std::size_t i = begin; i < end; ++i)
            if (i % 3 == 2 && i >= n / 3) throw std::runtime_error(std::to_string(i));
        });
      } catch (const std::exception& e) {
        said = e.what();
      }
      std::size_t first = n / 3;
      while (first % 3 != 2) ++first;
      wrong += said != std::to_string(first);
    }
  std::printf("%d\n", wrong);
}
