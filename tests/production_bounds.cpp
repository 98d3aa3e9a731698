// Test driver (CPU only): production_bounds against the in-order scan of
// choose_production_in_order, for random weights and for choices at and around
// every bound. Prints the number of choices compared and of disagreements.
#include <cmath>
#include <cstdio>
#include <vector>

#include "grammar.hpp"
#include "phase.hpp"

using namespace gagp_amd;

int main() {
  SplitMix random(0x5eed);
  long long compared = 0, wrong = 0;
  for (int table = 0; table < 4000; ++table) {
    const int n = 1 + int(random.bounded(16));
    const int kind = table % 5;
    std::vector<PProd> p(std::size_t(n), PProd{0, 0.0});
    PNt nt;
    nt.production_count = n;
    for (auto& x : p)
      x.weight = kind == 0 ? 1.0 : kind == 1 ? double(1 + random.bounded(9)) : kind == 2 ? random.unit() : kind == 3 ? double(random.bounded(3))
                                                                               : std::ldexp(random.unit(), int(random.bounded(60)) - 30);
    double maximum = 0;
    for (const auto& x : p) maximum = std::max(maximum, x.weight);
    if (table & 8 && maximum > 0) {
      nt.normalized = 1;
      for (auto& x : p) x.weight /= maximum;
      maximum = 1;
    }
    production_bounds(p.data(), nt);
    if (!(maximum > 0)) { wrong += nt.total != 0; continue; }
    const auto weight = [&](int i) { return nt.normalized ? p[std::size_t(i)].weight : p[std::size_t(i)].weight / maximum; };
    double total = 0;
    for (int i = 0; i < n; ++i) total += weight(i);
    wrong += nt.total != total;
    const auto check = [&](double choice) {
      if (!(choice >= 0) || choice > total) return;
      int scanned = -1, bounded = n - 1;
      double left = choice;
      for (int i = 0; i < n; ++i) {
        scanned = i;
        left -= weight(i);
        if (left < 0) break;
      }
      for (int i = n - 1; i >= 0; --i)
        if (choice < p[std::size_t(i)].below) bounded = i;
      ++compared;
      wrong += scanned != bounded;
    };
    for (int k = 0; k < 200; ++k) check(random.unit() * total);
    check(0);
    check(total);
    for (const auto& x : p) {
      double below = x.below, above = x.below;
      for (int k = 0; k < 8; ++k) {
        check(below);
        check(above);
        below = std::nextafter(below, 0.0);
        above = std::nextafter(above, 1e300);
      }
    }
  }
  std::printf("{\"compared\": %lld, \"wrong\": %lld}\n", compared, wrong);
}
