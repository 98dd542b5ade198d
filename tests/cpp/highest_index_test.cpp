// The largest index of a request's deltas (host/highest.hpp): every length to 40 and
// place of the largest, values with the sign bit set, and less time than one running
// maximum takes.
#include <algorithm>
#include <chrono>
#include <cstdio>
#include <vector>

#include "host/highest.hpp"

namespace {

__attribute__((noinline, optimize("no-tree-vectorize"))) uint32_t running(const uint32_t* idx, uint32_t n)
{
  uint32_t top = 0;
  for (uint32_t k = 0; k < n; ++k) top = std::max(top, idx[k]);
  return top;
}

__attribute__((noinline)) uint32_t highest(const uint32_t* idx, uint32_t n) { return dpc::highest_index(idx, n); }

template <class F>
double best_us(F&& f)
{
  double best = 1e9;
  for (int r = 0; r < 200; ++r) {
    const auto t0 = std::chrono::steady_clock::now();
    volatile auto x = f();
    (void)x;
    best = std::min(best, std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count());
  }
  return best;
}

}  // namespace

int main()
{
  int failures = 0;
  for (uint32_t offset = 0; offset < 4; ++offset)
    for (uint32_t n = 0; n <= 40; ++n)
      for (uint32_t at = 0; at < std::max(n, 1u); ++at)
        for (uint32_t top : {1u, 0x7fffffffu, 0x80000000u, 0xffffffffu}) {
          std::vector<uint32_t> v(offset + n + 1, 0xffffffffu);
          for (uint32_t k = 0; k < n; ++k) v[offset + k] = k == at ? top : (k * 2654435761u) % top;
          if (dpc::highest_index(v.data() + offset, n) != (n ? top : 0)) ++failures;
        }
  std::vector<uint32_t> idx(150000);
  for (size_t k = 0; k < idx.size(); ++k) idx[k] = static_cast<uint32_t>(k * 2654435761u) % 200000u;
  const uint32_t n = static_cast<uint32_t>(idx.size());
  const double one = best_us([&] { return running(idx.data(), n); });
  const double found = best_us([&] { return highest(idx.data(), n); });
  if (found > 0.7 * one) ++failures;
  std::printf("150000 indices: one running maximum %.1f us, highest %.1f us\nhighest index: %d failures\n", one, found,
              failures);
  return failures ? 1 : 0;
}
