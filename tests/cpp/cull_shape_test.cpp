// The workgroup size of the flat cull (cull_shape.hpp) on a device of 256 CUs: at the
// sizes where both were measured the faster one, or either where they were equal.
#include <cstdio>
#include <initializer_list>

#include "cull_shape.hpp"

int main()
{
  const struct {
    unsigned long n;
    unsigned want, with_diff;
  } measured[] = {{1, 64, 64},           {10007, 64, 64},       {60001, 64, 64},       {100003, 64, 64},
                  {150001, 64, 64},      {200003, 1024, 64},    {250007, 1024, 1024},  {262144, 1024, 1024},
                  {262145, 64, 64},      {300007, 64, 64},      {400009, 1024, 64},    {500003, 1024, 1024},
                  {600011, 1024, 64},    {700001, 1024, 1024},  {800003, 1024, 64},    {899999, 1024, 1024},
                  {1048576, 1024, 1024}, {4999999, 1024, 1024}};
  int failures = 0;
  for (const auto& m : measured)
    if (dpc::flat_cull_threads(m.n, 256, false) != m.want || dpc::flat_cull_threads(m.n, 256, true) != m.with_diff) {
      std::printf("%lu objects: %u threads, %u with the diff\n", m.n, dpc::flat_cull_threads(m.n, 256, false),
                  dpc::flat_cull_threads(m.n, 256, true));
      ++failures;
    }
  for (unsigned cus : {1u, 7u, 80u, 304u})  // any device gets one of the two
    for (unsigned long n : {1ul, 64ul, 1025ul, 300007ul, 900001ul})
      if (const unsigned t = dpc::flat_cull_threads(n, cus, n % 2); t != 64 && t != 1024) ++failures;
  std::printf("cull shape: %d failures\n", failures);
  return failures ? 1 : 0;
}
