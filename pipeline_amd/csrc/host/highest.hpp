// highest.hpp -- the largest of an array of 32-bit indices (host code).
#pragma once
#include <algorithm>
#include <cstdint>
#include <cstring>

namespace dpc {

// The largest of idx[0 .. n), 0 of none.  One running maximum is a chain of dependent
// steps, two cycles an index: 150,000 indices of a request took 104 us, where comparing
// each with a limit took 52 to 104 (as the loop lay in the code).  Two maxima of four
// indices each take 35 (four single ones 47), and the server's lock need not be held, as
// the limit is not needed.
inline uint32_t highest_index(const uint32_t* idx, uint32_t n)
{
  typedef uint32_t Four __attribute__((vector_size(16)));
  Four a = {}, b = {};
  uint32_t k = 0;
  for (; n - k >= 8; k += 8) {
    Four x, y;
    std::memcpy(&x, idx + k, 16);
    std::memcpy(&y, idx + k + 4, 16);
    a = x > a ? x : a;
    b = y > b ? y : b;
  }
  uint32_t top = 0;
  for (; k < n; ++k) top = std::max(top, idx[k]);
  for (int i = 0; i < 4; ++i) top = std::max(top, std::max<uint32_t>(a[i], b[i]));
  return top;
}

}  // namespace dpc
