// cull_shape.hpp -- the workgroup size of the single-view cull without an index array
// (host code).
#pragma once
#include <cstdint>

namespace dpc {

// Threads of a workgroup for n objects on a device of `cus` CUs, 1024 or 64.
//
// A workgroup of one wave spreads a short call over the device: 10,000 objects in
// workgroups of 1024 threads occupy 10 CUs, sixteen waves each (the kernel: 10,000
// objects 3.6 -> 2.8 us, 60,000 4.0 -> 3.2).  Where workgroups of 1024 fill their last
// row of CUs, starting sixteen times as many costs more than it spreads: calls in a
// row, 1024 against 64 threads, 200,003 objects (196 workgroups) 4.9 against 5.2 us,
// 250,007 (245) 5.2 : 5.8, 300,007 (293) 6.9 : 6.5, 400,009 (391) 7.5 : 7.8, 500,003
// (489) 8.0 : 8.9, 600,011 (586) 10.1 : 10.2, 700,001 (684) 10.7 : 11.7, 800,003 (782)
// 13.2 : 12.8, 899,999 (879) 13.8 : 14.6; 150,001 (147) 5.0 : 4.7.  So 1024 from three
// quarters of the rows' workgroups on; with the result's diff from four fifths (the
// cull and the diff, 400,009: 13.1 : 12.9, 600,011: 15.6 : 15.3, 800,003: 18.7 : 18.0,
// but 250,007: 10.5 : 10.9, 500,003: 13.6 : 14.2, 700,001: 16.4 : 16.9).  Longer calls
// wait for memory (1,048,576: 15.0 : 15.7; 4,999,999: 65.3 : 70.2).
constexpr uint32_t flat_cull_threads(uint64_t n, uint32_t cus, bool diff)
{
  const uint64_t groups = (n + 1023) / 1024, rows = (groups + cus - 1) / cus;
  return n > 900'000 || 20 * groups >= (diff ? 16 : 15) * rows * cus ? 1024 : 64;
}

}  // namespace dpc
