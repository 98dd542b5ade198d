// quick_cull.hpp -- a cheap test that decides most (object, frustum) pairs and
// says so, with the reference's result; the rest take the exact test.
//
// The exact test (obb_visible, dp/culling/cpu/src/ManagerImpl.cpp:199-289)
// transforms a point and three edges by the view-projection matrix, forms eight
// corners with separately rounded adds and compares each against six planes:
// 188 operations.  Its outcome depends on the rounding of those operations only
// where a corner lies within a rounding error of a plane.  Everywhere else any
// evaluation with a known error bound gives the same answer: here the clip-space
// centre of the object's world box (twice the centre, 2p + ex + ey + ez) and the
// radius of the world-axis-aligned box around it, about 50 operations with
// fused multiply-adds.  A pair closer to a plane than `eps`, a bound on all
// rounding errors of both evaluations, is left undecided.
//
// In terms of the exact sums over the eight corners, with w and c (= x, y or z)
// the clip coordinates, the reference reports an object culled when on some axis
// all corners have c <= -w, or all have w <= c and none has c <= -w.
//   visible   the centre lies inside all six planes: some corner then lies
//             strictly inside each of them
//   culled    x, y: |c| - radius(c) > |w| + radius(w): every corner is beyond the
//             same plane, and (for c > 0) no corner has c <= -w
//             z: every corner has z < -w; or every corner has w < z and z > -w
// z uses the sums z + w and w - z of the matrix's columns: for a distant far
// plane w - z hardly changes with the position, while z and w do.
//
// The bound.  u = 2^-24, A_j = |p_j| + |ex_j| + |ey_j| + |ez_j|, S_c = sum_j A_j
// |M_jc|, everything in the doubled scale.  Errors of the exact test's corners:
// 14 u S_c per coordinate (four-term products 4 u, three adds 3 u, doubled).
// Errors here: centre 12 u S_c, radii and chained sums 11 u S_c, the column sums
// and last adds 4 u more: below 41 u (S_c + S_w) together.  S_c + S_w <=
// 2 (n3 * s3 + n4 * sw) with n3, n4 the largest magnitudes of rows 0-2 and row 3
// and s3 = sum of A_j over x, y, z, sw = A_w.  eps = 2^-17 (n3 s3 + n4 sw) = 64 u
// (S_c + S_w)'s bound.  The added 2^-117 and 2^-130 cover underflow.  Operands
// of 2^56 (matrix) or 2^60 (object) and above, infinities and NaN make eps
// infinite or NaN, and every comparison below false: undecided.  So does an
// object whose edges have a w component.
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define DPC_HD __host__ __device__ __forceinline__
#else
#define DPC_HD inline
#endif

namespace dpc {

// What the quick test reads of an object (doubled scale).
struct QuickObj {
  float cx, cy, cz, cw;  // 2p + ex + ey + ez
  float hx, hy, hz;      // |ex| + |ey| + |ez| per component
  float s3, sw;          // the object's factors of eps
};

// What it reads of a view-projection matrix beside its elements.
struct alignas(16) QuickView {
  float lo[4], hi[4];  // rows of z + w and w - z
  float n3, n4;        // largest magnitude in rows 0-2, in row 3 (infinite from 2^56 on)
  float pad[2];
};

DPC_HD float quick_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// p, ex, ey, ez: the object's point and edges as the exact test takes them.
template <class V4>
DPC_HD QuickObj quick_obj(const V4& p, const V4& ex, const V4& ey, const V4& ez)
{
  QuickObj q;
  q.cx = quick_fma(2.0f, p.x, (ex.x + ey.x) + ez.x);
  q.cy = quick_fma(2.0f, p.y, (ex.y + ey.y) + ez.y);
  q.cz = quick_fma(2.0f, p.z, (ex.z + ey.z) + ez.z);
  q.cw = 2.0f * p.w;
  q.hx = (__builtin_fabsf(ex.x) + __builtin_fabsf(ey.x)) + __builtin_fabsf(ez.x);
  q.hy = (__builtin_fabsf(ex.y) + __builtin_fabsf(ey.y)) + __builtin_fabsf(ez.y);
  q.hz = (__builtin_fabsf(ex.z) + __builtin_fabsf(ey.z)) + __builtin_fabsf(ez.z);
  const float flat = (__builtin_fabsf(ex.w) + __builtin_fabsf(ey.w)) + __builtin_fabsf(ez.w);
  const float aw = __builtin_fabsf(p.w);
  const float a3 = ((__builtin_fabsf(p.x) + __builtin_fabsf(p.y)) + __builtin_fabsf(p.z)) + ((q.hx + q.hy) + q.hz);
  const bool fits = (flat == 0.0f) & (a3 + aw < 0x1p60f);  // (false for NaN)
  q.s3 = fits ? quick_fma(a3, 0x1p-17f, 0x1p-117f) : __builtin_inff();
  q.sw = quick_fma(aw, 0x1p-17f, 0x1p-117f);
  return q;
}

// The largest magnitude of the elements of row 3, or of rows 0-2, as a float:
// magnitudes compare as their bits do, NaN above infinity (integer operations,
// which run on the scalar unit for a wave-uniform matrix).
DPC_HD uint32_t quick_magnitude(float v) { return __builtin_bit_cast(uint32_t, v) & 0x7fffffffu; }

// (2^56 and above: infinite)
DPC_HD float quick_scale(uint32_t bits)
{
  return __builtin_bit_cast(float, bits >= 0x5b800000u ? 0x7f800000u : bits);
}

DPC_HD QuickView quick_view(const float* m)
{
  QuickView v;
  for (int j = 0; j < 4; ++j) {
    v.lo[j] = m[4 * j + 2] + m[4 * j + 3];
    v.hi[j] = m[4 * j + 3] - m[4 * j + 2];
  }
  uint32_t n3 = 0, n4 = 0;
  for (int k = 0; k < 12; ++k) {
    const uint32_t b = quick_magnitude(m[k]);
    n3 = b > n3 ? b : n3;
  }
  for (int k = 12; k < 16; ++k) {
    const uint32_t b = quick_magnitude(m[k]);
    n4 = b > n4 ? b : n4;
  }
  v.n3 = quick_scale(n3);
  v.n4 = quick_scale(n4);
  v.pad[0] = v.pad[1] = 0.0f;
  return v;
}

// less(a, b) answers a < b: as a bool, or on the device as the mask of the lanes
// where it holds (a comparison goes straight into a lane mask, while a condition
// formed from several would first be spread over a register and compared again).
// M: what it answers with.
template <class M>
struct QuickResult {
  M visible;  // certainly visible
  M culled;   // certainly culled (neither: undecided)
};

template <class M, class Less>
DPC_HD QuickResult<M> quick_test(const QuickObj& q, const float* m, const QuickView& v, Less&& less)
{
  const float eps = quick_fma(v.n3, q.s3, quick_fma(v.n4, q.sw, 0x1p-130f));
  // clip-space centre: x, y, w from the matrix, z + w and w - z from its column sums
  const float cx = quick_fma(q.cw, m[12], quick_fma(q.cz, m[8], quick_fma(q.cy, m[4], q.cx * m[0])));
  const float cy = quick_fma(q.cw, m[13], quick_fma(q.cz, m[9], quick_fma(q.cy, m[5], q.cx * m[1])));
  const float cw = quick_fma(q.cw, m[15], quick_fma(q.cz, m[11], quick_fma(q.cy, m[7], q.cx * m[3])));
  const float dl = quick_fma(q.cw, v.lo[3], quick_fma(q.cz, v.lo[2], quick_fma(q.cy, v.lo[1], q.cx * v.lo[0])));
  const float dh = quick_fma(q.cw, v.hi[3], quick_fma(q.cz, v.hi[2], quick_fma(q.cy, v.hi[1], q.cx * v.hi[0])));
  const float acx = __builtin_fabsf(cx), acy = __builtin_fabsf(cy);
  // radius(x) - |x|, radius(y) - |y|, |w| + radius(w), radius(z + w), (w - z) + radius(w - z)
  const float rx = quick_fma(q.hz, __builtin_fabsf(m[8]),
                             quick_fma(q.hy, __builtin_fabsf(m[4]), quick_fma(q.hx, __builtin_fabsf(m[0]), -acx)));
  const float ry = quick_fma(q.hz, __builtin_fabsf(m[9]),
                             quick_fma(q.hy, __builtin_fabsf(m[5]), quick_fma(q.hx, __builtin_fabsf(m[1]), -acy)));
  const float rw = quick_fma(q.hz, __builtin_fabsf(m[11]),
                             quick_fma(q.hy, __builtin_fabsf(m[7]),
                                       quick_fma(q.hx, __builtin_fabsf(m[3]), __builtin_fabsf(cw))));
  const float rl = quick_fma(q.hz, __builtin_fabsf(v.lo[2]),
                             quick_fma(q.hy, __builtin_fabsf(v.lo[1]), q.hx * __builtin_fabsf(v.lo[0])));
  const float rh = quick_fma(q.hz, __builtin_fabsf(v.hi[2]),
                             quick_fma(q.hy, __builtin_fabsf(v.hi[1]), quick_fma(q.hx, __builtin_fabsf(v.hi[0]), dh)));
  const float inner = cw - eps, outer = rw + eps;
  QuickResult<M> r;
  r.visible = less(acx, inner) & less(acy, inner) & less(eps, dl) & less(eps, dh);
  r.culled = less(outer, -rx) | less(outer, -ry) | less(dl + rl, -eps) | (less(rh, -eps) & less(eps, dl - rl));
  return r;
}

}  // namespace dpc
