// quick_cull.hpp -- a cheap test that decides most (object, frustum) pairs and
// says so, with the reference's result; the rest take the exact test.
//
// The exact test (obb_visible, dp/culling/cpu/src/ManagerImpl.cpp:199-289)
// transforms a point and three edges by the view-projection matrix, forms eight
// corners with separately rounded adds and compares each against six planes:
// 188 operations.  Its outcome depends on the rounding of those operations only
// where a corner lies within a rounding error of a plane.  Everywhere else any
// evaluation with a known error bound gives the same answer: here the clip-space
// centre of the object (twice the centre, 2p + ex + ey + ez) and a sphere around
// it: 28 fused multiply-adds, which run on the matrix cores, and 14 operations
// more.  A pair closer to a plane than `eps`, a bound on all rounding errors of both
// evaluations, is left undecided, and so is one whose sphere reaches a plane that
// its centre lies outside of: 2 to 10 in a thousand of the pairs of ordinary
// scenes, most of which do touch a plane.
//
// In terms of the exact sums over the eight corners, with w and c (= x, y or z)
// the clip coordinates, the reference reports an object culled when on some axis
// all corners have c <= -w, or all have w <= c and none has c <= -w.
//   visible   the centre lies inside all six planes: some corner then lies
//             strictly inside each of them
//   culled    x, y: |c| - |w| > r max(|Mw - Mc|, |Mw + Mc|) at the centre: every
//             corner is beyond the same plane, and (for c > 0) none has c <= -w
//             z: every corner has z < -w; or every corner has w < z and z > -w
// (Mc: the first three elements of a column of the matrix; r: the sphere's radius.)
// z uses the sums z + w and w - z of the matrix's columns: for a distant far
// plane w - z hardly changes with the position, while z and w do.
//
// The sphere (doubled scale): |+-ex +-ey +-ez|^2 is at most the sum of the edges'
// squares and twice the magnitudes of their products, which for the edges of a box
// under rotation and scale are zero.  Radius and norms are rounded up: by 2^-18 of
// their value, over ten times what their evaluation can lose, and by 2^-60, more
// than the underflow of squares hides.
//
// The bound.  u = 2^-24, A_j = |p_j| + |ex_j| + |ey_j| + |ez_j|, S_c = sum_j A_j
// |M_jc|, everything in the doubled scale.  S_c <= T = n3 s3 + n4 sw with n3, n4 the
// largest magnitudes of rows 0-2 and row 3, s3 >= sum of A_j over x, y, z (the
// edges' part is at most 3 r), sw = A_w.  Errors of the exact test's corners: 14 u
// S_c per coordinate (four-term products 4 u, three adds 3 u, doubled).  Errors
// here: the centre 3 u A_j and the products 8 u, 11 u S_c per coordinate; the sums
// and differences of columns 2 u more, 13 u (S_z + S_w) <= 26 u T for each of z + w
// and w - z.  What the norms lose before they are rounded up is below 2 u T.
//   z + w, w - z       28 + 26 + 2 = 56 u T
//   x and w, at twice the scale: 2 (14 u S_x + 14 u S_w) <= 56, x 22, w 52, the last
//   two adds 8, the norms 4: 142 u T, and 138 without the norms
// The bounds take 80 u T for z + w and w - z and 160 u T for x and y, and the tests
// for `visible` 80 and twice that: 2^-17 s3 and 2^-17 sw (128 u) times 0.625 and 1.25
// of n3 and n4.  The 2^-90 and 2^-117 added to the object's factors cover underflow.
//
// What the bound does not cover is left undecided: operands of 2^56 (matrix) or 2^60
// (object) and above, infinities and NaN, matrices whose rows 0-2 lie below 2^-47, and
// objects whose edges have a w component make n3, n4 or s3 infinite, and every bound
// +infinity or NaN.  No comparison for `culled` holds with one.  The test for `visible`
// takes its operands from medians, which drop a NaN (quick_med3):
//   both bounds of z infinite   eps is +infinity, below neither of z + w and w - z
//   one NaN (eps -infinity)     it comes from the radius, a norm or sw times n4.
//     The radius is NaN only where an edge has an infinite or NaN component (finite
//     ones overflow to magnitudes): that component of the centre is too, every
//     output is infinite or NaN, and `far` +infinity, below nothing.
//     A norm is NaN only where the column of its own output, z + w or w - z, has a
//     NaN; sw times n4 only where p.w is NaN, or infinite over a row 3 of zeros.  The
//     output is then NaN and `near` -infinity, above nothing.
//   x or y NaN (dropped by `far`)  only with operands that make both bounds so.
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
  float r;               // radius of a sphere around it that holds the object
  float s3, sw;          // the object's factors of eps
};

// What it reads of a view-projection matrix: rows of four clip-space outputs of the
// centre, all at twice their scale, 2x, 2y, z + w and w - z (whose sum is 2w), and
// the norms of their bounds, r n[i] + eps: of w - x or w + x (the larger, doubled),
// of w - y or w + y, of z + w and of w - z.  n3, n4: the largest magnitudes in rows
// 0-2 and in row 3 as factors of eps, [0] for x and y, [1] for z + w and w - z
// (infinite: decides nothing).
struct alignas(16) QuickView {
  float a[4][4];
  float n[4];
  float n34[2][2];  // [0]: n3, n4 for x and y
};

DPC_HD float quick_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// A square root of v or more (v >= 0, or NaN).
DPC_HD float quick_root(float v)
{
#ifdef __HIP_DEVICE_COMPILE__
  const float root = __builtin_amdgcn_sqrtf(v);  // (within an ulp, like the correctly rounded one)
#else
  const float root = __builtin_sqrtf(v);
#endif
  return quick_fma(root, 1.0f + 0x1p-18f, 0x1p-60f);
}

DPC_HD float quick_dot(float ax, float ay, float az, float bx, float by, float bz)
{
  return quick_fma(az, bz, quick_fma(ay, by, ax * bx));
}

// p, ex, ey, ez: the object's point and edges as the exact test takes them.
template <class V4>
DPC_HD QuickObj quick_obj(const V4& p, const V4& ex, const V4& ey, const V4& ez)
{
  QuickObj q;
  q.cx = quick_fma(2.0f, p.x, (ex.x + ey.x) + ez.x);
  q.cy = quick_fma(2.0f, p.y, (ex.y + ey.y) + ez.y);
  q.cz = quick_fma(2.0f, p.z, (ex.z + ey.z) + ez.z);
  q.cw = 2.0f * p.w;
  const float squares = (quick_dot(ex.x, ex.y, ex.z, ex.x, ex.y, ex.z) + quick_dot(ey.x, ey.y, ey.z, ey.x, ey.y, ey.z)) +
                        quick_dot(ez.x, ez.y, ez.z, ez.x, ez.y, ez.z);
  const float products = (__builtin_fabsf(quick_dot(ex.x, ex.y, ex.z, ey.x, ey.y, ey.z)) +
                          __builtin_fabsf(quick_dot(ey.x, ey.y, ey.z, ez.x, ez.y, ez.z))) +
                         __builtin_fabsf(quick_dot(ez.x, ez.y, ez.z, ex.x, ex.y, ex.z));
  q.r = quick_root(quick_fma(2.0f, products, squares));
  const float flat = (__builtin_fabsf(ex.w) + __builtin_fabsf(ey.w)) + __builtin_fabsf(ez.w);
  const float aw = __builtin_fabsf(p.w);
  const float a3 = quick_fma(3.0f, q.r, (__builtin_fabsf(p.x) + __builtin_fabsf(p.y)) + __builtin_fabsf(p.z));
  const bool fits = (flat == 0.0f) & (a3 + aw < 0x1p60f);  // (false for NaN)
  q.s3 = fits ? quick_fma(a3, 0x1p-17f, 0x1p-90f) : __builtin_inff();
  q.sw = quick_fma(aw, 0x1p-17f, 0x1p-117f);
  return q;
}

// v_med3_f32, in one instruction where a maximum first quiets its operands: the median,
// and with a NaN among them the smallest of the others.
DPC_HD float quick_med3(float a, float b, float c)
{
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_fmed3f(a, b, c);
#else
  if (a != a || b != b || c != c) return __builtin_fminf(__builtin_fminf(a, b), c);
  return __builtin_fmaxf(__builtin_fminf(a, b), __builtin_fminf(__builtin_fmaxf(a, b), c));
#endif
}

// The largest magnitude of the elements of row 3, or of rows 0-2, as a float:
// magnitudes compare as their bits do, NaN above infinity (integer operations,
// which run on the scalar unit for a wave-uniform matrix).
DPC_HD uint32_t quick_magnitude(float v) { return __builtin_bit_cast(uint32_t, v) & 0x7fffffffu; }

DPC_HD QuickView quick_view(const float* m)
{
  QuickView v;
  for (int j = 0; j < 4; ++j) {
    v.a[0][j] = 2.0f * m[4 * j];
    v.a[1][j] = 2.0f * m[4 * j + 1];
    v.a[2][j] = m[4 * j + 2] + m[4 * j + 3];
    v.a[3][j] = m[4 * j + 3] - m[4 * j + 2];
  }
  for (int c = 0; c < 2; ++c) {
    const float d0 = m[3] - m[c], d1 = m[7] - m[4 + c], d2 = m[11] - m[8 + c];
    const float s0 = m[3] + m[c], s1 = m[7] + m[4 + c], s2 = m[11] + m[8 + c];
    const float d = quick_dot(d0, d1, d2, d0, d1, d2), s = quick_dot(s0, s1, s2, s0, s1, s2);
    v.n[c] = 2.0f * quick_root(d > s ? d : s);  // (NaN: n3 is NaN too)
  }
  for (int i = 2; i < 4; ++i)
    v.n[i] = quick_root(quick_dot(v.a[i][0], v.a[i][1], v.a[i][2], v.a[i][0], v.a[i][1], v.a[i][2]));
  uint32_t n3 = 0, n4 = 0;
  for (int k = 0; k < 12; ++k) {
    const uint32_t b = quick_magnitude(m[k]);
    n3 = b > n3 ? b : n3;
  }
  for (int k = 12; k < 16; ++k) {
    const uint32_t b = quick_magnitude(m[k]);
    n4 = b > n4 ? b : n4;
  }
  // (2^56 and above, and below 2^-47, where 2^-90 n3 would not cover underflow)
  const float f3 = n3 >= 0x5b800000u || n3 < 0x28000000u ? __builtin_inff() : __builtin_bit_cast(float, n3);
  const float f4 = n4 >= 0x5b800000u ? __builtin_inff() : __builtin_bit_cast(float, n4);
  v.n34[0][0] = 1.25f * f3;
  v.n34[0][1] = 1.25f * f4;
  v.n34[1][0] = 0.625f * f3;
  v.n34[1][1] = 0.625f * f4;
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

// out: the view's four outputs at the object's centre; bound: r n[i] + eps.  For
// `visible`, in place of eps itself the smaller bound of z + w and w - z serves: of
// one of them the norm is small wherever near and far plane lie apart.
template <class M, class Less>
DPC_HD QuickResult<M> quick_decide(const float (&out)[4], const float (&bound)[4], Less&& less)
{
  const float ax = __builtin_fabsf(out[0]), ay = __builtin_fabsf(out[1]), l = out[2], h = out[3];
  float inf = __builtin_inff();
#ifdef __HIP_DEVICE_COMPILE__
  asm("" : "+s"(inf));  // (the compiler would take the medians for a maximum and minima)
#endif
  const float far = quick_med3(ax, ay, inf), near = quick_med3(l, h, -inf), eps = quick_med3(bound[2], bound[3], -inf);
  const float w = l + h, aw = __builtin_fabsf(w);
  QuickResult<M> r;
  r.visible = less(far, quick_fma(-2.0f, eps, w)) & less(eps, near);
  r.culled = less(aw + bound[0], ax) | less(aw + bound[1], ay) | less(bound[2], -l) |
             (less(bound[3], -h) & less(bound[2], l));
  return r;
}

// The outputs and bounds of one object and view.  The device computes them with
// matrix instructions that add one product after the other, fused, in this order.
template <class M, class Less>
DPC_HD QuickResult<M> quick_test(const QuickObj& q, const QuickView& v, Less&& less)
{
  float out[4], bound[4];
  for (int i = 0; i < 4; ++i) {
    out[i] = quick_fma(q.cw, v.a[i][3], quick_fma(q.cz, v.a[i][2], quick_fma(q.cy, v.a[i][1], q.cx * v.a[i][0])));
    bound[i] = quick_fma(q.sw, v.n34[i / 2][1], quick_fma(q.s3, v.n34[i / 2][0], q.r * v.n[i]));
  }
  return quick_decide<M>(out, bound, less);
}

}  // namespace dpc
