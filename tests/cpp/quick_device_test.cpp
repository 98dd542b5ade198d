// The quick visibility test (pipeline_amd/csrc/quick_cull.hpp) in the form that the
// device runs, whose medians drop a NaN operand, against the oracle's exact test, on
// the CPU: every kind of operand that its bound does not cover, alone and together, in
// an object and in a view.  Whatever it decides has to be the oracle's answer.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>

#include "oracle.h"
#include "quick_cull.hpp"

namespace {

struct V4 {
  float x, y, z, w;
};

constexpr float kInf = std::numeric_limits<float>::infinity();
const float kNaN = std::numeric_limits<float>::quiet_NaN();
const float kOdd[] = {0.0f, -0.0f, 1e-45f, 0x1p-126f, 0x1p-47f, 0x1p-48f, 0x1p55f, 0x1p56f, 0x1p59f, 0x1p60f, -0x1p63f, 0x1p64f,
                      -0x1p100f, 3e38f, -3e38f, kInf, -kInf, kNaN};
constexpr int kOdds = static_cast<int>(sizeof kOdd / sizeof kOdd[0]);

std::mt19937_64 rng(20270113);
int pick(int n) { return static_cast<int>(rng() % static_cast<unsigned>(n)); }
float uniform(float lo, float hi) { return std::uniform_real_distribution<float>(lo, hi)(rng); }

long failures = 0, decided = 0, pairs = 0;

void check(const float obb[16], const float vp[16])
{
  V4 v[4];
  std::memcpy(v, obb, sizeof v);
  const auto r = dpc::quick_test<bool>(dpc::quick_obj(v[0], v[1], v[2], v[3]), dpc::quick_view(vp),
                                       [](float a, float b) { return a < b; });
  const bool want = orc_is_visible_obb(vp, obb) != 0;
  ++pairs;
  decided += r.visible || r.culled;
  if ((r.visible && !want) || (r.culled && want)) {
    if (++failures <= 10) std::printf("quick says %s, the oracle %s\n", r.visible ? "visible" : "culled", want ? "visible" : "culled");
  }
}

void medians()
{
  const float v[] = {-kInf, -2.0f, 0.0f, 3.0f, kInf};
  for (float a : v)
    for (float b : v) {
      if (dpc::quick_med3(a, b, kInf) != std::fmax(a, b) || dpc::quick_med3(a, b, -kInf) != std::fmin(a, b)) ++failures;
      if (dpc::quick_med3(kNaN, a, b) != std::fmin(a, b) || dpc::quick_med3(a, kNaN, b) != std::fmin(a, b)) ++failures;
    }
  if (dpc::quick_med3(kNaN, kNaN, kInf) != kInf || dpc::quick_med3(kNaN, kNaN, -kInf) != -kInf) ++failures;
}

}  // namespace

int main()
{
  medians();
  // objects around the eye of an orthographic view, or of a perspective one: most are
  // visible before their odd values, and all that the medians decide is `visible`
  for (int k = 0; k < 6000000; ++k) {
    float vp[16] = {}, o[16] = {};
    if (pick(2)) {
      vp[0] = vp[5] = 0.01f;
      vp[10] = -0.01f;
      vp[15] = 1.0f;
    } else {
      vp[0] = vp[5] = 1.0f;
      vp[10] = -1.0f;
      vp[11] = -1.0f;
      vp[14] = -0.2f;
    }
    if (pick(2))
      for (float& m : vp) m += uniform(-0.001f, 0.001f);
    for (int c = 0; c < 3; ++c) o[c] = uniform(-5, 5);
    o[2] -= 20;
    o[3] = 1.0f;
    for (int e = 1; e < 4; ++e)
      for (int c = 0; c < 3; ++c) o[4 * e + c] = uniform(-2, 2);
    const int n = pick(9), where = pick(4);  // in one column, one row, the object or anywhere
    const int at = pick(4);
    for (int i = 0; i < n; ++i) {
      const float odd = kOdd[pick(kOdds)];
      if (where == 0) vp[4 * pick(4) + at] = odd;
      else if (where == 1) vp[4 * at + pick(4)] = odd;
      else if (where == 2) o[pick(16)] = odd;
      else (pick(2) ? o : vp)[pick(16)] = odd;
    }
    check(o, vp);
  }
  std::printf("quick cull, device form: %ld of %ld pairs decided\nquick cull, device form: %ld failures\n", decided, pairs, failures);
  return failures ? 1 : 0;
}
