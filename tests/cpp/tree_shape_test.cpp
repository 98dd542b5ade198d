// The tiles' shape that a propagation plan takes by default (tree_plan.hpp): shallow
// trees of up to 75,000 nodes, whose nodes all lie in the last pass, are cut into tiles
// of few steps, and every schedule passes the planner's own check.
#include <cstdio>
#include <vector>

#include "tree_plan.hpp"

namespace tp = dpc::tileplan;

int main()
{
  long failures = 0, trees = 0;
  const std::vector<std::vector<unsigned>> shapes = {{1000, 19}, {20, 249}, {20, 999}, {200, 24}, {200, 373}, {17, 17, 17}, {27, 27, 27},
                                                     {32, 32, 32}, {5, 5, 5, 5, 5}, {1, 74000}, {74000, 1}, {300, 1, 1, 200}};
  for (const auto& children : shapes) {
    std::vector<uint32_t> par{0};
    std::vector<uint64_t> off{1};
    uint64_t first = 0, last = 1;
    for (unsigned n : children) {
      for (uint64_t p = first; p < last; ++p) par.insert(par.end(), n, static_cast<uint32_t>(p));
      first = last;
      last = par.size();
      off.push_back(last);
    }
    const tp::Shape shape = tp::default_shape(off.back());
    const uint32_t ring = shape.threads == 256 ? 576 : 1152;
    unsigned longest = 0;
    for (const auto& st : tp::schedule(par.data(), off.data(), off.size() - 1, shape.threads, ring, 1024, 1024, 32, 32, 64, shape.last_steps)) {
      if (st.kind != tp::Step::kTiles) continue;
      const std::string why = tp::check_run(par.data(), off.data(), tp::limits_for(shape.threads, st.run.ring, shape.last_steps), st.run);
      if (!why.empty()) {
        std::printf("%s\n", why.c_str());
        ++failures;
      }
      for (size_t t = 0; t < st.run.tiles(); ++t) {
        const unsigned steps = st.run.segs[st.run.tile_seg[t]].tile_steps;
        longest = steps > longest ? steps : longest;
      }
    }
    // a step of the last pass, the ancestors (256 at most in these), and what a step's end leaves over
    if (longest > 3) {
      std::printf("%llu slots, %zu passes: %u steps\n", static_cast<unsigned long long>(off.back()), children.size(), longest);
      ++failures;
    }
    ++trees;
  }
  if (tp::default_shape(75000).last_steps != 1 || tp::default_shape(75001).last_steps != 4) ++failures;
  std::printf("tree shape: %ld trees, %ld failures\n", trees, failures);
  return failures ? 1 : 0;
}
