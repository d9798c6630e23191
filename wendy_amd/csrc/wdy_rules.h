// Rules of the host code that decide how kernels are launched, in plain C++:
// they are tested without a GPU.
#pragma once

#include <algorithm>
#include <cstdint>

namespace wdy {

// How the pair sums of ny points over n sheets are launched, `block` threads to
// a block: enough blocks to fill the GPU, stretches no shorter than 4 sheets per
// thread and at most 128 of them (one thread adds up their sums).  Few points
// (under 4096) take 4 to a block: their sheets come from L2 anyway, and 16
// would leave too few blocks.  No sheets are one empty stretch.
struct PairPlan {
  uint32_t qp, splits, per;  // points per block, stretches, sheets in each
};
inline PairPlan pair_plan(uint32_t n, uint32_t ny, uint32_t block) {
  PairPlan p;
  p.qp = ny >= 4096 ? 16 : 4;
  const uint32_t bx = (ny + p.qp - 1) / p.qp;
  const uint32_t most = std::min<uint32_t>(128, std::max<uint32_t>(1, n / (4 * block)));
  p.splits = std::min(most, std::max<uint32_t>(1, (1024 + bx - 1) / bx));
  p.per = std::max<uint32_t>(1, (n + p.splits - 1) / p.splits);
  p.splits = std::max<uint32_t>(1, (n + p.per - 1) / p.per);
  return p;
}

// Whether a window of launch q leaves its simulation alone, `word` being the
// simulation's: 0, or 1 + the launch in which a window could not vouch for its
// core.  Only an earlier launch's failure counts: every wave of every window of
// this launch then decides alike, also those that read the word after another
// window of the launch has set it.  (What this launch writes is not read: the
// interval is redone from what it was given.)
constexpr bool span_leaves(uint32_t word, uint32_t q) { return word != 0 && word != q + 1; }

// The launches of a simulation are numbered in a ring, so that 1 + the number is
// never 0.  launch_of: the place of launch `q` in `count` launches from `first`
// on, or -1.
constexpr uint32_t LAUNCH_RING = 0xffffffffu;
constexpr uint32_t next_launch(uint32_t q) { return q + 1 == LAUNCH_RING ? 0 : q + 1; }
constexpr int64_t launch_of(uint32_t q, uint32_t first, uint32_t count) {
  const uint64_t d = ((uint64_t)q + LAUNCH_RING - first) % LAUNCH_RING;
  return d < count ? (int64_t)d : -1;
}

// The ways of cutting an interval of nleap steps into launches that a plan tries:
// fn(K, launches) with K steps a launch, for every number of launches up to 8,
// then for numbers a quarter apart.  (In 64 bits: nleap may be any positive int.)
template <class F>
inline void each_split(int nleap, F fn) {
  for (int64_t L = 1; L <= nleap; L = L < 8 ? L + 1 : L + L / 4) {
    const int64_t K = (nleap + L - 1) / L;
    fn((int)K, (int)((nleap + K - 1) / K));
  }
}

}  // namespace wdy
