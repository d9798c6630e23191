// Shared declarations of the multi-step window kernels (wdy_span.hip).
#pragma once

#include "wdy_internal.h"

namespace wdy {

// Words of the reports windows make with atomics; a window uses the word of
// its number.  (With one word for all, the atomics of a launch took up to
// 70 us: longer than its steps.)
constexpr u32 SPAN_SLOTS = 64;
constexpr u32 SPAN_STAT_INIT = 0x7f000000u;  // no window has reported

// Arguments of one launch: K leapfrog steps of one simulation whose sheets
// are stored in sorted order (position, then sheet index).
struct SpanArgs {
  u32 n, T, H, nwin, K;
  const u64 *kin;
  const double *vin;
  const i32 *iin;
  const double *min;  // unequal masses only, like mout, cin, cout
  const u64 *cin;     // fixed-point mass below each sheet
  u64 *kout;
  double *vout;
  i32 *iout;
  double *mout;
  u64 *cout;
  double pre, h, hlast;  // drift before the first force; step; last drift
  double mq, totmass, omega2, fscale, finv;  // omega2: 0 without the term
  double amax0, amax1;  // |acceleration| <= amax0 + amax1 * |x|
  ExtForce ext;
  double t;              // force time of the first step
  const u64 *vmax_in;    // [SPAN_SLOTS] bits of the largest |v| of the state read
  u64 *vmax_out;         // of the state written (cleared by an earlier launch)
  u64 *vmax_clr;         // cleared for the next launch
  u32 *stat;             // [SPAN_SLOTS] float bits of the smallest halo width /
                         // reach; 0: a window could not vouch for its core
  u32 *stat_host;        // one window: set to 0 if a sheet is no longer finite
                         // (pinned host memory)
  u32 *stat_clr;         // stat words of the next interval, to be reset
};

// Window shapes: one wave (WaveSort), or a workgroup (BinRank).
struct SpanShape {
  int threads, cap;
  bool bin;
};
constexpr int SPAN_NSHAPES = 10;
const SpanShape &span_shape(int i);
int span_launch(hipStream_t st, int shape, bool eq, const SpanArgs &a);

}  // namespace wdy
