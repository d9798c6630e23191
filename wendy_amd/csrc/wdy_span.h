// Shared declarations of the multi-step window kernels (wdy_span.hip).
#pragma once

#include <vector>

#include "wdy_batch.h"
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
  u32 id0;  // the simulation's first sheet index
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
  double *xo, *vo;  // de-sorted positions and velocities as well (or null)
  double pre, h, hlast;  // drift before the first force; step; last drift
  double mq, totmass, omega2, fscale, finv;  // omega2: 0 without the term
  double amax0, amax1;  // |acceleration| <= amax0 + amax1 * |x|
  ExtForce ext;
  double t;              // force time of the first step
  // [SPAN_SLOTS] bits of the largest |v| of the state read, of the state
  // written (cleared by an earlier launch), and words cleared for the next
  // launch; all null where one window takes the whole simulation for good
  const u64 *vmax_in;
  u64 *vmax_out;
  u64 *vmax_clr;
  u32 *stat;             // [SPAN_SLOTS] float bits of the smallest halo width /
                         // reach, with several windows (or null)
  u32 *stat_clr;         // stat words of the next interval, to be reset (or null)
  u32 *stat_host;        // copies of stat in pinned host memory (or null)
  // set to fail_value = 1 + the launch's number if a window could not vouch for its
  // core, or a sheet is no longer finite: what the launch wrote may then be out
  // of order or lack sheets, and the later launches, for which that is the input,
  // leave (span_leaves)
  u32 *fail;
  u32 fail_value;
  u32 *fail_host;        // set too, in pinned host memory (or null)
};

// Window shapes: one wave (WaveSheets), or a workgroup (BinRank).
struct SpanShape {
  int threads, cap, cap_un;  // sheets, with equal and with unequal masses
  bool bin;
};
constexpr int SPAN_NSHAPES = 10;
int span_launch(hipStream_t st, int shape, bool eq, const SpanArgs &a);

// ---- many simulations per launch (a batch) -----------------------------------
// What the device keeps and reports of a batch's simulations.
struct SpanMany {
  u64 *cf[2];   // fixed-point mass below each sheet, per set (null: none unequal)
  u64 *vmax;    // [vslot][3][SPAN_SLOTS]: the word sets of SpanArgs
  u32 *fail;    // [simulation] 0, or 1 + the launch of the interval that failed
  u32 *intact;  // [simulation] pinned: 0 once a window failed (multi-window ones)
  double *info; // [simulation][SPAN_INFO] pinned: SPAN_NW widths, max |v|, max |x|
};
constexpr u32 SPAN_NW = 10;
constexpr u32 SPAN_INFO = 12;
// Sets shape and each simulation's T, H, nwin, K, L, vslot for intervals of
// nleap steps of h from what the device reported; L = 0 where the windows do
// not hold.  reach[i] scales simulation i's halo.
void span_many_plan(std::vector<BatchDesc> &d, const double *info,
                    const std::vector<double> &reach, double h, int nleap, int *shape);
// Launch q of interval iv since the plan; list: (simulation, window) of nwin
// windows, those of simulations with equal masses before the others.
int span_many_launch(hipStream_t st, int shape, const BatchDesc *descs,
                     const uint2 *list, u32 neq, u32 nun, const BatchArrays &arr,
                     const SpanMany &m, u32 q, u32 iv);

}  // namespace wdy
