// Sorting of nearly sorted sheets on chip, for kernels that run several
// leapfrog steps without going back to memory: one wave holds up to 64 * PER
// sheets in registers, PER consecutive ranks per lane, and re-sorts them after
// each drift by odd-even transposition, ending as soon as the order is right:
// no LDS, no barrier, ~10 instructions per sheet and rank of displacement.
// Exact for any input (positions, then sheet index).
#pragma once

#include "wdy_lds.h"

namespace wdy {

// the wave's minimum, in every lane
__device__ __forceinline__ u32 wave_min_u32(u32 x) {
  u32 y;
  y = dpp_mov<DPP_SHR1, 0xf>(~0u, x); x = y < x ? y : x;
  y = dpp_mov<DPP_SHR2, 0xf>(~0u, x); x = y < x ? y : x;
  y = dpp_mov<DPP_SHR4, 0xf>(~0u, x); x = y < x ? y : x;
  y = dpp_mov<DPP_SHR8, 0xf>(~0u, x); x = y < x ? y : x;
  y = dpp_mov<DPP_BCAST15, 0xa>(~0u, x); x = y < x ? y : x;
  y = dpp_mov<DPP_BCAST31, 0xc>(~0u, x); x = y < x ? y : x;
  return wave_last(x);
}

// lane i gets lane i+1's (SHL) or lane i-1's (SHR) value across the whole
// wave; the last (first) lane keeps `old`
constexpr int DPP_WAVE_SHL1 = 0x130, DPP_WAVE_SHR1 = 0x138;

template <int CTRL>
__device__ __forceinline__ double dpp_mov_f64(double old, double x) {
  const u64 r = dpp_mov<CTRL, 0xf>((u64)__double_as_longlong(old),
                                   (u64)__double_as_longlong(x));
  return __longlong_as_double((long long)r);
}

// (x, i) comes after (y, j); false when either position is NaN
__device__ __forceinline__ bool after(double x, i32 i, double y, i32 j) {
  return x > y || (x == y && i > j);
}

// The wave's sheets: rank lane * PER + q in x[q], v[q], id[q] and, with MASS,
// m[q] and mf[q] (its mass as it is and in fixed point).  Slots past the last
// sheet hold NaN positions, which never move.
template <int PER, bool MASS>
struct WaveSheets {
  double x[PER], v[PER], m[MASS ? PER : 1];
  u64 mf[MASS ? PER : 1];
  i32 id[PER];

  __device__ __forceinline__ void swap_if(bool s, int a, int b) {
    const double xa = x[a], va = v[a];
    const i32 ia = id[a];
    x[a] = s ? x[b] : xa;
    x[b] = s ? xa : x[b];
    v[a] = s ? v[b] : va;
    v[b] = s ? va : v[b];
    id[a] = s ? id[b] : ia;
    id[b] = s ? ia : id[b];
    if constexpr (MASS) {
      const double ma = m[a];
      const u64 fa = mf[a];
      m[a] = s ? m[b] : ma;
      m[b] = s ? ma : m[b];
      mf[a] = s ? mf[b] : fa;
      mf[b] = s ? fa : mf[b];
    }
  }

  // one double round of odd-even transposition: the lanes' boundaries, then
  // the pairs inside the lanes.  TIES: equal positions go by sheet index
  // (else they stay as they are).  xn: the next lane's x[0].
  template <bool TIES>
  __device__ __forceinline__ void round(double xn) {
    const double nan = __builtin_nan("");
    auto wrong = [](double xa, i32 ia, double xb, i32 ib) {
      return TIES ? after(xa, ia, xb, ib) : xa > xb;
    };
    const double xp = dpp_mov_f64<DPP_WAVE_SHR1>(nan, x[PER - 1]);
    const i32 in = (i32)dpp_mov<DPP_WAVE_SHL1, 0xf>(0u, (u32)id[0]);
    const i32 ip = (i32)dpp_mov<DPP_WAVE_SHR1, 0xf>(0u, (u32)id[PER - 1]);
    const bool hi = wrong(x[PER - 1], id[PER - 1], xn, in);
    const bool lo = wrong(xp, ip, x[0], id[0]);
    const double vn = dpp_mov_f64<DPP_WAVE_SHL1>(0.0, v[0]);
    const double vp = dpp_mov_f64<DPP_WAVE_SHR1>(0.0, v[PER - 1]);
    if constexpr (MASS) {
      const double mn = dpp_mov_f64<DPP_WAVE_SHL1>(0.0, m[0]);
      const double mp = dpp_mov_f64<DPP_WAVE_SHR1>(0.0, m[PER - 1]);
      const u64 fn = dpp_mov<DPP_WAVE_SHL1, 0xf>((u64)0, mf[0]);
      const u64 fp = dpp_mov<DPP_WAVE_SHR1, 0xf>((u64)0, mf[PER - 1]);
      m[PER - 1] = hi ? mn : m[PER - 1];
      m[0] = lo ? mp : m[0];
      mf[PER - 1] = hi ? fn : mf[PER - 1];
      mf[0] = lo ? fp : mf[0];
    }
    x[PER - 1] = hi ? xn : x[PER - 1];
    x[0] = lo ? xp : x[0];
    v[PER - 1] = hi ? vn : v[PER - 1];
    v[0] = lo ? vp : v[0];
    id[PER - 1] = hi ? in : id[PER - 1];
    id[0] = lo ? ip : id[0];
#pragma unroll
    for (int q = 1; q + 1 < PER; q += 2)
      swap_if(wrong(x[q], id[q], x[q + 1], id[q + 1]), q, q + 1);
#pragma unroll
    for (int q = 0; q + 1 < PER; q += 2)
      swap_if(wrong(x[q], id[q], x[q + 1], id[q + 1]), q, q + 1);
  }

  // sorts the wave's sheets; true when anything may have moved
  __device__ __forceinline__ bool sort() {
    static_assert(PER % 2 == 0, "pairs inside the lanes");
    const double nan = __builtin_nan("");
    bool moved = false;
    while (true) {
      // the smallest step from one rank to the next: positive when every
      // pair is in order (NaN, at the ends, does not count)
      const double xn = dpp_mov_f64<DPP_WAVE_SHL1>(nan, x[0]);
      double d = xn - x[PER - 1];
#pragma unroll
      for (int q = 0; q + 1 < PER; ++q) d = fmin(d, x[q + 1] - x[q]);
      if (__builtin_expect(__ballot(d <= 0.0) == 0, 1)) return moved;
      moved = true;
      if (__ballot(d < 0.0) == 0) break;
      round<false>(xn);
    }
    // in order but for exactly equal positions
    while (true) {
      const double xn = dpp_mov_f64<DPP_WAVE_SHL1>(nan, x[0]);
      const i32 in = (i32)dpp_mov<DPP_WAVE_SHL1, 0xf>(0u, (u32)id[0]);
      bool o = after(x[PER - 1], id[PER - 1], xn, in);
#pragma unroll
      for (int q = 0; q + 1 < PER; ++q) o = o || after(x[q], id[q], x[q + 1], id[q + 1]);
      if (__ballot(o) == 0) return moved;
      round<true>(xn);
    }
  }
};

}  // namespace wdy
