// Sorting of nearly sorted sheets on chip, for kernels that run several
// leapfrog steps without going back to memory.  Both forms are exact (positions,
// then sheet index) for finite positions, BinRank for a window that was in order
// when it was loaded.  Otherwise a place may be taken twice and another by no
// sheet, always inside the window: callers find out and do it again another way.
//
// * WaveSheets: one wave holds up to 64 * PER sheets in registers, PER
//   consecutive ranks per lane, and re-sorts them after each drift by odd-even
//   transposition, ending as soon as the order is right: no LDS, no barrier,
//   ~10 instructions per sheet and rank of displacement.  For steps that move
//   sheets a few ranks.
// * BinRank: a workgroup's sheets stay in the registers of the threads that
//   loaded them and only their ranks change: a counting pass over position
//   bins in LDS, then each sheet ranks itself in its bin.  Its cost does not
//   depend on the displacement.
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

  // the next lane's x[0], and the smallest step from one rank to the next in
  // d: positive when every pair is in order (NaN, at the ends, does not count)
  __device__ __forceinline__ double step_min(double &d) const {
    const double xn = dpp_mov_f64<DPP_WAVE_SHL1>(__builtin_nan(""), x[0]);
    d = xn - x[PER - 1];
#pragma unroll
    for (int q = 0; q + 1 < PER; ++q) d = fmin(d, x[q + 1] - x[q]);
    return xn;
  }
  __device__ __forceinline__ void sort_rounds(double xn) {
    double d;
    do {
      round<false>(xn);
      xn = step_min(d);
    } while (__ballot(d < 0.0) != 0);
    if (__ballot(d == 0.0) == 0) return;
    // in order but for exactly equal positions
    bool o;
    do {
      xn = dpp_mov_f64<DPP_WAVE_SHL1>(__builtin_nan(""), x[0]);
      round<true>(xn);
      xn = dpp_mov_f64<DPP_WAVE_SHL1>(__builtin_nan(""), x[0]);
      const i32 in = (i32)dpp_mov<DPP_WAVE_SHL1, 0xf>(0u, (u32)id[0]);
      o = after(x[PER - 1], id[PER - 1], xn, in);
#pragma unroll
      for (int q = 0; q + 1 < PER; ++q) o = o || after(x[q], id[q], x[q + 1], id[q + 1]);
    } while (__ballot(o) != 0);
  }

  // sorts the wave's sheets; true when anything may have moved.  (One forward
  // branch where nothing moves: taken branches, ~30 cycles each, were half of
  // a step of three sheets: 254 -> 138.)
  __device__ __forceinline__ bool sort() {
    static_assert(PER % 2 == 0, "pairs inside the lanes");
    double d;
    const double xn = step_min(d);
    const bool move = __ballot(d <= 0.0) != 0;
    if (__builtin_expect(move, 0)) sort_rounds(xn);
    return move;
  }
};

// ---- BinRank -----------------------------------------------------------------
template <int WT_, int PER_>
struct RankShape {
  static constexpr int WT = WT_, PER = PER_, CAP = WT_ * PER_, NWAVE = WT_ / 64;
};

// Bins: the window is cut into BIN_SEGS segments by rank, finer towards its
// ends, and each segment's range of positions (when the launch starts) is cut
// into as many bins as it has of them: outliers and tails take a few bins and
// leave the rest theirs.  (With bins of one width over the window, 1000 sheets
// of which two lie far out shared a few bins: 110 us a step.)  A thread keeps
// its sheets' segments; they seldom change.  A window whose segments are about
// as dense as each other takes bins of one width, which costs a quarter less.
constexpr int BIN_SEGS = 16;
struct BinSeg {
  double lo, scale, next;  // its first position, bins per length, the next's first
  u32 base, cnt;
};
// the start of segment k, out of 256
__device__ __forceinline__ u32 bin_seg_start(u32 k) {
  const u32 j = k <= 8 ? k : 16 - k;  // 0 1 4 16 32 56 80 104 128
  const u32 e = j == 0 ? 0u : j <= 3 ? 1u << (2 * (j - 1)) : 24 * j - 64;
  return k <= 8 ? e : 256 - e;
}

// LDS: positions and sheet indices in bin order, two sets of bin counters (one
// is cleared while the other is used) and, with unequal masses, the masses in
// rank order, then the mass below each rank: 20 and 28 B per sheet.
//
// A step is a chain of four barriers, seven with unequal masses; with every window on a CU of its
// own their latency bounds it (256 sheets 0.85 us, 1024 1.2, 4096 3.6), else the
// CUs' issue rate, ~100 instructions per sheet and step.  Unequal masses go to
// LDS in the new order after the ranking (4096 sheets: 5.4 us; with a prefix over
// the bins' slots and the mass summed while ranking, 6.5).  A sheet is compared
// with its bin's positions themselves: with the places in the bin, rounded to
// 32 bits and masked at the bin's end, a step took a quarter longer, and the
// LDS held 4096 sheets where it now holds 7168.
template <class SH, bool MASS>
struct BinRank {
  static constexpr int CAP = SH::CAP, PER = SH::PER, WT = SH::WT, NWAVE = SH::NWAVE;
  static constexpr int NB = CAP, WPT = NB / WT;  // bins, bins per thread
  static_assert(NWAVE <= 16, "one row of lanes scans the waves' totals");
  static constexpr int PAD = 4;  // slots read past the last sheet
  static constexpr size_t BYTES = 8ull * (CAP + PAD) +
                                  (MASS ? 8ull * CAP : 0ull) +
                                  16ull * 16 + 4ull * CAP +
                                  8ull * (NB + 1) + (BIN_SEGS + 1) * sizeof(BinSeg);
  static_assert(NB % 256 == 0, "whole bins in every segment");
  double *xs;
  u64 *ms;  // masses in rank order, then the mass below each rank
  u64 *red, *redm;
  i32 *id;
  u32 *bins;  // [2][NB + 1]: one more, the end of the last bin
  BinSeg *seg;  // [BIN_SEGS], and the window as one
  double x0, scale;  // of the window as one segment
  bool segs;         // else one segment
  u32 s;
  u32 g[PER];  // the sheets' segments

  // kin: the keys of the window's w sheets, in order; d, d1: how far a sheet may
  // move in the launch and in one of its steps.  The segments go by rank as if there were eL ranks more in a
  // length d below the first sheet and eR in d above the last (each 0 or the
  // same): where the sheets go that leave the window.
  __device__ BinRank(u64 *base, u32 w, const u64 *kin, u32 eL, u32 eR, double d,
                     double d1) {
    seg = (BinSeg *)base;
    xs = (double *)(seg + BIN_SEGS + 1);
    ms = (u64 *)(xs + CAP + PAD);
    red = MASS ? ms + CAP : ms;
    redm = red + 16;
    id = (i32 *)(redm + 16);
    bins = (u32 *)(id + CAP);
    s = 0;
    clear(0);
    const u32 t = threadIdx.x;
    if (t < BIN_SEGS) {
      const u32 f0 = bin_seg_start(t), f1 = bin_seg_start(t + 1);
      BinSeg q;
      // (in signed numbers: the compiler here takes a `u < eL ? 0 : u - eL`
      // inside a min() to mean that u >= eL)
      const u32 e = max(eL, eR);
      const double per = e ? d / (double)e : 0.0;
      auto at = [&](u32 u) {
        const i32 r = (i32)u - (i32)eL, over = r - (i32)w;
        const double x = decode_pos(kin[max(0, min(r, (i32)w - 1))]);
        return x + per * (double)(r < 0 ? r : max(over, 0));
      };
      const u32 tot = eL + w + eR;
      q.lo = at(tot * f0 >> 8);
      const double hi = at(tot * f1 >> 8);
      q.next = t + 1 < BIN_SEGS ? hi : __builtin_inf();
      q.base = (u32)NB / 256 * f0;
      q.cnt = (u32)NB / 256 * (f1 - f0);
      const double range = hi - q.lo;
      q.scale = range > 1.0e-300 && range < 1.0e300 ? (double)q.cnt / range : 0.0;
      seg[t] = q;
      // one segment does while none of these would have six times its share
      // of sheets per bin
      const double first = at(0), last = at(tot), all = last - first;
      const bool full = !((double)q.cnt * all <= 6.0 * (double)NB * range);
      const u32 any = __ballot(full) != 0 ? 1u : 0u;
      // sheets that a step moves further than they are apart (all of them may
      // start at one place, and so in one bin: 6144 of them took 45 ms an interval
      // of 20 steps, now 0.4): over where they can go
      const bool apart = e > 0 || !(all < 2.0 * d1);
      if (t == 0) {
        const double to = apart ? all : all + 2.0 * d;
        q.lo = apart ? first : first - d;
        q.scale = to > 1.0e-300 && to < 1.0e300 ? (double)NB / to : 0.0;
        q.base = apart ? any : 0u;
        seg[BIN_SEGS] = q;
      }
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const u32 e = i * WT + t;
      g[i] = 0;
#pragma unroll
      for (u32 k = 1; k < BIN_SEGS; ++k)
        g[i] += e + eL >= (eL + w + eR) * bin_seg_start(k) >> 8 ? 1u : 0u;
    }
    if (threadIdx.x < 16) red[threadIdx.x] = redm[threadIdx.x] = 0;
    if (threadIdx.x < PAD) xs[w + threadIdx.x] = __builtin_inf();
    __syncthreads();
    x0 = seg[BIN_SEGS].lo;
    scale = seg[BIN_SEGS].scale;
    segs = __builtin_amdgcn_readfirstlane(seg[BIN_SEGS].base) != 0;
  }
  __device__ __forceinline__ void clear(u32 b) {
    const u32 t = threadIdx.x;
#pragma unroll
    for (int q = 0; q < WPT; ++q) {
      bins[b * (NB + 1) + q * WT + t] = 0;
    }
  }
  // exclusive prefix of one value per thread over the workgroup; one barrier
  template <class T>
  __device__ __forceinline__ T scan_excl(T v, u64 *r) {
    const u32 lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    const T inc = wave_incl_add(v);
    if (lane == 63u) r[wv] = inc;
    return inc - v;
  }
  // the total of the waves before this one (after the barrier)
  template <class T>
  __device__ __forceinline__ T waves_before(const u64 *r) {
    const u32 lane = threadIdx.x & 63u;
    const u32 wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    T x = (T)r[lane & 15u];
    x += dpp_mov<DPP_SHR1, 0xf>((T)0, x);
    x += dpp_mov<DPP_SHR2, 0xf>((T)0, x);
    if (NWAVE > 4) x += dpp_mov<DPP_SHR4, 0xf>((T)0, x);
    if (NWAVE > 8) x += dpp_mov<DPP_SHR8, 0xf>((T)0, x);
    // (lane wv - 1 holds the inclusive total of wave wv - 1)
    const u32 src = wv ? wv - 1u : 0u;
    T y;
    if constexpr (sizeof(T) == 8)
      y = ((T)(u32)__builtin_amdgcn_readlane((int)(x >> 32), src) << 32) |
          (u32)__builtin_amdgcn_readlane((int)x, src);
    else
      y = (u32)__builtin_amdgcn_readlane((int)x, src);
    return wv ? y : (T)0;
  }

  // Sheets i * WT + t < w of this thread move from x[i] to x[i] + p[i]; r[i]
  // becomes the sheet's rank and c[i] the mass below it, base included.
  // SEGS: as `segs` says.
  template <bool SEGS>
  __device__ __forceinline__ void step(u32 w, double (&x)[PER],
                                       const double (&p)[PER], u32 (&r)[PER],
                                       const i32 (&ids)[PER],
                                       const u64 (&m)[PER], u64 (&c)[PER],
                                       u64 base) {
    const u32 t = threadIdx.x;
    u32 *const bn = bins + (s & 1u) * (NB + 1);
    u32 b[PER], slot[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      slot[i] = 0;
      x[i] = x[i] + p[i];
      double lo = x0, sc = scale;
      u32 first = 0, cnt = NB;
      if constexpr (SEGS) {
        BinSeg sg = seg[g[i]];
        if ((x[i] < sg.lo && g[i] > 0) || x[i] >= sg.next) {
          while (g[i] > 0 && x[i] < seg[g[i]].lo) --g[i];
          while (g[i] < BIN_SEGS - 1 && x[i] >= seg[g[i]].next) ++g[i];
          sg = seg[g[i]];
        }
        lo = sg.lo;
        sc = sg.scale;
        first = sg.base;
        cnt = sg.cnt;
      }
      // non-decreasing in x; below the first segment's start: with its first; a
      // segment's last bin also takes what rounds beyond it
      const double q = fmin(fmax((x[i] - lo) * sc, 0.0), (double)cnt);
      b[i] = first + min((u32)q, cnt - 1);
      if (i * WT + t < w) {
        slot[i] = atomicAdd(&bn[b[i]], 1u);  // its place in the bin
      }
    }
    __syncthreads();
    {
      u32 loc[WPT];
      u32 sum = 0;
#pragma unroll
      for (int q = 0; q < WPT; ++q) {
        loc[q] = bn[t * WPT + q];
        sum += loc[q];
      }
      u32 run = scan_excl<u32>(sum, red);
      __syncthreads();
      run += waves_before<u32>(red);
#pragma unroll
      for (int q = 0; q < WPT; ++q) {
        bn[t * WPT + q] = run;
        run += loc[q];
      }
      if (t == 0) bn[NB] = w;
    }
    __syncthreads();
    u32 lo[PER], hi[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      lo[i] = hi[i] = 0;
      if (i * WT + t < w) {
        lo[i] = bn[b[i]];
        hi[i] = bn[b[i] + 1u];
        slot[i] += lo[i];
        xs[slot[i]] = x[i];
        id[slot[i]] = ids[i];
      }
    }
    clear((s & 1u) ^ 1u);
    ++s;
    __syncthreads();
    // Rank inside the bin: the sheets of the bin below.  The first PAD slots are
    // read at once without a look at where the bin ends: what lies beyond is in
    // a later bin, so above.
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      u32 k = lo[i], eq = 0;
      double y[PAD];
#pragma unroll
      for (int q = 0; q < PAD; ++q) y[q] = xs[lo[i] + q];
#pragma unroll
      for (int q = 0; q < PAD; ++q) {
        k += y[q] < x[i] ? 1u : 0u;
        eq += y[q] == x[i] ? 1u : 0u;
      }
      for (u32 a = lo[i] + PAD; a < hi[i]; ++a) {
        const double z = xs[a];
        k += z < x[i] ? 1u : 0u;
        eq += z == x[i] ? 1u : 0u;
      }
      if (eq > 1) {  // exactly equal positions go by sheet index
        for (u32 a = lo[i]; a < hi[i]; ++a)
          if (xs[a] == x[i] && id[a] < ids[i]) k += 1;
      }
      r[i] = k;
    }
    if constexpr (MASS) {  // the masses in the new order, then what is below
#pragma unroll
      for (int i = 0; i < PER; ++i)
        if (i * WT + t < w) ms[r[i]] = m[i];
      __syncthreads();
      u64 lm[PER], sum = 0;
#pragma unroll
      for (int q = 0; q < PER; ++q) {
        lm[q] = t * PER + q < w ? ms[t * PER + q] : 0ull;
        sum += lm[q];
      }
      u64 run = scan_excl<u64>(sum, redm);
      __syncthreads();
      run += base + waves_before<u64>(redm);
#pragma unroll
      for (int q = 0; q < PER; ++q) {
        ms[t * PER + q] = run;
        run += lm[q];
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < PER; ++i) c[i] = ms[r[i]];
    }
  }
};

}  // namespace wdy
