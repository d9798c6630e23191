// Several leapfrog steps per launch for medium simulations.
//
// The sheets are kept in sorted order; a launch cuts them into windows of T
// consecutive ranks (the core) with H more on each side (the halo), and every
// window runs K steps on its sheets by itself: the force on a sheet is its
// rank, or the mass below it, and the ranks outside a window do not change
// until a sheet has crossed its halo.  Windows prove on the device that none
// could have (Reach below); a window that cannot marks the simulation, whose
// later launches leave, and the host, which sees the verdict when it settles,
// redoes the interval from the set it started from, with wider halos.
//
// What bounds the one-step kernel at these sizes is not the GPU's rates but a
// launch per step, ~12 us of dependent phases each.  Measured, us per interval
// of 20 steps of h = 2.5e-4 on the sech^2 disk, one launch per step -> windows,
// equal / unequal masses: 2^14 244 -> 30 / 270 -> 41, 2^16 267 -> 51 / 306 ->
// 66, 2^18 415 -> 98 / 485 -> 131, 2^20 870 -> 312 / 954 -> 477, 2^21 1178 -> 807
// / 1649 -> 1316.  What bounds a window is the latency of its step, ~1 us of LDS round trips and barriers
// (0.2-0.5 us for one wave), and from ~256 windows on the CUs' issue rate.
#include <algorithm>
#include <cmath>
#include <new>
#include <type_traits>

#include "wdy_rank.h"
#include "wdy_rules.h"
#include "wdy_span.h"

namespace wdy {
namespace {

__device__ __forceinline__ double bits_double(u64 b) {
  return __longlong_as_double((long long)b);
}

// What the sheets outside a window can do in one launch.  No sheet moves
// further than D: V bounds every speed (the largest now, plus K kicks of at
// most amax each, 3% to spare), and every window checks it on its own sheets.
// So outside sheets, and the ones they may have crossed, stay below xl + D or
// above xr - D, and a sheet that ends strictly between was never out of order
// with them: its rank, and so its force, was right at every step.
struct Reach {
  double xl, xr, V, D;
  u32 a, b, w, c0, c1;
  bool ok;
  float slack;
};

__device__ __forceinline__ Reach span_reach(const SpanArgs &A, const u32 j) {
  Reach R;
  R.c0 = j * A.T;
  R.c1 = min(A.n, R.c0 + A.T);
  R.a = R.c0 > A.H ? R.c0 - A.H : 0u;
  R.b = min(A.n, R.c1 + A.H);
  R.w = R.b - R.a;
  R.xl = decode_pos(A.kin[R.a]);
  R.xr = decode_pos(A.kin[R.b - 1]);
  const double xm = fmax(fabs(decode_pos(A.kin[0])), fabs(decode_pos(A.kin[A.n - 1])));
  const double amax = A.amax0 + A.amax1 * xm;  // of any sheet, all forces
  const double S = fabs(A.pre) + (double)(A.K - 1) * fabs(A.h) + fabs(A.hlast);
  const u64 vin = A.vmax_in ? wave_max(A.vmax_in[threadIdx.x & (SPAN_SLOTS - 1)]) : 0ull;
  R.V = 1.03 * (bits_double(vin) + (double)A.K * fabs(A.h) * amax);
  R.D = R.V * S * 1.0001 + (double)(A.K + 2) * 3.0e-16 * xm;
  if (A.nwin == 1) R.V = 1.7976931348623157e308;  // no outside: finite is enough
  // neighbouring windows' safe zones meet at the core boundaries
  R.ok = true;
  R.slack = 3.0e38f;
  if (R.a > 0) {
    const double d = decode_pos(A.kin[R.c0]) - R.xl;
    R.ok = d > R.D;
    R.slack = (float)(d / R.D);
  }
  if (R.b < A.n) {
    const double d = R.xr - decode_pos(A.kin[R.c1]);
    R.ok = R.ok && d > R.D;
    R.slack = fminf(R.slack, (float)(d / R.D));
  }
  if (j == 0 && threadIdx.x < SPAN_SLOTS) {
    if (A.vmax_clr) A.vmax_clr[threadIdx.x] = 0;
    if (A.stat_clr) A.stat_clr[threadIdx.x] = SPAN_STAT_INIT;
  }
  return R;
}

// Sheet of final rank r (in the whole simulation) ended at x with speed v:
// checks it and stores it if it belongs to the core.
template <bool EQ>
__device__ __forceinline__ void span_store(const SpanArgs &A, Reach &R, u32 r,
                                           double x, double v, i32 id, double m,
                                           u64 c, double &vm) {
  if (r >= R.c0 && r < R.c1) {
    R.ok = R.ok && fabs(v) <= R.V && fabs(x) < __builtin_inf() &&
           (R.a == 0 || x > R.xl + R.D) && (R.b == A.n || x < R.xr - R.D);
    if (r == R.c0 && R.a > 0) R.slack = fminf(R.slack, (float)((x - R.xl) / R.D));
    if (r + 1 == R.c1 && R.b < A.n) R.slack = fminf(R.slack, (float)((R.xr - x) / R.D));
    vm = fmax(vm, fabs(v));
    A.kout[r] = encode_pos(x);
    A.vout[r] = v;
    A.iout[r] = id;
    if (!EQ) {
      A.mout[r] = m;
      A.cout[r] = c;
    }
    if (A.xo) {
      A.xo[id] = x;
      A.vo[id] = v;
    }
  }
}

// One thread of the window reports: sb, its verdict (the float bits of its
// slack, 0: it cannot vouch for its core); vm, the bits of the core's largest
// speed.
__device__ __forceinline__ u32 span_verdict(const Reach &R) {
  return R.ok ? min(__float_as_uint(fmaxf(R.slack, 0.f)), SPAN_STAT_INIT) : 0u;
}
__device__ __forceinline__ void span_report(const SpanArgs &A, u32 j, u32 sb, u64 vm) {
  const u32 q = j & (SPAN_SLOTS - 1);
  if (sb == 0) {
    *A.fail = A.fail_value;
    if (A.fail_host) *A.fail_host = A.fail_value;
    return;
  }
  // (a stale word only costs an atomic that changes nothing; the host's copies
  // are for the next plan's halos, where a lost race does not matter)
  if (A.nwin > 1 && A.stat && sb < A.stat[q]) {
    atomicMin(A.stat + q, sb);
    if (A.stat_host) A.stat_host[q] = sb;
  }
  if (A.vmax_out && vm > A.vmax_out[q])
    atomicMax((unsigned long long *)A.vmax_out + q, (unsigned long long)vm);
}

// ---- windows of one wave ---------------------------------------------------------
template <int PER, bool EQ, bool EXT>
__device__ __forceinline__ void span_wave(const SpanArgs &A, const u32 j) {
  const u32 lane = threadIdx.x & 63u;
  Reach R = span_reach(A, j);
  WaveSheets<PER, !EQ> s;
  double g[PER];  // the gravity of rank lane * PER + q
  u64 c0 = 0;     // mass below this lane's first sheet
  const u32 e0 = lane * PER;
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    s.x[q] = __builtin_nan("");
    s.v[q] = 0.0;
    s.id[q] = 0;
    if (!EQ) {
      s.m[q] = 0.0;
      s.mf[q] = 0;
    }
    const u32 i = R.a + e0 + q;
    if (e0 + q < R.w) {
      s.x[q] = decode_pos(A.kin[i]);
      s.v[q] = A.vin[i];
      s.id[q] = A.iin[i];
      if (!EQ) {
        s.m[q] = A.min[i];
        s.mf[q] = mass_fix(s.m[q], A.fscale, (u32)s.id[q] - A.id0);
      }
    }
    if (EQ) g[q] = (A.totmass - 2.0 * ((double)i * A.mq)) - A.mq;
  }
  const u64 cbase = EQ ? 0ull : A.cin[R.a];
  auto gravity = [&] {  // after a change of order (unequal masses)
    u64 sum = 0;
#pragma unroll
    for (int q = 0; q < PER; ++q) sum += s.mf[q];
    c0 = cbase + (wave_incl_add(sum) - sum);
    u64 c = c0;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      g[q] = (A.totmass - 2.0 * ((double)(long long)c * A.finv)) - s.m[q];
      c += s.mf[q];
    }
  };
  if (A.pre != 0.0) {
#pragma unroll
    for (int q = 0; q < PER; ++q) s.x[q] = s.x[q] + A.pre * s.v[q];
    (void)s.sort();
  }
  if constexpr (!EQ) gravity();
  double vtop = 0.0, tf = A.t;
  for (u32 k = 0; k < A.K; ++k) {
    const double hd = k + 1 == A.K ? A.hlast : A.h;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      double F = g[q];
      F = F - A.omega2 * s.x[q];
      const double acc = (EXT ? ext_accel(A.ext, s.x[q], tf) : 0.0) + F;
      s.v[q] = s.v[q] + A.h * acc;
      s.x[q] = s.x[q] + hd * s.v[q];
      vtop = fmax(vtop, fabs(s.v[q]));
    }
    tf = tf + A.h;
    const bool moved = s.sort();
    if constexpr (!EQ)
      if (moved) gravity();
  }
  // (slots past the window: their speeds grew from zero by at most amax a step)
  R.ok = R.ok && vtop <= R.V;
  double vm = 0.0;
  u64 c = c0;
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    if (e0 + q < R.w)
      span_store<EQ>(A, R, R.a + e0 + q, s.x[q], s.v[q], s.id[q], EQ ? 0.0 : s.m[q], c, vm);
    if (!EQ) c += s.mf[q];
  }
  const u64 wm = wave_max((u64)__double_as_longlong(vm));
  const u32 sb = wave_min_u32(span_verdict(R));
  if (lane == 0) span_report(A, j, sb, wm);
}

// ---- windows of one workgroup ----------------------------------------------------
// word: *A.fail, or 0
template <class SH, bool EQ, bool EXT>
__device__ __forceinline__ void span_block(const SpanArgs &A, const u32 j, u32 word) {
  constexpr int WT = SH::WT, PER = SH::PER, NWAVE = SH::NWAVE;
  extern __shared__ u64 lds_dyn[];
  __shared__ u64 s_vm[NWAVE];
  __shared__ u32 s_sb[NWAVE];
  const u32 t = threadIdx.x;
  Reach R = span_reach(A, j);
  double x[PER], v[PER], m[PER], p[PER];
  u64 mf[PER], c[PER];
  i32 id[PER];
  u32 r[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const u32 e = i * WT + t;
    r[i] = e;
    x[i] = v[i] = m[i] = 0.0;
    mf[i] = c[i] = 0;
    id[i] = 0;
    if (e < R.w) {
      x[i] = decode_pos(A.kin[R.a + e]);
      v[i] = A.vin[R.a + e];
      id[i] = A.iin[R.a + e];
      if (!EQ) {
        m[i] = A.min[R.a + e];
        mf[i] = mass_fix(m[i], A.fscale, (u32)id[i] - A.id0);
        c[i] = A.cin[R.a + e];
      }
    }
  }
  const u64 cbase = EQ ? 0ull : A.cin[R.a];
  if (span_leaves(word, A.fail_value - 1u)) return;
  BinRank<SH, !EQ> rk(lds_dyn, R.w, A.kin + R.a, R.a > 0 ? (A.H + 1) / 2 : 0,
                       R.b < A.n ? (A.H + 1) / 2 : 0, R.D, R.D / (double)A.K);
  bool slow = true;  // every speed within the bound
  auto steps = [&](auto segs) {
    constexpr bool SEGS = decltype(segs)::value;
    if (A.pre != 0.0) {
#pragma unroll
      for (int i = 0; i < PER; ++i) p[i] = A.pre * v[i];
      rk.template step<SEGS>(R.w, x, p, r, id, mf, c, cbase);
    }
    double tf = A.t;
    for (u32 k = 0; k < A.K; ++k) {
      const double hd = k + 1 == A.K ? A.hlast : A.h;
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        double F;
        if (EQ)
          F = (A.totmass - 2.0 * ((double)(R.a + r[i]) * A.mq)) - A.mq;
        else
          F = (A.totmass - 2.0 * ((double)(long long)c[i] * A.finv)) - m[i];
        F = F - A.omega2 * x[i];
        const double acc = (EXT ? ext_accel(A.ext, x[i], tf) : 0.0) + F;
        v[i] = v[i] + A.h * acc;
        p[i] = hd * v[i];
        slow = slow && (fabs(v[i]) <= R.V || i * WT + t >= R.w);
      }
      tf = tf + A.h;
      rk.template step<SEGS>(R.w, x, p, r, id, mf, c, cbase);
    }
  };
  if (rk.segs)
    steps(std::true_type{});
  else
    steps(std::false_type{});
  R.ok = R.ok && slow;
  double vm = 0.0;
#pragma unroll
  for (int i = 0; i < PER; ++i)
    if (i * WT + t < R.w)
      span_store<EQ>(A, R, R.a + r[i], x[i], v[i], id[i], m[i], c[i], vm);
  const u64 wm = wave_max((u64)__double_as_longlong(vm));
  const u32 wb = wave_min_u32(span_verdict(R));
  if ((t & 63u) == 0) {
    s_vm[t >> 6] = wm;
    s_sb[t >> 6] = wb;
  }
  __syncthreads();
  if (t == 0) {
    u64 q = 0;
    u32 sb = SPAN_STAT_INIT;
    for (int i = 0; i < NWAVE; ++i) {
      q = s_vm[i] > q ? s_vm[i] : q;
      sb = min(sb, s_sb[i]);
    }
    span_report(A, j, sb, q);
  }
}

template <int PER, bool EQ, bool EXT>
__global__ __launch_bounds__(64) void k_span_wave(SpanArgs A) {
  if (span_leaves(*A.fail, A.fail_value - 1u)) return;
  span_wave<PER, EQ, EXT>(A, blockIdx.x);
}

template <class SH, bool EQ, bool EXT>
__global__ __launch_bounds__(SH::WT) void k_span_block(SpanArgs A) {
  // read now, looked at once the window's sheets are under way too: 480 us an
  // interval of 2^20 lognormal sheets, looked at first 491
  span_block<SH, EQ, EXT>(A, blockIdx.x, *(const volatile u32 *)A.fail);
}

template <int PER, bool EQ>
int launch_wave(hipStream_t st, const SpanArgs &a) {
  if (a.ext.kind)
    k_span_wave<PER, EQ, true><<<a.nwin, 64, 0, st>>>(a);
  else
    k_span_wave<PER, EQ, false><<<a.nwin, 64, 0, st>>>(a);
  WDY_CHECK_LAUNCH();
  return WDY_OK;
}

template <class SH, bool EQ, bool EXT>
int launch_block_one(hipStream_t st, const SpanArgs &a) {
  auto fn = k_span_block<SH, EQ, EXT>;
  const size_t lds = BinRank<SH, !EQ>::BYTES;
  if (lds > 65536)
    WDY_HIP(hipFuncSetAttribute((const void *)fn,
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds));
  fn<<<a.nwin, SH::WT, lds, st>>>(a);
  WDY_CHECK_LAUNCH();
  return WDY_OK;
}

template <class SH>
int launch_block(hipStream_t st, bool eq, const SpanArgs &a) {
  if (a.ext.kind)
    return eq ? launch_block_one<SH, true, true>(st, a)
              : launch_block_one<SH, false, true>(st, a);
  return eq ? launch_block_one<SH, true, false>(st, a)
            : launch_block_one<SH, false, false>(st, a);
}

// Windows of many simulations: one wave (PER > 0: PER sheets per lane) or
// workgroup per (simulation, window).
template <int PER, class SH, bool EQ>
__global__ __launch_bounds__(PER ? 64 : SH::WT) void k_span_many(
    const BatchDesc *__restrict__ descs, const uint2 *__restrict__ list, BatchArrays arr,
    SpanMany M, u32 q, u32 iv) {
  const uint2 e = list[blockIdx.x];
  const BatchDesc d = descs[e.x];
  const int done = (int)(q * d.K);
  if (span_leaves(M.fail[d.eslot], q) || done >= d.nleap) return;
  const int K = min((int)d.K, d.nleap - done);
  const u32 ep = iv * d.L + q;  // launches since the plan
  const int in = d.cur ^ (int)(ep & 1u), out = in ^ 1;
  SpanArgs A;
  A.n = d.n;
  A.T = d.T;
  A.H = d.H;
  A.nwin = d.nwin;
  A.K = (u32)K;
  A.id0 = d.id0;
  A.kin = arr.key[in] + d.off;
  A.vin = arr.vel[in] + d.off;
  A.iin = arr.idx[in] + d.off;
  A.kout = arr.key[out] + d.off;
  A.vout = arr.vel[out] + d.off;
  A.iout = arr.idx[out] + d.off;
  if (!EQ) {
    A.min = arr.mass[in] + d.off;
    A.cin = M.cf[in] + d.off;
    A.mout = arr.mass[out] + d.off;
    A.cout = M.cf[out] + d.off;
  }
  A.xo = A.vo = nullptr;
  A.pre = done == 0 ? d.h / 2. : 0.0;
  A.h = d.h;
  A.hlast = done + K == d.nleap ? d.h / 2. : d.h;
  A.mq = d.mq;
  A.totmass = d.totmass;
  A.omega2 = d.flags & 2u ? d.omega2 : 0.0;
  A.fscale = d.fscale;
  A.finv = d.finv;
  A.amax0 = fabs(d.totmass);
  A.amax1 = A.omega2;
  A.t = 0.0;
  u64 *const vm = d.nwin > 1 ? M.vmax + (u64)d.vslot * 3u * SPAN_SLOTS : nullptr;
  A.vmax_in = vm ? vm + (ep % 3u) * SPAN_SLOTS : nullptr;
  A.vmax_out = vm ? vm + ((ep + 1u) % 3u) * SPAN_SLOTS : nullptr;
  A.vmax_clr = vm ? vm + ((ep + 2u) % 3u) * SPAN_SLOTS : nullptr;
  A.stat = nullptr;
  A.stat_clr = nullptr;
  A.stat_host = nullptr;
  A.fail = M.fail + d.eslot;
  A.fail_value = q + 1u;
  A.fail_host = nullptr;
  if constexpr (PER > 0)
    span_wave<PER, EQ, false>(A, e.y);
  else
    span_block<SH, EQ, false>(A, e.y, 0u);
}

template <int PER, class SH, bool EQ>
int launch_many(hipStream_t st, const BatchDesc *descs, const uint2 *list, u32 nblk,
                const BatchArrays &arr, const SpanMany &m, u32 q, u32 iv) {
  if (nblk == 0) return WDY_OK;
  auto fn = k_span_many<PER, SH, EQ>;
  const size_t lds = PER ? 0 : BinRank<SH, !EQ>::BYTES;
  if (lds > 65536)
    WDY_HIP(hipFuncSetAttribute((const void *)fn,
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds));
  fn<<<nblk, PER ? 64 : SH::WT, lds, st>>>(descs, list, arr, m, q, iv);
  WDY_CHECK_LAUNCH();
  return WDY_OK;
}

}  // namespace

// Window shapes and what they cost, in us, measured on the sech^2 disk with
// step sizes of 0.1 to 700 ranks: a step (and the sort that opens an interval)
// takes `lat` + `latd` * sqrt(ranks of displacement per step) while every window
// has a CU to itself, `two` times that or `sat` per 256 windows when they share
// the CUs (in steps of one window per CU for the two largest shapes: `per`); a
// launch `base` plus `basew` per window.  [0] equal masses, [1] unequal.
struct SpanCost {
  double lat[2], latd[2], sat[2], two, per, base[2], basew[2];
};
static const SpanShape kShapes[SPAN_NSHAPES] = {
    {64, 128, 128, false}, {64, 256, 256, false}, {256, 256, 256, true},
    {256, 512, 512, true}, {512, 512, 512, true}, {512, 1024, 1024, true},
    {1024, 2048, 2048, true}, {512, 2048, 2048, true}, {1024, 4096, 4096, true},
    {1024, 7168, 5120, true}};
static const SpanCost kCost[SPAN_NSHAPES] = {
    {{0.16, 0.32}, {0.20, 0.29}, {0.025, 0.05}, 1.0, 1.0, {5.5, 5.5}, {0.0042, 0.0042}},
    {{0.27, 0.45}, {0.28, 0.45}, {0.05, 0.10}, 1.0, 1.0, {5.5, 5.5}, {0.005, 0.005}},
    {{0.85, 1.30}, {0., 0.}, {0.16, 0.30}, 1.0, 1.0, {6.5, 7.0}, {0.0035, 0.0035}},
    {{1.05, 1.60}, {0., 0.}, {0.45, 0.80}, 1.4, 1.0, {6.5, 7.0}, {0.004, 0.004}},
    {{0.90, 1.40}, {0., 0.}, {0.70, 1.20}, 1.6, 1.0, {6.5, 7.0}, {0.0045, 0.0045}},
    {{1.20, 1.90}, {0., 0.}, {1.20, 1.90}, 2.0, 1.0, {6.5, 7.0}, {0.0045, 0.0055}},
    {{1.90, 3.10}, {0., 0.}, {1.90, 3.10}, 1.8, 1.0, {6.5, 8.0}, {0.009, 0.015}},
    {{2.50, 3.90}, {0., 0.}, {2.20, 3.40}, 1.6, 1.0, {6.5, 8.5}, {0.008, 0.012}},
    {{3.55, 5.40}, {0., 0.}, {3.55, 5.40}, 1.0, 1. / 256., {7.0, 8.0}, {0.025, 0.04}},
    {{6.00, 6.30}, {0., 0.}, {6.00, 6.30}, 1.0, 1. / 256., {11., 11.}, {0.043, 0.05}}};

// Halo ranks taken over ranks the reach is expected to cross; that follows
// the smallest halo width the windows report, so it only has to cover what one
// interval changes (2^20 lognormal sheets: 482 us an output with 1.15, 418 with
// this).
constexpr double SPAN_MARGIN = 1.07;
// (a batch's plan stays for many intervals)
constexpr double SPAN_MANY_MARGIN = 1.3;
constexpr int SPAN_KBIN = 64;  // steps per launch of the binned shapes (their
                               // bins are those of its start)

static int cap_of(int shape, bool eq) {
  return eq ? kShapes[shape].cap : kShapes[shape].cap_un;
}

int span_launch(hipStream_t st, int shape, bool eq, const SpanArgs &a) {
  // every window within the shape's capacity, every sheet in one core
  const u32 span = a.nwin > 1 ? a.T + 2 * a.H : a.n;
  if (span > (u32)cap_of(shape, eq) || a.T < 1 || a.nwin < 1 || a.K < 1 ||
      (u64)a.nwin * a.T < (u64)a.n || (u64)(a.nwin - 1) * a.T >= (u64)a.n || (a.nwin > 1 && a.H < 1))
    return fail(WDY_ERUNTIME, "span_launch: %u windows of %u + 2 * %u sheets do "
                "not fit shape %d (n = %u)", a.nwin, a.T, a.H, shape, a.n);
  switch (shape) {
    case 0: return eq ? launch_wave<2, true>(st, a) : launch_wave<2, false>(st, a);
    case 1: return eq ? launch_wave<4, true>(st, a) : launch_wave<4, false>(st, a);
    case 2: return launch_block<RankShape<256, 1>>(st, eq, a);
    case 3: return launch_block<RankShape<256, 2>>(st, eq, a);
    case 4: return launch_block<RankShape<512, 1>>(st, eq, a);
    case 5: return launch_block<RankShape<512, 2>>(st, eq, a);
    case 6: return launch_block<RankShape<1024, 2>>(st, eq, a);
    case 7: return launch_block<RankShape<512, 4>>(st, eq, a);
    case 8: return launch_block<RankShape<1024, 4>>(st, eq, a);
    default: break;
  }
  // what the LDS holds: 20 B per sheet with equal masses, else 28
  using E = RankShape<1024, 7>;
  using U = RankShape<1024, 5>;
  if (a.ext.kind)
    return eq ? launch_block_one<E, true, true>(st, a)
              : launch_block_one<U, false, true>(st, a);
  return eq ? launch_block_one<E, true, false>(st, a)
            : launch_block_one<U, false, false>(st, a);
}

template <int PER, class SH>
static int launch_many_both(hipStream_t st, const BatchDesc *descs, const uint2 *list,
                            u32 neq, u32 nun, const BatchArrays &arr, const SpanMany &m,
                            u32 q, u32 iv) {
  if (int rc = launch_many<PER, SH, true>(st, descs, list, neq, arr, m, q, iv)) return rc;
  return launch_many<PER, SH, false>(st, descs, list + neq, nun, arr, m, q, iv);
}

int span_many_launch(hipStream_t st, int shape, const BatchDesc *descs,
                     const uint2 *list, u32 neq, u32 nun, const BatchArrays &arr,
                     const SpanMany &m, u32 q, u32 iv) {
  auto go = [&](auto fn) { return fn(st, descs, list, neq, nun, arr, m, q, iv); };
  switch (shape) {
    case 0: return go(launch_many_both<2, RankShape<256, 1>>);
    case 1: return go(launch_many_both<4, RankShape<256, 1>>);
    case 3: return go(launch_many_both<0, RankShape<256, 2>>);
    case 5: return go(launch_many_both<0, RankShape<512, 2>>);
    case 7: return go(launch_many_both<0, RankShape<512, 4>>);
    case 8: return go(launch_many_both<0, RankShape<1024, 4>>);
    case 9: return launch_many<0, RankShape<1024, 7>, true>(st, descs, list, neq, arr, m, q, iv);
    default: return fail(WDY_ERUNTIME, "span_many_launch: shape %d", shape);
  }
}

// Ranks that a distance takes where sheets are densest; width[k]: the smallest
// width of 2^(k + 2) ranks (1e308: fewer sheets than that).
static double ranks_of(const double *width, double dx) {
  double w0 = 0.0, r0 = 0.0;
  for (u32 k = 0; k < SPAN_NW; ++k) {
    const double w = width[k], r = (double)(4u << k);
    if (!(w < 1e300)) break;
    if (w >= dx) return r0 + (r - r0) * (dx - w0) / (w - w0);
    w0 = w;
    r0 = r;
  }
  return w0 > 0.0 ? r0 * (dx / w0) : 1e12;
}

// One shape and K serve the whole batch.  Simulations too dense for them stay
// with the workgroup-per-simulation kernel, whose time is that of the largest:
// measured, us per step, 100 sheets 3.4, 1000 4.9, 2000 6.9, above 2048 (a
// sliding pass) 5.2 ns per sheet.
void span_many_plan(std::vector<BatchDesc> &d, const double *info,
                    const std::vector<double> &reach, double h, int nleap, int *shape) {
  const double ah = std::fabs(h);
  u32 maxn = 0;
  bool un = false;
  for (const BatchDesc &q : d) {
    maxn = std::max(maxn, q.n);
    un = un || !(q.flags & 1u);
  }
  auto other = [&](u32 n) {
    return nleap * (n <= 2048 ? 3.4 + 1.7e-3 * n : 5.2e-3 * n);
  };
  double all = 0.0;  // 512 of its workgroups run at a time
  for (const BatchDesc &q : d) all += other(q.n) / 512.0;
  double best = std::max(other(maxn), all);
  int bs = -1, bk = 0;
  auto amax = [&](size_t i) {  // |acceleration| of any sheet
    return std::fabs(d[i].totmass) +
           (d[i].flags & 2u ? d[i].omega2 * info[i * SPAN_INFO + SPAN_NW + 1] : 0.0);
  };
  auto finite = [&](size_t i) {  // one that is not would take the others along
    return std::isfinite(info[i * SPAN_INFO + SPAN_NW]) && std::isfinite(amax(i));
  };
  auto halo = [&](size_t i, int K) {
    const double *w = info + i * SPAN_INFO;
    const double dx = 1.04 * (w[SPAN_NW] + ah * K * amax(i)) * ah * (K + 0.5);
    return std::ceil(SPAN_MANY_MARGIN * reach[i] * ranks_of(w, dx)) + 2.0;
  };
  double disp = 0.0;  // ranks of displacement per step
  for (size_t i = 0; i < d.size(); ++i) {
    const double *w = info + i * SPAN_INFO;
    if (finite(i)) disp = std::max(disp, ranks_of(w, ah * (w[SPAN_NW] + ah * amax(i))));
  }
  if (h != 0.0)
    each_split(nleap, [&](int K, int launches) {
      for (int s : {0, 1, 3, 5, 7, 8, 9}) {
        if ((kShapes[s].bin && K > SPAN_KBIN) || (s == 9 && un)) continue;
        const SpanCost &k = kCost[s];
        double W = 0.0, rest = 0.0;
        for (size_t i = 0; i < d.size(); ++i) {
          const double cap = cap_of(s, d[i].flags & 1u);
          const double H = d[i].n <= cap ? 0.0 : halo(i, K);
          if (finite(i) && 2.0 * H + cap / 16 <= cap) W += std::ceil(d[i].n / (cap - 2.0 * H));
          else rest = std::max(rest, other(d[i].n));
        }
        if (W == 0.0) continue;
        double step = k.lat[un] + k.latd[un] * std::sqrt(disp);
        if (W > 256.0)
          step = std::max(step * k.two, (kShapes[s].bin ? 1.0 : 1.0 + std::sqrt(disp)) * k.sat[un] * std::ceil(W * k.per) / (256.0 * k.per));
        const double cost =
            launches * (k.base[un] + k.basew[un] * W + K * step) + step + rest + 5.0;
        if (cost < best) {
          best = cost;
          bs = s;
          bk = K;
        }
      }
    });
  *shape = bs;
  u32 vslot = 0;
  for (size_t i = 0; i < d.size(); ++i) {
    BatchDesc &q = d[i];
    q.L = q.K = q.T = q.H = q.nwin = q.vslot = 0;
    if (bs < 0) continue;
    const double cap = cap_of(bs, q.flags & 1u), H = q.n <= cap ? 0.0 : halo(i, bk);
    if (!finite(i) || !(2.0 * H + cap / 16 <= cap)) continue;
    q.H = (u32)H;
    q.T = q.n <= cap ? q.n : (u32)cap - 2 * q.H;
    q.nwin = (q.n + q.T - 1) / q.T;
    q.K = (u32)bk;
    q.L = (u32)(((int64_t)nleap + bk - 1) / bk);
    if (q.nwin > 1) q.vslot = vslot++;
  }
}

// ---- a simulation's intervals --------------------------------------------------
namespace {

// vmax: three sets of words, all zero but the first of set `at`; stat: both
// sets of stat words, then the fail word; width (may be null): the words of k_span_widths
__global__ void k_span_init(u64 *vmax, u32 *stat, u32 at, u64 v, u64 *width) {
  const u32 t = threadIdx.x;
  if (width && t < 16) width[t] = ~0ull;
  for (u32 q = t; q < 3 * SPAN_SLOTS; q += blockDim.x)
    vmax[q] = q == at * SPAN_SLOTS ? v : 0ull;
  for (u32 q = t; q < 2 * SPAN_SLOTS; q += blockDim.x) stat[q] = SPAN_STAT_INIT;
  if (t == 0) stat[2 * SPAN_SLOTS] = 0;
}

// the largest |v|, into the words (zero before) of one set
__global__ __launch_bounds__(256) void k_span_absmax(u32 n, const double *__restrict__ vel,
                                                     u64 *vmax) {
  double m = 0.0;
  for (u32 i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
    m = fmax(m, fabs(vel[i]));
  const u64 w = wave_max((u64)__double_as_longlong(m));
  if ((threadIdx.x & 63u) == 0)
    atomicMax((unsigned long long *)vmax + (blockIdx.x & (SPAN_SLOTS - 1)),
              (unsigned long long)w);
}

// The smallest widths of 2^(k + 2) consecutive ranks, k < SPAN_NW: how far
// apart the sheets are where they are densest, at every halo size.  `starts`
// windows, `stride` ranks apart.  A few blocks, each with one atomic per width:
// with one per wave and width they took 128 us at 10^5 sheets.
__global__ __launch_bounds__(256) void k_span_widths(u32 n, u32 starts, u32 stride,
                                                     const u64 *__restrict__ key,
                                                     u64 *__restrict__ out) {
  __shared__ u64 s_w[4][SPAN_NW];
  u64 w[SPAN_NW];
#pragma unroll
  for (u32 k = 0; k < SPAN_NW; ++k) w[k] = ~0ull;
  for (u32 q = blockIdx.x * 256 + threadIdx.x; q < starts; q += gridDim.x * 256) {
    const u32 i = q * stride;
    const double x0 = decode_pos(key[i]);
#pragma unroll
    for (u32 k = 0; k < SPAN_NW; ++k)
      if (i + (4u << k) < n) {
        const u64 d = (u64)__double_as_longlong(decode_pos(key[i + (4u << k)]) - x0);
        w[k] = d < w[k] ? d : w[k];
      }
  }
#pragma unroll
  for (u32 k = 0; k < SPAN_NW; ++k) {
    const u64 m = wave_min(w[k]);
    if ((threadIdx.x & 63u) == 0) s_w[threadIdx.x >> 6][k] = m;
  }
  __syncthreads();
  if (threadIdx.x < SPAN_NW) {
    u64 m = s_w[0][threadIdx.x];
    for (int q = 1; q < 4; ++q) m = s_w[q][threadIdx.x] < m ? s_w[q][threadIdx.x] : m;
    if (m < out[threadIdx.x]) atomicMin((unsigned long long *)out + threadIdx.x, m);
  }
}

// Fixed-point mass below each sheet, in three passes over tiles of FIX_TILE.
constexpr u32 FIX_TILE = 4096;
__global__ __launch_bounds__(256) void k_fix_sums(u32 n, const double *__restrict__ mass,
                                                  const i32 *__restrict__ idx,
                                                  double fscale, u64 *sums) {
  __shared__ u64 s_red[4];
  u64 v = 0;
  for (u32 q = 0; q < FIX_TILE / 256; ++q) {
    const u32 i = blockIdx.x * FIX_TILE + q * 256 + threadIdx.x;
    if (i < n) v += mass_fix(mass[i], fscale, (u32)idx[i]);
  }
  u64 tot;
  (void)block_excl_u64<4>(v, s_red, &tot);
  if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}
__global__ __launch_bounds__(256) void k_fix_top(u32 nt, u64 *sums) {
  __shared__ u64 s_red[4];
  u64 run = 0;
  for (u32 b = 0; b < nt; b += 256) {
    const u32 i = b + threadIdx.x;
    const u64 v = i < nt ? sums[i] : 0ull;
    u64 tot;
    const u64 e = block_excl_u64<4>(v, s_red, &tot);
    if (i < nt) sums[i] = run + e;
    run += tot;
    __syncthreads();
  }
}
__global__ __launch_bounds__(256) void k_fix_apply(u32 n, const double *__restrict__ mass,
                                                   const i32 *__restrict__ idx,
                                                   double fscale, const u64 *sums,
                                                   u64 *__restrict__ out) {
  __shared__ u64 s_red[4];
  const u32 base = blockIdx.x * FIX_TILE + threadIdx.x * (FIX_TILE / 256);
  u64 m[FIX_TILE / 256], v = 0;
#pragma unroll
  for (u32 q = 0; q < FIX_TILE / 256; ++q) {
    m[q] = base + q < n ? mass_fix(mass[base + q], fscale, (u32)idx[base + q]) : 0ull;
    v += m[q];
  }
  u64 run = sums[blockIdx.x] + block_excl_u64<4>(v, s_red, nullptr);
#pragma unroll
  for (u32 q = 0; q < FIX_TILE / 256; ++q) {
    if (base + q < n) out[base + q] = run;
    run += m[q];
  }
}

// payload of sorted sheet i from its slot before the sort
__global__ __launch_bounds__(256) void k_span_gather(
    u32 n, const u64 *__restrict__ ks, const u32 *__restrict__ perm,
    const double *__restrict__ v, const i32 *__restrict__ id,
    const double *__restrict__ m, u64 *__restrict__ ko, double *__restrict__ vo,
    i32 *__restrict__ io, double *__restrict__ mo) {
  const u32 i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const u32 src = sorted_slot(perm, i, n);
  ko[i] = ks[i];
  vo[i] = v[src];
  io[i] = id[src];
  if (mo) mo[i] = m[src];
}

}  // namespace

// An interval that has not been checked yet.
struct SpanPending {
  SpanRedo again;       // what would have to be redone
  int start = 0;        // the set it started from
  double t0 = 0.0;
  u32 nwin = 0;
  double ratio = 0.0;   // halo ranks taken over ranks expected
  u32 first = 0, count = 0;  // its launches
};

struct SpanCtx {
  u64 *cf[3] = {nullptr, nullptr, nullptr};  // unequal masses: mass below
  u64 *vmax = nullptr;    // [3][SPAN_SLOTS]
  u32 *stat = nullptr;    // [2][SPAN_SLOTS], then the fail word
  u64 *h_buf = nullptr;   // pinned: [16] words of the widths, then
  u32 *h_stat = nullptr;  // [SPAN_SLOTS], then the fail word
  double fscale = 1.0, finv = 1.0;
  double width[16] = {};  // smallest width of 2^(k + 2) ranks at the start
  double vmax_h = 0.0;    // largest |v| at the start
  double xmax_h = 0.0;    // largest |x| at the start
  double reach = 1.0;     // ranks of a launch's reach over those the two give
  u32 epoch = 0, iv = 0;  // launches (word sets) and intervals so far
  u32 launch = 0;         // the next launch's number
  int fails = 0;          // intervals redone in a row
  bool single = false;    // one window or none
  // given up for steps of this size or longer, in intervals of this time or longer
  double up_h = 1e308, up_t = 1e308;
  SpanPlan last;          // the last search's result, for
  double l_h = 0.0, l_a0 = 0.0, l_a1 = 0.0;  // these
  int l_nleap = 0;
  bool l_single = false, l_ok = false;
  double fall = 0.8;      // how fast `reach` falls again
  bool off = false;       // for good
  SpanPending pend[SPAN_QUEUE];
  int npend = 0;
};

// |acceleration| of a sheet at x <= a0 + a1 * |x|
static void span_amax(const wdy_sim *s, double *a0, double *a1) {
  const ExtForce &f = s->ext;
  *a0 = std::fabs(s->totmass);
  *a1 = s->omega2 >= 0.0 ? s->omega2 : 0.0;
  if (f.kind == WDY_EXT_HARMONIC) *a1 += std::fabs(f.p0);
  if (f.kind == WDY_EXT_ISOTHERMAL) *a0 += std::fabs(f.p0 / f.p1);
  if (f.kind == WDY_EXT_PULSE) *a0 += std::fabs(f.p0);
}

// How far a sheet may move in `drift` time units after `kicks` time units of
// acceleration, and the ranks that takes where the sheets are densest.
static double span_reach_x(const wdy_sim *s, double drift, double kicks) {
  double a0, a1;
  span_amax(s, &a0, &a1);
  return 1.04 * (s->span->vmax_h + kicks * (a0 + a1 * s->span->xmax_h)) * drift;
}
static double span_ranks(const wdy_sim *s, double dx) {
  return ranks_of(s->span->width, dx);
}

// The windows of a launch that drifts `drift` time units in all and kicks for
// `kicks`: false when the shape cannot hold a core and its halos.
struct SpanGeom {
  u32 T, H, nwin;
  double est;  // ranks the reach is expected to cross
};
static bool span_geom(const wdy_sim *s, int shape, double reach, double drift,
                      double kicks, SpanGeom *g) {
  const u32 n = (u32)s->n, cap = (u32)cap_of(shape, s->equal_mass);
  g->est = span_ranks(s, span_reach_x(s, drift, kicks));
  if (n <= cap) {  // one window, no halo
    g->T = n;
    g->H = 0;
    g->nwin = 1;
    return true;
  }
  if (s->span->single) return false;
  const double H = std::ceil(SPAN_MARGIN * reach * g->est) + 2.0;
  if (!(2.0 * H + cap / 16 <= cap)) return false;
  g->H = (u32)H;
  g->T = cap - 2 * g->H;
  g->nwin = (n + g->T - 1) / g->T;
  return true;
}

// Time units a launch of K steps from step `done` of the interval drifts: the
// interval opens and closes with half a drift.
static double span_drift(double ah, int64_t done, int64_t K, int nleap) {
  return ah * ((double)K + (done == 0 ? 0.5 : 0.0) - (done + K == nleap ? 0.5 : 0.0));
}

static bool span_search(const wdy_sim *s, double h, int nleap, SpanPlan *plan);

bool span_plan(wdy_sim *s, double h, int nleap, SpanPlan *plan) {
  if (!s->span || s->span->off || !(h != 0.0) || !std::isfinite(h)) return false;
  SpanCtx &c = *s->span;
  // (shorter steps or intervals try again what was given up for these)
  const bool given_up =
      std::fabs(h) >= c.up_h && std::fabs(h) * (double)nleap >= c.up_t;
  if (given_up && !s->small_class) return false;
  c.single = given_up;
  // The search takes 5-15 us of host time: its result is kept for the intervals
  // that follow, while the halos they call for are those of the plan.
  double a0, a1;  // (an external force may have come or gone)
  span_amax(s, &a0, &a1);
  if (h != c.l_h || nleap != c.l_nleap || c.single != c.l_single || a0 != c.l_a0 ||
      a1 != c.l_a1 ||
      !(c.reach <= c.last.reach && c.reach >= 0.9 * c.last.reach)) {
    c.l_h = h;
    c.l_nleap = nleap;
    c.l_single = c.single;
    c.l_a0 = a0;
    c.l_a1 = a1;
    c.last.reach = 1.02 * c.reach;
    c.l_ok = span_search(s, h, nleap, &c.last);
  }
  *plan = c.last;
  return c.l_ok;
}

static bool span_search(const wdy_sim *s, double h, int nleap, SpanPlan *plan) {
  const u32 n = (u32)s->n;
  const int un = s->equal_mass ? 0 : 1;
  const double ah = std::fabs(h);
  // ranks in one step (a number also where the field at the outermost sheet
  // overflows: one window has no halos to fail)
  const double d = std::min(span_ranks(s, span_reach_x(s, ah, ah)), 1e12);
  double best = 1e300;
  each_split(nleap, [&](int K, int launches) {
    for (int i = 0; i < SPAN_NSHAPES; ++i) {
      const SpanCost &k = kCost[i];
      if (kShapes[i].bin && K > SPAN_KBIN) continue;
      double cost = 0.0;
      // the first launch and the others
      for (int q = 0; q < 2 && cost < best; ++q) {
        const int count = q == 0 ? 1 : launches - 1;
        if (count == 0) break;
        SpanGeom g;
        if (!span_geom(s, i, plan->reach, span_drift(ah, (int64_t)q * K, K, nleap), ah * K, &g)) {
          cost = 1e300;
          break;
        }
        double step = k.lat[un] + k.latd[un] * std::sqrt(d);
        if (g.nwin > 256)
          step = std::max(step * k.two, k.sat[un] * std::ceil(g.nwin * k.per) / (256.0 * k.per));
        // (sheets that cross a good part of their window every step also change
        // its segments: us per 20 steps, windows / one step per launch: 8000 sheets
        // at h = 0.1 254 / 240, 10^4 261 / 242, 32768 at 0.03 297 / 253; at half of
        // that the windows win, 20000 at 0.03 235 / 249)
        if (!un && g.nwin > 1 && d > 800.0) step *= 1.4;
        cost += count * (k.base[un] + k.basew[un] * g.nwin + K * step) + (q == 0 ? step : 0.0);
      }
      if (cost < best) {
        best = cost;
        plan->shape = i;
        plan->K = (u32)K;
      }
    }
  });
  if (s->small_class) return best < 1e300;
  // the one-step kernel over the whole GPU, measured on the sech^2 disk (us
  // per step, equal / unequal masses; the windows have to win clearly): 14 / 15 at 2^16, 21 / 24 at 2^18, 43 /
  // 48 at 2^20, 59 / 82 at 2^21, 92 / 130 at 2^22
  return 1.1 * best < nleap * (un ? 15.0 + 3.2e-5 * n : 14.0 + 2.0e-5 * n);
}

bool span_context(wdy_sim *s) {
  s->span = new (std::nothrow) SpanCtx();
  return s->span != nullptr;
}

void span_take(wdy_sim *s, Carve &k) {
  SpanCtx &c = *s->span;
  const size_t N = (size_t)s->n;
  k.take(c.vmax, 3 * SPAN_SLOTS + 16);
  k.take(c.stat, 2 * SPAN_SLOTS + 1);
  if (!s->equal_mass)
    for (int b = 0; b < 3; ++b) k.take(c.cf[b], N);
}

int span_create(wdy_sim *s, double xmax, double vmax) {
  SpanCtx *c = s->span;
  c->xmax_h = xmax;
  c->vmax_h = vmax;
  int e = 0;  // the fixed-point scale of the other paths: 2^k * totmass <= 2^62
  (void)frexp(s->totmass > 0.0 ? s->totmass : 1.0, &e);
  c->fscale = ldexp(1.0, 62 - e);
  c->finv = ldexp(1.0, e - 62);
  u64 *const width = c->vmax + 3 * SPAN_SLOTS;
  c->h_buf = (u64 *)(s->h_block + 64);
  c->h_stat = (u32 *)(c->h_buf + 16);
  u64 bits;
  __builtin_memcpy(&bits, &vmax, 8);
  k_span_init<<<1, 256, 0, s->stream>>>(c->vmax, c->stat, c->epoch % 3u, bits, width);
  // (2^18 starting ranks are enough for a density)
  const u32 n = (u32)s->n, stride = (n + (1u << 18) - 1) >> 18;
  const u32 starts = (n + stride - 1) / stride;
  k_span_widths<<<std::min<u32>((starts + 255) / 256, 128), 256, 0, s->stream>>>(
      n, starts, stride, s->key[s->cur], width);
  WDY_CHECK_LAUNCH();
  WDY_HIP(hipMemcpyAsync(c->h_buf, width, 16 * 8, hipMemcpyDeviceToHost, s->stream));
  return span_prefix(s);
}

// The widths, once the work span_create enqueued has finished.
void span_created(wdy_sim *s) {
  SpanCtx &c = *s->span;
  for (u32 k = 0; k < SPAN_NW; ++k) {
    if (c.h_buf[k] == ~0ull) c.width[k] = 1e308;
    else __builtin_memcpy(&c.width[k], &c.h_buf[k], 8);
  }
}

void span_free(wdy_sim *s) {
  SpanCtx *c = s->span;
  if (!c) return;
  delete c;
  s->span = nullptr;
}

void span_off(wdy_sim *s) {
  if (s->span) s->span->off = true;
}

// The masses below each sheet of the current (sorted) set.
int span_prefix(wdy_sim *s) {
  s->span_sorted = true;
  if (s->equal_mass) return WDY_OK;
  SpanCtx &c = *s->span;
  const u32 n = (u32)s->n, nt = (n + FIX_TILE - 1) / FIX_TILE;
  u64 *sums = (u64 *)s->tile_sums;  // N / 4096 + 2 words
  k_fix_sums<<<nt, 256, 0, s->stream>>>(n, s->mass[s->cur], s->idx[s->cur], c.fscale,
                                        sums);
  k_fix_top<<<1, 256, 0, s->stream>>>(nt, sums);
  k_fix_apply<<<nt, 256, 0, s->stream>>>(n, s->mass[s->cur], s->idx[s->cur], c.fscale,
                                         sums, c.cf[s->cur]);
  WDY_CHECK_LAUNCH();
  return WDY_OK;
}

static int span_vmax(wdy_sim *s) {
  SpanCtx &c = *s->span;
  const u32 n = (u32)s->n;
  k_span_init<<<1, 256, 0, s->stream>>>(c.vmax, c.stat, c.epoch % 3u, 0ull, nullptr);
  const u32 grid = std::min<u32>((n + 1023) / 1024, 1024);
  k_span_absmax<<<grid, 256, 0, s->stream>>>(n, s->vel[s->cur],
                                             c.vmax + SPAN_SLOTS * (c.epoch % 3u));
  WDY_CHECK_LAUNCH();
  return WDY_OK;
}

// Brings a state that other steps left in another order back into sorted
// order (by position; exact ties are put in order by the first step).
static int span_resort(wdy_sim *s) {
  if (int rc = launch_sort_state(s)) return rc;
  const u32 n = (u32)s->n;
  const int in = s->cur, out = (s->cur + 1) % 3;
  k_span_gather<<<(n + 255) / 256, 256, 0, s->stream>>>(
      n, s->key[in], s->perm[0], s->vel[in], s->idx[in], s->mass[in], s->key[out],
      s->vel[out], s->idx[out], s->equal_mass ? nullptr : s->mass[out]);
  WDY_CHECK_LAUNCH();
  s->cur = out;
  warm_invalidate(s);
  if (int rc = span_prefix(s)) return rc;
  return span_vmax(s);
}

// Whether the next interval may be enqueued before those in flight are checked.
// Each starts from the current set and writes only the two others, so an interval
// that failed can go back to its start: the next would write there, but its
// launches leave if one before them has failed.
bool span_chains(wdy_sim *s) {
  return s->span && s->span->npend > 0 && s->span->npend < SPAN_QUEUE;
}

// Enqueues one output interval, which span_settle checks once the caller has
// recorded ev1 behind it.
int span_interval(wdy_sim *s, double h, int nleap, const SpanPlan &p, double *xo,
                  double *vo) {
  SpanCtx &c = *s->span;
  if (!s->span_sorted)
    if (int rc = span_resort(s)) return rc;
  const int start = s->cur;
  const int so[2] = {(start + 1) % 3, (start + 2) % 3};
  SpanArgs a;
  a.n = (u32)s->n;
  a.id0 = 0;
  a.h = h;
  a.mq = s->m_equal;
  a.totmass = s->totmass;
  a.omega2 = s->omega2 >= 0.0 ? s->omega2 : 0.0;
  a.fscale = c.fscale;
  a.finv = c.finv;
  a.ext = s->ext;
  span_amax(s, &a.amax0, &a.amax1);
  if (c.npend == 0) {  // (nothing writes there now)
    for (u32 q = 0; q < SPAN_SLOTS; ++q) c.h_stat[q] = SPAN_STAT_INIT;
    c.h_stat[SPAN_SLOTS] = 0;
  }
  SpanPending pend;
  pend.again = {h, nleap, xo, vo};
  pend.start = start;
  pend.t0 = s->t0;
  pend.first = c.launch;
  a.stat_host = c.h_stat;
  a.fail_host = c.h_stat + SPAN_SLOTS;
  const u32 set = c.iv++ & 1u;
  a.stat = c.stat + SPAN_SLOTS * set;
  a.stat_clr = c.stat + SPAN_SLOTS * (set ^ 1u);
  a.fail = c.stat + 2 * SPAN_SLOTS;
  double t = s->t0;
  int in = start, q = 0;
  for (int done = 0; done < nleap; ++q) {
    const int K = std::min<int>((int)p.K, nleap - done);
    const int out = so[q & 1];
    const double ah = std::fabs(h);
    SpanGeom g;
    if (!span_geom(s, p.shape, p.reach, span_drift(ah, done, K, nleap), ah * K, &g))
      return fail(WDY_ERUNTIME, "span_interval: no windows for shape %d", p.shape);
    if (done == 0) {
      pend.nwin = g.nwin;
      pend.ratio = g.H / std::max(g.est, 1e-300);
    }
    a.T = g.T;
    a.H = g.H;
    a.nwin = g.nwin;
    a.K = (u32)K;
    a.fail_value = c.launch + 1u;
    c.launch = next_launch(c.launch);
    ++pend.count;
    a.kin = s->key[in];
    a.vin = s->vel[in];
    a.iin = s->idx[in];
    a.min = s->mass[in];
    a.cin = c.cf[in];
    a.kout = s->key[out];
    a.vout = s->vel[out];
    a.iout = s->idx[out];
    a.mout = s->mass[out];
    a.cout = c.cf[out];
    a.xo = done + K == nleap ? xo : nullptr;
    a.vo = done + K == nleap ? vo : nullptr;
    a.pre = done == 0 ? h / 2. : 0.0;
    a.hlast = done + K == nleap ? h / 2. : h;
    a.t = t;
    a.vmax_in = c.vmax + SPAN_SLOTS * (c.epoch % 3u);
    a.vmax_out = c.vmax + SPAN_SLOTS * ((c.epoch + 1u) % 3u);
    a.vmax_clr = c.vmax + SPAN_SLOTS * ((c.epoch + 2u) % 3u);
    ++c.epoch;
    if (s->timing) timer_begin(s->timer, s->stream, KC_WARM);
    const int rc = span_launch(s->stream, p.shape, s->equal_mass, a);
    if (s->timing) timer_end(s->timer, s->stream, KC_WARM);
    if (rc) return rc;
    for (int k = 0; k < K; ++k) t = t + h;
    done += K;
    in = out;
  }
  c.pend[c.npend++] = pend;
  s->cur = in;
  if (s->ext.kind) s->t0 = t;
  return WDY_OK;
}

// Waits for and checks the intervals in flight.  redo[0 .. *count): the first that
// failed and those after it, which did not run; the state is back at its start,
// with the halo estimate widened, and the caller must redo them.
int span_settle(wdy_sim *s, SpanRedo *redo, int *count) {
  *count = 0;
  SpanCtx *cp = s->span;
  if (!cp || cp->npend == 0) return WDY_OK;
  SpanCtx &c = *cp;
  WDY_HIP(hipEventSynchronize(s->ev1));
  const int n = c.npend;
  c.npend = 0;
  const u32 word = c.h_stat[SPAN_SLOTS];
  int bad = n;
  for (int i = 0; word && i < n && bad == n; ++i)
    if (launch_of(word - 1u, c.pend[i].first, c.pend[i].count) >= 0) bad = i;
  if (word && bad == n)
    return fail(WDY_ERUNTIME, "a window of launch %u failed, which is not in flight", word - 1u);
  for (int i = 0; i < bad; ++i)
    if (!s->small_class) s->warm_steps += c.pend[i].again.nleap;
  if (bad == n) {
    c.fails = 0;
    u32 st = SPAN_STAT_INIT;
    for (u32 q = 0; q < SPAN_SLOTS; ++q) st = std::min(st, c.h_stat[q]);
    double ratio = 0.0;
    for (int i = 0; i < n; ++i)
      if (c.pend[i].nwin > 1) ratio = std::max(ratio, c.pend[i].ratio);
    if (ratio > 0.0 && st < SPAN_STAT_INIT) {
      float slack;
      __builtin_memcpy(&slack, &st, 4);
      // ranks the reach took over those expected.  It falls slowly, and not
      // below what the widths say: the cores' boundaries are a few of the
      // places where the next plan may put its own.
      c.reach = std::max(std::max(ratio / slack, c.fall * c.reach), 1.0);
    }
    return WDY_OK;
  }
  const SpanPending &p = c.pend[bad];
  for (int i = bad; i < n; ++i) redo[(*count)++] = c.pend[i].again;
  s->cur = p.start;
  s->t0 = p.t0;
  s->fail_overflow += 1;
  c.reach = std::min(2.0 * c.reach, 1e6);
  c.fall = 0.97;
  ++c.fails;
  if (p.nwin == 1) c.off = true;  // not finite
  else if (c.fails >= (s->small_class ? 2 : 3)) {
    c.up_h = std::min(c.up_h, std::fabs(p.again.h));
    c.up_t = std::min(c.up_t, std::fabs(p.again.h) * (double)p.again.nleap);
  }
  return span_vmax(s);
}

}  // namespace wdy
