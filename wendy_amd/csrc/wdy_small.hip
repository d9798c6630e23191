// Small-N path: one workgroup runs a whole output interval (all nleap
// leapfrog steps) in a single launch, with the sorted positions in LDS.
//
// Layout (small mode of a sim):
//   key[0][i], idx[0][i]   sorted (position key, sheet index) pairs, the
//                          reference's xi[] array (wendy/wendy.h:12-16)
//   vel[0][j], mass[0][j]  velocity and mass*twopiG of sheet j, in original
//                          sheet order (the reference's v[] and m[])
// LDS holds the (key, index) pairs: 12 B per sheet.  Each step re-sorts them
// with odd-even transposition rounds until a round swaps nothing: the input is
// the previous step's order, and sheets move only a few ranks per step, so a
// few rounds suffice (any input still ends sorted; it just takes more rounds).
// Pairs compare by (key, index), so exactly tied positions are ordered by
// sheet index.  The mass prefix is a single-thread sequential sum for
// n <= SEQ_SCAN_MAX (the reference's exact summation order,
// wendy/wendy.c:359-360) and a blocked parallel scan above.
//
// Up to 512 sheets (k_small_wave) one wave holds everything in registers,
// 2, 4 or 8 consecutive ranks per lane.
#include "wdy_rank.h"

namespace wdy {
namespace {

constexpr u32 SEQ_SCAN_MAX = 512;

__device__ __forceinline__ bool pair_less(u64 ka, i32 ia, u64 kb, i32 ib) {
  return ka < kb || (ka == kb && ia < ib);
}

// Sorts (ks, is)[0..n) in LDS by odd-even transposition until no swap.
__device__ void lds_transposition_sort(u64 *ks, i32 *is, u32 n) {
  const u32 t = threadIdx.x, T = blockDim.x;
  while (true) {
    int sw = 0;
#pragma unroll
    for (u32 ph = 0; ph < 2; ++ph) {
      for (u32 p = t; 2 * p + ph + 1 < n; p += T) {
        const u32 a = 2 * p + ph;
        const u64 ka = ks[a], kb = ks[a + 1];
        const i32 ia = is[a], ib = is[a + 1];
        if (pair_less(kb, ib, ka, ia)) {
          ks[a] = kb;
          ks[a + 1] = ka;
          is[a] = ib;
          is[a + 1] = ia;
          sw = 1;
        }
      }
      __syncthreads();
    }
    if (!__syncthreads_or(sw)) break;
  }
}

// Exclusive prefix of mass[is[i]] over sorted slots into cum[], blocked over
// threads (each thread sums a contiguous chunk sequentially).
__device__ void block_mass_prefix(const i32 *is, const double *mass,
                                  double *cum, u32 n, double *s_part) {
  const u32 t = threadIdx.x, T = blockDim.x;
  const u32 per = (n + T - 1) / T;
  const u32 b = t * per;
  double acc = 0.0;
  for (u32 j = 0; j < per && b + j < n; ++j) acc = acc + mass[is[b + j]];
  s_part[t] = acc;
  __syncthreads();
  if (t == 0) {
    double run = 0.0;
    for (u32 q = 0; q < T; ++q) {
      const double v = s_part[q];
      s_part[q] = run;
      run = run + v;
    }
  }
  __syncthreads();
  double run = s_part[t];
  for (u32 j = 0; j < per && b + j < n; ++j) {
    cum[b + j] = run;
    run = run + mass[is[b + j]];
  }
}

// smem: 12 B per sheet; s_part: one word per thread, for n > SEQ_SCAN_MAX
template <bool EQ, bool HARM>
__device__ __forceinline__ void small_interval(
    u32 n, u64 *__restrict__ key_g, i32 *__restrict__ id_g,
    double *__restrict__ vel, const double *__restrict__ mass,
    double *__restrict__ cum, double mq, double totmass, double omega2,
    double h, int nleap, double *__restrict__ acc_out,
    double *__restrict__ cum_out, const ExtForce &ext, double t0, u64 *smem,
    double *s_part) {
  u64 *ks = smem;
  i32 *is = (i32 *)(smem + n);
  const u32 t = threadIdx.x, T = blockDim.x;
  const double hh = h / 2.;
  for (u32 i = t; i < n; i += T) {
    const i32 id = id_g[i];
    is[i] = id;
    // half drift (wendy/wendy.c:318-323,398)
    ks[i] = encode_pos(decode_pos(key_g[i]) + hh * vel[id]);
  }
  __syncthreads();
  double tf = t0;  // time of this step's force (wendy/wendy.c:401-408)
  for (int step = 0; step < nleap; ++step) {
    const bool last = step == nleap - 1;
    const double hd = last ? hh : h;
    lds_transposition_sort(ks, is, n);
    if (!EQ) {
      if (n <= SEQ_SCAN_MAX) {
        if (t == 0) {
          double c = 0.0;
          for (u32 i = 0; i < n; ++i) {
            cum[i] = c;
            c = c + mass[is[i]];
          }
        }
      } else {
        block_mass_prefix(is, mass, cum, n, s_part);
      }
      __syncthreads();
    }
    for (u32 i = t; i < n; i += T) {
      const i32 id = is[i];
      double x = decode_pos(ks[i]);
      const double C = EQ ? (double)i * mq : cum[i];
      const double m = EQ ? mq : mass[id];
      double F = (totmass - 2.0 * C) - m;
      if (HARM) F = F - omega2 * x;
      const double a = (ext.kind ? ext_accel(ext, x, tf) : 0.0) + F;
      const double v = vel[id] + h * a;
      vel[id] = v;
      x = x + hd * v;
      ks[i] = encode_pos(x);
      if (last && acc_out) acc_out[id] = a;
      if (last && cum_out) cum_out[i] = C;
    }
    tf = tf + h;
    __syncthreads();
  }
  for (u32 i = t; i < n; i += T) {
    key_g[i] = ks[i];
    id_g[i] = is[i];
  }
}

template <bool EQ, bool HARM>
__global__ __launch_bounds__(1024) void k_small_advance(
    u32 n, u64 *__restrict__ key_g, i32 *__restrict__ id_g,
    double *__restrict__ vel, const double *__restrict__ mass,
    double *__restrict__ cum, double mq, double totmass, double omega2,
    double h, int nleap, double *__restrict__ acc_out,
    double *__restrict__ cum_out, ExtForce ext, double t0) {
  extern __shared__ u64 smem[];
  __shared__ double s_part[1024];
  small_interval<EQ, HARM>(n, key_g, id_g, vel, mass, cum, mq, totmass, omega2, h,
                           nleap, acc_out, cum_out, ext, t0, smem, s_part);
}

// The same for up to 64 * PER sheets, by one wave with the sheets of
// consecutive ranks in a lane's registers: no barrier, no memory traffic
// within the interval.  A step is a chain of dependent instructions (force,
// kick, drift, the test of the order), so what bounds it is their latency:
// measured, us per step, before (k_small_advance) -> now: 3 sheets 0.77 ->
// 0.058, 101 sheets with tracers 4.4 -> 0.22, 512 sheets that move ~2 ranks a
// step 2.2 -> 0.9 with equal masses.  The rounds of the sort grow with the
// displacement as before, at about half the time each.
// The unequal masses' prefix stays the reference's sequential sum, bit for bit.
template <int PER, bool EQ, bool HARM, bool EXT>
__global__ __launch_bounds__(64) void k_small_wave(
    u32 n, u64 *__restrict__ key_g, i32 *__restrict__ id_g,
    double *__restrict__ vel, const double *__restrict__ mass,
    double *__restrict__ cum, double mq, double totmass, double omega2, double h,
    int nleap, double *__restrict__ acc_out, double *__restrict__ cum_out,
    ExtForce ext, double t0, double *__restrict__ xo, double *__restrict__ vo) {
  extern __shared__ u64 smem[];
  __shared__ double s_m[EQ ? 1 : 64 * PER + 8];  // masses in sorted order
  __shared__ double s_id[EQ ? 1 : 64 * PER];     // masses by sheet index
  const u32 lane = threadIdx.x & 63u, e0 = lane * PER;
  WaveSheets<PER, false> s;
  double m[PER], C[PER], g[PER], a[PER];
  const double hh = h / 2.;
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    s.x[q] = __builtin_nan("");
    s.v[q] = 0.0;
    s.id[q] = 0;
    a[q] = 0.0;
    C[q] = 0.0;
    m[q] = 0.0;
    if (e0 + q < n) {
      s.id[q] = id_g[e0 + q];
      s.v[q] = vel[s.id[q]];
      // half drift (wendy/wendy.c:318-323,398)
      s.x[q] = decode_pos(key_g[e0 + q]) + hh * s.v[q];
    }
    if (EQ) {
      C[q] = (double)(e0 + q) * mq;
      g[q] = (totmass - 2.0 * C[q]) - mq;
    }
  }
  if (!EQ) {
    for (u32 i = lane; i < n; i += 64) s_id[i] = mass[i];
    if (lane < 8) s_m[64 * PER + lane] = 0.0;
    __syncthreads();
  }
  // The masses below: C[0] of a lane and its masses give its C and its end; the
  // whole is the sequential sum, bit for bit, exactly when every lane's end is
  // the next one's C[0].  After a change of order that mostly holds with the
  // starts as they were (where it does not, rounding went the other way and the
  // starts move on lane by lane for a few rounds; then everything is summed
  // again from the first lane in doubt).
  u32 k0 = 0;  // lanes up to here have the right C[0]
  auto sum_from_k0 = [&] {
#pragma unroll
    for (int q = 0; q < PER; ++q) s_m[e0 + q] = m[q];
    __syncthreads();
    const u64 c = (u64)__double_as_longlong(C[0]);
    double run = __longlong_as_double((long long)(
        ((u64)(u32)__builtin_amdgcn_readlane((int)(c >> 32), k0) << 32) |
        (u32)__builtin_amdgcn_readlane((int)c, k0)));
    // each lane adds up every mass from lane k0's first to its own first (the
    // loads ahead of the chain of additions, zeros from its own on)
    for (u32 k = k0 * PER; k < n; k += 8) {
      double w[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) w[q] = s_m[k + q];
#pragma unroll
      for (int q = 0; q < 8; ++q) run = run + (k + q < e0 ? w[q] : 0.0);
    }
    if (lane >= k0) C[0] = run;
    __syncthreads();
  };
  bool first = true;
  auto prefix = [&] {  // unequal masses, after a change of order
    bool diff = first;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const double mq_ = e0 + q < n ? s_id[s.id[q]] : 0.0;
      diff = diff || mq_ != m[q];
      m[q] = mq_;
    }
    if (__ballot(diff) == 0) return;
    if (first) sum_from_k0();
    first = false;
    for (int round = 0;; ++round) {
      double run = C[0];
#pragma unroll
      for (int q = 0; q < PER; ++q) {
        C[q] = run;
        run = run + m[q];
      }
      const double next = dpp_mov_f64<DPP_WAVE_SHL1>(run, C[0]);
      const u64 bad = __ballot(run != next);
      if (bad == 0 || round > 6) break;
      if (round == 6) {
        k0 = (u32)__ffsll((long long)bad) - 1u;
        sum_from_k0();
      } else {
        C[0] = dpp_mov_f64<DPP_WAVE_SHR1>(0.0, run);
      }
    }
#pragma unroll
    for (int q = 0; q < PER; ++q) g[q] = (totmass - 2.0 * C[q]) - m[q];
  };
  (void)s.sort();
  if constexpr (!EQ) prefix();
  double tf = t0;  // time of this step's force (wendy/wendy.c:401-408)
  for (int step = 0; step < nleap; ++step) {
    const double hd = step == nleap - 1 ? hh : h;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      double F = g[q];
      if (HARM) F = F - omega2 * s.x[q];
      a[q] = (EXT ? ext_accel(ext, s.x[q], tf) : 0.0) + F;
      s.v[q] = s.v[q] + h * a[q];
      s.x[q] = s.x[q] + hd * s.v[q];
    }
    tf = tf + h;
    if (step == nleap - 1) break;
    const bool moved = s.sort();
    if constexpr (!EQ)
      if (moved) prefix();
  }
  // (a sheet that overflowed compares with nothing: in the keys' order then,
  // from the start, which is still in memory)
  bool over = false;
#pragma unroll
  for (int q = 0; q < PER; ++q)
    over = over || (e0 + q < n && !(fabs(s.x[q]) < __builtin_inf() &&
                                    fabs(s.v[q]) < __builtin_inf()));
  if (__builtin_expect(__ballot(over) != 0, 0)) {
    small_interval<EQ, HARM>(n, key_g, id_g, vel, mass, cum, mq, totmass, omega2, h,
                             nleap, acc_out, cum_out, ext, t0, smem, nullptr);
    __syncthreads();
    for (u32 i = lane; xo && i < n; i += 64) {
      xo[id_g[i]] = decode_pos(key_g[i]);
      vo[i] = vel[i];
    }
    return;
  }
#pragma unroll
  for (int q = 0; q < PER; ++q)
    if (e0 + q < n) {
      key_g[e0 + q] = encode_pos(s.x[q]);
      id_g[e0 + q] = s.id[q];
      vel[s.id[q]] = s.v[q];
      if (xo) {
        xo[s.id[q]] = s.x[q];
        vo[s.id[q]] = s.v[q];
      }
      if (acc_out) acc_out[s.id[q]] = a[q];
      if (cum_out) cum_out[e0 + q] = C[q];
    }
}

template <int PER, bool EXT>
int launch_wave(wdy_sim *s, double h, int nleap, double *acc, double *cum, double *xo,
                double *vo) {
  const bool harm = s->omega2 >= 0.0;
#define WDY_WAVE(EQ, HARM)                                                    \
  k_small_wave<PER, EQ, HARM, EXT><<<1, 64, (size_t)s->n * 12 + 16, s->stream>>>( \
      (u32)s->n, s->key[0], s->idx[0], s->vel[0], s->mass[0], s->cum,         \
      s->m_equal, s->totmass, s->omega2, h, nleap, acc, cum, s->ext, s->t0,   \
      xo, vo)
  if (s->equal_mass) {
    if (harm) WDY_WAVE(true, true); else WDY_WAVE(true, false);
  } else {
    if (harm) WDY_WAVE(false, true); else WDY_WAVE(false, false);
  }
#undef WDY_WAVE
  WDY_CHECK_LAUNCH();
  return WDY_OK;
}

template <bool EXT>
int launch_wave_per(wdy_sim *s, double h, int nleap, double *acc, double *cum,
                    double *xo, double *vo) {
  if (s->n <= 128) return launch_wave<2, EXT>(s, h, nleap, acc, cum, xo, vo);
  if (s->n <= 256) return launch_wave<4, EXT>(s, h, nleap, acc, cum, xo, vo);
  return launch_wave<8, EXT>(s, h, nleap, acc, cum, xo, vo);
}

}  // namespace

u32 small_max_n(int device) {
  int lds = 0;
  if (hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock,
                            device) != hipSuccess)
    lds = 65536;
  // 12 B per sheet of dynamic LDS, plus 8 KiB of static LDS
  const long cap = ((long)lds - 8192 - 64) / 12;
  return cap > 0 ? (u32)cap : 0u;
}

int launch_small_advance(wdy_sim *s, double h, int nleap, double *acc_out,
                         double *cum_out, double *xo, double *vo) {
  const u32 n = (u32)s->n;
  if (small_wave(s)) {
    if (s->timing) timer_begin(s->timer, s->stream, KC_LEAP);
    const int rc =
        s->ext.kind ? launch_wave_per<true>(s, h, nleap, acc_out, cum_out, xo, vo)
                    : launch_wave_per<false>(s, h, nleap, acc_out, cum_out, xo, vo);
    if (s->timing) timer_end(s->timer, s->stream, KC_LEAP);
    return rc;
  }
  u32 threads = ((n / 2 + 63) / 64) * 64;
  if (threads < 64) threads = 64;
  if (threads > 1024) threads = 1024;
  const size_t lds = (size_t)n * 12 + 16;
  const bool harm = s->omega2 >= 0.0;
  if (s->timing) timer_begin(s->timer, s->stream, KC_LEAP);
#define WDY_SMALL(EQ, HARM)                                                   \
  do {                                                                        \
    auto fn = k_small_advance<EQ, HARM>;                                      \
    if (lds > 65536)                                                          \
      WDY_HIP(hipFuncSetAttribute((const void *)fn,                           \
                                  hipFuncAttributeMaxDynamicSharedMemorySize, \
                                  (int)lds));                                 \
    fn<<<1, threads, lds, s->stream>>>(n, s->key[0], s->idx[0], s->vel[0],    \
                                       s->mass[0], s->cum, s->m_equal,        \
                                       s->totmass, s->omega2, h, nleap,       \
                                       acc_out, cum_out, s->ext, s->t0);      \
  } while (0)
  if (s->equal_mass) {
    if (harm) WDY_SMALL(true, true); else WDY_SMALL(true, false);
  } else {
    if (harm) WDY_SMALL(false, true); else WDY_SMALL(false, false);
  }
#undef WDY_SMALL
  if (s->timing) timer_end(s->timer, s->stream, KC_LEAP);
  WDY_CHECK_LAUNCH();
  return WDY_OK;
}

}  // namespace wdy
