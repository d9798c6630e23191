// Batched ensemble: thousands of independent simulations of uneven N advance
// together, ONE launch per output interval.
//
// A batch's first interval, and every interval of the serving pool, runs one
// 512-thread workgroup per simulation through all of its leapfrog steps (a
// persistent workgroup per simulation; descriptors are ordered largest first so
// the longest workgroups start first).  Its time is that of the largest
// simulation: 3.4 ms for 10 steps of 65536 sheets.
//
// From the second interval of the same steps on a batch runs in windows
// (wdy_span.h), one workgroup or wave per (simulation, window) and several steps
// per launch, planned on the host from the densities and speeds that k_batch_form reports.
// Nothing waits for the host within a plan: a window that cannot vouch for its
// core marks its simulation, whose later launches then leave it alone, and
// k_batch_advance, which ends every interval, redoes the rest of the interval
// from the marked launch's input (its two sets alternate by launch) and brings
// it back into the windows' form.  Measured, us per interval of 10 steps at
// h = 1e-3, before -> with windows: 100 disks of 5000-20000 sheets 962 -> 99
// (lognormal masses 1183 -> 131), 4 of 40000-60000 2704 -> 58, 400 of 50-60
// 44 -> 13, 2000 of 64-512 156 -> 29, 384 of 256-65536 3600 -> 410.
//  State lives in one arena:
// simulation k occupies [off_k, off_k + n_k) of two buffer sets of SoA arrays
// (key = order-preserving position encoding, velocity, global sheet index,
// mass * twopiG); `cur` in the descriptor says which set is current.
//
// * n <= BLOCK (2048): the whole simulation stays in LDS for the interval;
//   each step sorts it with the LDS bucket sort (a full sort: any input
//   order), then computes force, kick and drift in sorted order.
// * n > BLOCK: each step is one pass of a window sliding along the previous
//   order (slide_step): sorted in LDS, its lower part final and written out
//   with force, kick and drift, its upper half kept for the next window.
//   When a sheet has fallen more than BLOCK/4 ranks behind its previous place
//   (the first step from an arbitrary input order, for one) the pass detects
//   it and the step is redone in full: the arena range is sorted in place
//   with a block odd-even merge sort -- sort aligned blocks of BLOCK sheets
//   in LDS, then blocks offset by BLOCK/2 -- repeated until every block
//   boundary is in order (each block sort only permutes its own block, so
//   ordered boundaries mean the range is sorted; any input order finishes
//   within ceil(2n/BLOCK) + 1 rounds), then a last pass computes force, kick
//   and drift block by block, carrying the rank and the fixed-point mass
//   prefix, and writes the other buffer set.
//
// Arithmetic is the reference's (wendy/wendy.c:318-333, 371-383); ties break
// by sheet index; the unequal-mass prefix is exact fixed point (as in the
// warm-start step), equal masses use rank * m.
#include <algorithm>
#include <cmath>
#include <new>
#include <vector>

#include "wdy_batch.h"
#include "wdy_lds.h"
#include "wdy_span.h"

namespace wdy {

namespace {

// 512 threads, windows of 2048 sheets: 70 KB of LDS, two workgroups per
// CU, so that one's barriers overlap the other's work (one 1024-thread
// workgroup with 4096-sheet windows per CU measured 23% slower)
using BSH = Shape<512, 2048>;
constexpr int BWT = BSH::WT, BLOCK = BSH::CAP, BPER = BSH::PER;
constexpr int BNWAVE = BSH::NWAVE;

// Sorts A[lo, lo + c) (c <= BLOCK) in place by (key, index), via LDS.
__device__ void block_sort_inplace(Lds<BSH, false> &s, u64 *key, double *vel,
                                   i32 *idx, double *mass, u64 lo, u32 c,
                                   u64 *s_red, u64 *s_mm) {
  const u32 t = threadIdx.x;
#pragma unroll
  for (int i = 0; i < BPER; ++i) {
    const u32 e = i * BWT + t;
    if (e < c) {
      s.key[e] = key[lo + e];
      s.v[e] = vel[lo + e];
      s.id[e] = idx[lo + e];
      s.m[e] = mass ? mass[lo + e] : 0.0;
    }
  }
  __syncthreads();
  lds_bucket_sort<BSH, false>(s, c, s_red, s_mm, nullptr);
#pragma unroll
  for (int i = 0; i < BPER; ++i) {
    const u32 r = i * BWT + t;
    if (r < c) {
      const u32 e = s.ord[r];
      key[lo + r] = s.key[e];
      vel[lo + r] = s.v[e];
      idx[lo + r] = s.id[e];
      if (mass) mass[lo + r] = s.m[e];
    }
  }
  __syncthreads();
}

// Force, kick and drift of the sorted sheets s.ord[0..c) whose ranks start
// at rank0; `run` is the fixed-point mass below the first of them.  New
// keys and velocities are written back into LDS; returns the updated run.
__device__ u64 block_leap(Lds<BSH, false> &s, const BatchDesc &d, u32 c,
                          u64 rank0, u64 run, double hd, u64 *s_red) {
  const u32 t = threadIdx.x;
  const bool eq = d.flags & 1u, harm = d.flags & 2u;
  const u32 r0 = t * BPER;  // ranks r0 .. r0 + BPER - 1 in order
  u64 local = 0, total = 0, mf[BPER];
  if (!eq) {
    u64 part = 0;
#pragma unroll
    for (int i = 0; i < BPER; ++i) {
      mf[i] = 0;
      if (r0 + i < c) {
        const u32 e = s.ord[r0 + i];
        mf[i] = mass_fix(s.m[e], d.fscale, (u32)s.id[e] - d.id0);
      }
      part += mf[i];
    }
    local = block_excl_u64<BNWAVE>(part, s_red, &total);
  }
  u64 pre = run + local;
#pragma unroll
  for (int i = 0; i < BPER; ++i) {
    const u32 r = r0 + i;
    if (r < c) {
      const u32 e = s.ord[r];
      double x = decode_pos(s.key[e]);
      double F;
      if (eq) {
        F = (d.totmass - 2.0 * ((double)(rank0 + r) * d.mq)) - d.mq;
      } else {
        const double me = s.m[e];
        F = (d.totmass - 2.0 * ((double)pre * d.finv)) - me;
        pre += mf[i];
      }
      if (harm) F = F - d.omega2 * x;
      const double a = 0.0 + F;
      const double v = s.v[e] + d.h * a;
      x = x + hd * v;
      s.v[e] = v;
      s.key[e] = encode_pos(x);
    }
  }
  __syncthreads();
  return run + total;
}

// One leapfrog step of a simulation with n > BLOCK sheets, from the arrays
// key..mass (positions already drifted to the force time) into ko..mo, in
// ONE pass: a window of BLOCK sheets slides along the previous order by
// STRIDE = BLOCK - KEEP sheets; each window is sorted in LDS, all but its
// upper KEEP sheets are final (force, kick, drift, written out) and those
// stay, in their LDS slots, for the next window, whose new sheets fill the
// slots just written out.  The first window holds KEEP + ((n - BLOCK) mod
// STRIDE) sheets (BLOCK when that remainder is 0) so that every later one
// is full.  That holds while no sheet has fallen more than KEEP ranks behind
// its place in the previous order; a sheet arriving below one already
// written shows that it did not,
// and the step reports failure (the inputs are untouched, so the caller
// redoes the step in full).  Returns true on success.
__device__ bool slide_step(Lds<BSH, false> &s, const BatchDesc &d, u32 n,
                           const u64 *key, const double *vel, const i32 *idx,
                           const double *mass, u64 *ko, double *vo, i32 *io,
                           double *mo, double hd, u64 *s_red, u64 *s_mm,
                           u32 *s_ok, u64 *s_last) {
  constexpr u32 KEEP = BLOCK / 4, STRIDE = BLOCK - KEEP;
  const u32 t = threadIdx.x;
  if (t == 0) *s_ok = 1u;
  const u32 rem = (n - (u32)BLOCK) % STRIDE;
  u32 c = rem ? KEEP + rem : (u32)BLOCK;  // sheets in the current window
  u32 lo = 0, done = 0, ne = 0;
  bool first = true;
  u64 run = 0;
  while (done < n) {
    // this window's new sheets: all c at first; then STRIDE of them, into
    // the slots written out last (s.ord[0 .. ne)) and the ones the first
    // window left unused ([c_prev, BLOCK))
    const u32 cprev = c, cn = first ? c : STRIDE;
    if (!first) c = BLOCK;
#pragma unroll
    for (int i = 0; i < BPER; ++i) {
      const u32 jn = i * BWT + t;
      if (jn < cn) {
        const u32 e = first ? jn : (jn < ne ? (u32)s.ord[jn] : cprev + (jn - ne));
        const u32 g = lo + jn;
        s.key[e] = key[g];
        s.v[e] = vel[g];
        s.id[e] = idx[g];
        s.m[e] = mass ? mass[g] : 0.0;
      }
    }
    lo += cn;
    __syncthreads();
    lds_bucket_sort<BSH, false>(s, c, s_red, s_mm, nullptr);
    ne = lo == n ? c : c - KEEP;  // sheets final in this window
    if (t == 0) {
      const u32 e0 = s.ord[0];
      if (!first && pair_lt(s.key[e0], s.id[e0], s_last[0], (i32)s_last[1]))
        *s_ok = 0u;  // precedes a sheet already written
      const u32 el = s.ord[ne - 1];
      s_last[0] = s.key[el];
      s_last[1] = (u64)(u32)s.id[el];
    }
    __syncthreads();
    run = block_leap(s, d, ne, done, run, hd, s_red);
#pragma unroll
    for (int i = 0; i < BPER; ++i) {
      const u32 r = i * BWT + t;
      if (r < ne) {
        const u32 e = s.ord[r];
        ko[done + r] = s.key[e];
        vo[done + r] = s.v[e];
        io[done + r] = s.id[e];
        if (mo) mo[done + r] = s.m[e];
      }
    }
    __syncthreads();
    done += ne;
    first = false;
  }
  const bool ok = *s_ok != 0u;
  __syncthreads();
  return ok;
}

__device__ __forceinline__ bool ordered(const u64 *key, const i32 *idx,
                                        u64 a, u64 b) {
  const u64 ka = key[a], kb = key[b];
  return ka < kb || (ka == kb && idx[a] <= idx[b]);
}

// The arena range of one simulation into sorted order, in place: block
// odd-even merge sort, until every boundary of the offset blocks is in order.
// False when that takes more rounds than any input needs.
__device__ bool range_sort(Lds<BSH, false> &s, u32 n, u64 *key, double *vel, i32 *idx,
                           double *mass, u64 *s_red, u64 *s_mm, u32 *s_flag) {
  const u32 t = threadIdx.x, half = BLOCK / 2;
  const u32 max_rounds = (2 * n + BLOCK - 1) / BLOCK + 1;
  bool sorted = false;
  for (u32 round = 0; round < max_rounds && !sorted; ++round) {
    for (u32 lo = 0; lo < n; lo += BLOCK)
      block_sort_inplace(s, key, vel, idx, mass, lo, min((u32)BLOCK, n - lo),
                         s_red, s_mm);
    for (u32 lo = half; lo < n; lo += BLOCK)
      block_sort_inplace(s, key, vel, idx, mass, lo, min((u32)BLOCK, n - lo),
                         s_red, s_mm);
    // every boundary of the offset blocks in order -> the range is sorted
    if (t == 0) *s_flag = 1;
    __syncthreads();
    for (u32 b = half + (u32)t * BLOCK; b < n; b += (u32)BWT * BLOCK)
      if (!ordered(key, idx, b - 1, b)) *s_flag = 0;
    __syncthreads();
    sorted = *s_flag != 0;
    __syncthreads();
  }
  return sorted;
}

// Brings set a into the form the windows read: sorted, with the mass below
// each sheet and the speed words of the next launch (ep since the plan), and
// tells the host the densities and the largest speed.
__device__ void window_form(Lds<BSH, false> &s, const BatchDesc &d, const BatchArrays &A,
                            const SpanMany &M, int a, u32 ep, u32 *err, u64 *s_red,
                            u64 *s_mm, u32 *s_flag) {
  const u32 t = threadIdx.x, n = d.n;
  const bool eq = d.flags & 1u;
  u64 *key = A.key[a] + d.off;
  double *vel = A.vel[a] + d.off;
  i32 *idx = A.idx[a] + d.off;
  double *mass = eq ? nullptr : A.mass[a] + d.off;
  if (!range_sort(s, n, key, vel, idx, mass, s_red, s_mm, s_flag) && t == 0)
    atomicOr(err + d.eslot, 1u);
  if (!eq) {
    u64 *cf = M.cf[a] + d.off;
    u64 run = 0;
    for (u32 lo = 0; lo < n; lo += BLOCK) {
      u64 m[BPER], part = 0, total;
#pragma unroll
      for (int i = 0; i < BPER; ++i) {
        const u32 r = lo + t * BPER + i;
        m[i] = r < n ? mass_fix(mass[r], d.fscale, (u32)idx[r] - d.id0) : 0ull;
        part += m[i];
      }
      u64 c = run + block_excl_u64<BNWAVE>(part, s_red, &total);
#pragma unroll
      for (int i = 0; i < BPER; ++i) {
        const u32 r = lo + t * BPER + i;
        if (r < n) cf[r] = c;
        c += m[i];
      }
      run += total;
      __syncthreads();
    }
  }
  // [0, SPAN_NW): ~width, so that all are maxima; then the speed
  u64 top[SPAN_NW + 1];
#pragma unroll
  for (u32 k = 0; k <= SPAN_NW; ++k) top[k] = 0;
  for (u32 i = t; i < n; i += BWT) {
    const double x = decode_pos(key[i]);
    top[SPAN_NW] = max(top[SPAN_NW], (u64)__double_as_longlong(fabs(vel[i])));
#pragma unroll
    for (u32 k = 0; k < SPAN_NW; ++k)
      if (i + (4u << k) < n)
        top[k] = max(top[k], ~(u64)__double_as_longlong(decode_pos(key[i + (4u << k)]) - x));
  }
#pragma unroll
  for (u32 k = 0; k <= SPAN_NW; ++k) {
    const u64 w = wave_max(top[k]);
    __syncthreads();
    if ((t & 63u) == 0) s_red[t >> 6] = w;
    __syncthreads();
    u64 m = 0;
    for (int q = 0; q < BNWAVE; ++q) m = max(m, s_red[q]);
    top[k] = m;
  }
  if (t == 0) {
    double *info = M.info + (u64)d.eslot * SPAN_INFO;
#pragma unroll
    for (u32 k = 0; k < SPAN_NW; ++k)
      info[k] = top[k] ? __longlong_as_double((long long)~top[k]) : 1e308;
    info[SPAN_NW] = __longlong_as_double((long long)top[SPAN_NW]);
    info[SPAN_NW + 1] = fmax(fabs(decode_pos(key[0])), fabs(decode_pos(key[n - 1])));
  }
  if (d.nwin > 1)
    for (u32 i = t; i < 3 * SPAN_SLOTS; i += BWT)
      M.vmax[(u64)d.vslot * 3u * SPAN_SLOTS + i] =
          i == (ep % 3u) * SPAN_SLOTS ? top[SPAN_NW] : 0ull;
}

// WINDOWS: with windows, launched after those of interval iv.  Simulations in
// windows only take part when one failed: the rest of the interval from the
// failed launch's input, then window_form.
template <bool WINDOWS>
__global__ __launch_bounds__(BWT) void k_batch_advance(
    const BatchDesc *__restrict__ descs, BatchArrays A, u32 *err, SpanMany M, u32 iv) {
  extern __shared__ u64 lds_dyn[];
  Lds<BSH, false> s(lds_dyn);
  __shared__ u64 s_red[BNWAVE];
  __shared__ u64 s_mm[2 * BNWAVE];
  __shared__ u32 s_flag;
  __shared__ u64 s_last[2];
  const BatchDesc d = descs[blockIdx.x];
  const u32 t = threadIdx.x;
  const u32 n = d.n;
  if (d.nleap <= 0 || n == 0) return;
  const bool eq = d.flags & 1u;
  const double hh = d.h / 2.;
  // the sets that interval iv since the descriptors' upload starts and ends in
  const u32 per = d.L ? d.L : (u32)d.nleap;
  int a = d.cur ^ (int)((iv * per) & 1u), step0 = 0;
  const int end = a ^ (int)(per & 1u);
  if (WINDOWS) {
    if (d.L) {
      const u32 f = M.fail[d.eslot];
      if (f == 0) return;
      if (t == 0 && d.nwin > 1) M.intact[d.eslot] = 0;
      step0 = (int)((f - 1u) * d.K);
      a ^= (int)((f - 1u) & 1u);
    }
  }

  if (n <= (u32)BLOCK) {
    // ---- the whole simulation in LDS for the interval ------------------------
    u64 *key = A.key[a] + d.off;
    double *vel = A.vel[a] + d.off;
    i32 *idx = A.idx[a] + d.off;
    double *mass = eq ? nullptr : A.mass[a] + d.off;
#pragma unroll
    for (int i = 0; i < BPER; ++i) {
      const u32 e = i * BWT + t;
      if (e < n) {
        const double v = vel[e];
        // first half drift
        s.key[e] = step0 ? key[e] : encode_pos(decode_pos(key[e]) + hh * v);
        s.v[e] = v;
        s.id[e] = idx[e];
        s.m[e] = mass ? mass[e] : 0.0;
      }
    }
    __syncthreads();
    for (int step = step0; step < d.nleap; ++step) {
      lds_bucket_sort<BSH, false>(s, n, s_red, s_mm, nullptr);
      (void)block_leap(s, d, n, 0, 0, step == d.nleap - 1 ? hh : d.h, s_red);
    }
    const int b = end;
    u64 *ko = A.key[b] + d.off;
    double *vo = A.vel[b] + d.off;
    i32 *io = A.idx[b] + d.off;
    double *mo = eq ? nullptr : A.mass[b] + d.off;
#pragma unroll
    for (int i = 0; i < BPER; ++i) {
      const u32 r = i * BWT + t;
      if (r < n) {
        const u32 e = s.ord[r];
        ko[r] = s.key[e];
        vo[r] = s.v[e];
        io[r] = s.id[e];
        if (mo) mo[r] = s.m[e];
      }
    }
    if (WINDOWS && d.L) {
      __syncthreads();
      window_form(s, d, A, M, end, (iv + 1) * d.L, err, s_red, s_mm, &s_flag);
      if (t == 0) M.fail[d.eslot] = 0;
    }
    return;
  }

  // ---- larger simulations: arena-resident, block odd-even merge sort ---------
  if (step0 == 0) {  // first half drift, in place
    u64 *key = A.key[a] + d.off;
    const double *vel = A.vel[a] + d.off;
    for (u32 i = t; i < n; i += BWT) key[i] = encode_pos(decode_pos(key[i]) + hh * vel[i]);
    __syncthreads();
  }
  for (int step = step0; step < d.nleap; ++step) {
    u64 *key = A.key[a] + d.off;
    double *vel = A.vel[a] + d.off;
    i32 *idx = A.idx[a] + d.off;
    double *mass = eq ? nullptr : A.mass[a] + d.off;
    {  // one sliding pass; else the full sort below
      const int b = a ^ 1;
      if (slide_step(s, d, n, key, vel, idx, mass, A.key[b] + d.off,
                     A.vel[b] + d.off, A.idx[b] + d.off,
                     eq ? nullptr : A.mass[b] + d.off,
                     step == d.nleap - 1 ? hh : d.h, s_red, s_mm, &s_flag,
                     s_last)) {
        a = b;
        continue;
      }
    }
    const bool sorted = range_sort(s, n, key, vel, idx, mass, s_red, s_mm, &s_flag);
    if (!sorted && t == 0) atomicOr(err + d.eslot, 1u);  // not expected: bound above
    // force, kick, drift, block by block, into the other buffer set
    const int b = a ^ 1;
    u64 *ko = A.key[b] + d.off;
    double *vo = A.vel[b] + d.off;
    i32 *io = A.idx[b] + d.off;
    double *mo = eq ? nullptr : A.mass[b] + d.off;
    const double hd = step == d.nleap - 1 ? hh : d.h;
    u64 run = 0;
    for (u32 lo = 0; lo < n; lo += BLOCK) {
      const u32 c = min((u32)BLOCK, n - lo);
#pragma unroll
      for (int i = 0; i < BPER; ++i) {
        const u32 e = i * BWT + t;
        if (e < c) {
          s.key[e] = key[lo + e];
          s.v[e] = vel[lo + e];
          s.id[e] = idx[lo + e];
          s.m[e] = mass ? mass[lo + e] : 0.0;
          s.ord[e] = (unsigned short)e;
        }
      }
      __syncthreads();
      run = block_leap(s, d, c, lo, run, hd, s_red);
#pragma unroll
      for (int i = 0; i < BPER; ++i) {
        const u32 e = i * BWT + t;
        if (e < c) {
          ko[lo + e] = s.key[e];
          vo[lo + e] = s.v[e];
          io[lo + e] = s.id[e];
          if (mo) mo[lo + e] = s.m[e];
        }
      }
      __syncthreads();
    }
    a = b;
  }
  if (WINDOWS && d.L) {
    if (a != end) {
      for (u32 i = t; i < n; i += BWT) {
        const u64 p = d.off + i;
        A.key[end][p] = A.key[a][p];
        A.vel[end][p] = A.vel[a][p];
        A.idx[end][p] = A.idx[a][p];
        if (!eq) A.mass[end][p] = A.mass[a][p];
      }
      __syncthreads();
    }
    window_form(s, d, A, M, end, (iv + 1) * d.L, err, s_red, s_mm, &s_flag);
    if (t == 0) M.fail[d.eslot] = 0;
  }
}

// Every simulation's current set into the windows' form, before a plan's first
// interval.
__global__ __launch_bounds__(BWT) void k_batch_form(const BatchDesc *__restrict__ descs,
                                                    BatchArrays A, SpanMany M, u32 *err) {
  extern __shared__ u64 lds_dyn[];
  Lds<BSH, false> s(lds_dyn);
  __shared__ u64 s_red[BNWAVE];
  __shared__ u64 s_mm[2 * BNWAVE];
  __shared__ u32 s_flag;
  const BatchDesc d = descs[blockIdx.x];
  const u32 t = threadIdx.x;
  window_form(s, d, A, M, d.cur, 0u, err, s_red, s_mm, &s_flag);
  if (t == 0) {
    M.fail[d.eslot] = 0;
    M.intact[d.eslot] = 1;
  }
}

}  // namespace

void batch_desc_fill(BatchDesc &d, const double *m, u32 n, double totmass,
                     double omega2) {
  bool eq = true;
  for (u32 i = 1; i < n && eq; ++i) eq = m[i] == m[0];
  d.off = 0;
  d.n = n;
  d.flags = (eq ? 1u : 0u) | (omega2 >= 0.0 ? 2u : 0u);
  d.cur = 0;
  d.nleap = 0;
  d.eslot = 0;
  d.T = d.H = d.nwin = d.K = d.L = d.vslot = d.id0 = 0;
  d.h = 0.0;
  d.mq = m[0];
  d.totmass = totmass;
  d.omega2 = omega2 >= 0.0 ? omega2 : -1.0;
  // fixed-point scale of the exact prefix: 2^k * totmass <= 2^62
  int e = 0;
  (void)frexp(totmass > 0.0 ? totmass : 1.0, &e);
  d.fscale = ldexp(1.0, 62 - e);
  d.finv = ldexp(1.0, e - 62);
}

int batch_launch(hipStream_t st, const BatchDesc *d_descs, int count,
                 const BatchArrays &arr, u32 *err, const SpanMany *many, u32 iv) {
  if (count <= 0) return WDY_OK;
  const size_t lds = Lds<BSH, false>::BYTES;
  auto fn = many ? k_batch_advance<true> : k_batch_advance<false>;
  WDY_HIP(hipFuncSetAttribute((const void *)fn,
                              hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds));
  fn<<<count, BWT, lds, st>>>(d_descs, arr, err, many ? *many : SpanMany{}, iv);
  WDY_CHECK_LAUNCH();
  return WDY_OK;
}

}  // namespace wdy

// ============================================================================
// Host side: the wdy_batch handle
// ============================================================================
namespace wdy {
namespace {

// (idx2: the set that is written first, so that it never holds anything else)
__global__ void k_batch_init(u64 n, const double *__restrict__ x,
                             u64 *__restrict__ key, i32 *__restrict__ idx,
                             i32 *__restrict__ idx2) {
  const u64 i = (u64)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  key[i] = encode_pos(x[i]);
  idx[i] = idx2[i] = (i32)i;
}

// One workgroup per descriptor: de-sort its current set into x_out, v_out
// (arena order, i.e. each simulation's sheets in input order).
__global__ void k_batch_desort(const BatchDesc *__restrict__ descs,
                               BatchArrays A, u32 iv, double *__restrict__ xo,
                               double *__restrict__ vo) {
  const BatchDesc d = descs[blockIdx.x];
  const int c = d.cur ^ (int)((iv * (d.L ? d.L : (u32)d.nleap)) & 1u);
  for (u32 i = threadIdx.x; i < d.n; i += blockDim.x) {
    const u64 p = d.off + i;
    const i32 j = A.idx[c][p];
    xo[j] = decode_pos(A.key[c][p]);
    vo[j] = A.vel[c][p];
  }
}

}  // namespace
}  // namespace wdy

using namespace wdy;

struct wdy_batch {
  int device = 0;
  hipStream_t stream = nullptr;
  int64_t nsims = 0;
  u64 ntot = 0;
  BatchArrays arr{};
  BatchDesc *d_desc = nullptr;
  std::vector<BatchDesc> h_desc;  // launch order: largest first, as uploaded
  u32 iv = 0;                     // intervals since that upload
  // windows
  SpanMany many{};
  bool planned = false;  // for these step parameters
  int shape = -1;        // -1: no simulation in windows
  u32 neq = 0, nun = 0;  // windows of the equal and the unequal simulations
  u32 launches = 0;
  uint2 *d_list = nullptr;
  std::vector<double> reach;  // per descriptor
  double *out_x = nullptr, *out_v = nullptr;
  u32 *err = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  double h = -1.0;
  int nleap = -1;
};

static void batch_free(wdy_batch *b) {
  if (!b) return;
  for (int s = 0; s < 2; ++s) {
    if (b->arr.key[s]) (void)hipFree(b->arr.key[s]);
    if (b->arr.vel[s]) (void)hipFree(b->arr.vel[s]);
    if (b->arr.idx[s]) (void)hipFree(b->arr.idx[s]);
    if (b->arr.mass[s]) (void)hipFree(b->arr.mass[s]);
  }
  for (u64 *p : b->many.cf)
    if (p) (void)hipFree(p);
  if (b->many.vmax) (void)hipFree(b->many.vmax);
  if (b->many.fail) (void)hipFree(b->many.fail);
  if (b->many.info) (void)hipHostFree(b->many.info);
  if (b->d_list) (void)hipFree(b->d_list);
  if (b->d_desc) (void)hipFree(b->d_desc);
  if (b->out_x) (void)hipFree(b->out_x);
  if (b->out_v) (void)hipFree(b->out_v);
  if (b->err) (void)hipFree(b->err);
  if (b->ev0) (void)hipEventDestroy(b->ev0);
  if (b->ev1) (void)hipEventDestroy(b->ev1);
  if (b->stream) (void)hipStreamDestroy(b->stream);
  delete b;
}

static int batch_upload(wdy_batch *b) {
  WDY_HIP(hipMemcpyAsync(b->d_desc, b->h_desc.data(), b->h_desc.size() * sizeof(BatchDesc),
                         hipMemcpyHostToDevice, b->stream));
  WDY_HIP(hipStreamSynchronize(b->stream));
  return WDY_OK;
}

// Every simulation's current set into the windows' form.
static int batch_form(wdy_batch *b) {
  const size_t lds = Lds<BSH, false>::BYTES;
  WDY_HIP(hipFuncSetAttribute((const void *)k_batch_form,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  k_batch_form<<<(unsigned)b->h_desc.size(), BWT, lds, b->stream>>>(b->d_desc, b->arr,
                                                                    b->many, b->err);
  WDY_CHECK_LAUNCH();
  return WDY_OK;
}

// Windows for the step parameters that batch_plan has set.
static int batch_windows(wdy_batch *b) {
  std::vector<BatchDesc> &d = b->h_desc;
  SpanMany &m = b->many;
  const size_t S = d.size();
  if (!m.fail) WDY_HIP(hipMalloc(&m.fail, S * 4));
  if (!m.info)
    WDY_HIP(hipHostMalloc((void **)&m.info, S * (SPAN_INFO * 8 + 4), hipHostMallocDefault));
  m.intact = (u32 *)(m.info + S * SPAN_INFO);
  for (u64 *&p : m.cf)
    if (b->arr.mass[0] && !p) WDY_HIP(hipMalloc(&p, b->ntot * 8));
  if (int rc = batch_form(b)) return rc;
  WDY_HIP(hipStreamSynchronize(b->stream));
  int shape = -1;
  span_many_plan(d, m.info, b->reach, b->h, b->nleap, &shape);
  if (shape < 0) return batch_upload(b);
  std::vector<uint2> list[2];
  size_t words = 0;
  b->launches = 0;
  for (size_t k = 0; k < S; ++k) {
    for (u32 j = 0; d[k].L && j < d[k].nwin; ++j)
      list[d[k].flags & 1u ? 0 : 1].push_back(make_uint2((u32)k, j));
    words += d[k].nwin > 1 ? 1 : 0;
    b->launches = std::max(b->launches, d[k].L);
  }
  b->neq = (u32)list[0].size();
  b->nun = (u32)list[1].size();
  list[0].insert(list[0].end(), list[1].begin(), list[1].end());
  if (b->d_list) WDY_HIP(hipFree(b->d_list));
  b->d_list = nullptr;
  WDY_HIP(hipMalloc(&b->d_list, list[0].size() * sizeof(uint2)));
  WDY_HIP(hipMemcpyAsync(b->d_list, list[0].data(), list[0].size() * sizeof(uint2),
                         hipMemcpyHostToDevice, b->stream));
  if (m.vmax) WDY_HIP(hipFree(m.vmax));
  m.vmax = nullptr;
  WDY_HIP(hipMalloc(&m.vmax, (words ? words : 1) * SPAN_SLOTS * 3 * 8));
  if (int rc = batch_upload(b)) return rc;
  // the speed words of the plan's first launch
  if (int rc = batch_form(b)) return rc;
  b->shape = shape;
  return WDY_OK;
}

// Step parameters and, if asked for, windows; without memory for those the
// workgroup-per-simulation kernel goes on.
static int batch_plan(wdy_batch *b, double h, int nleap, bool windows) {
  std::vector<BatchDesc> &d = b->h_desc;
  WDY_HIP(hipStreamSynchronize(b->stream));
  for (size_t k = 0; k < d.size(); ++k) {
    BatchDesc &q = d[k];
    q.cur ^= (int)((b->iv * (q.L ? q.L : (u32)q.nleap)) & 1u);
    if (b->shape >= 0 && q.L) {
      if (b->many.intact[k] == 0) b->reach[k] *= 1.6;
    }
    q.L = q.nwin = 0;
    q.h = h;
    q.nleap = nleap;
  }
  b->iv = 0;
  b->h = h;
  b->nleap = nleap;
  b->shape = -1;
  if (int rc = batch_upload(b)) return rc;
  b->planned = windows;
  if (!windows) return WDY_OK;
  int rc;
  try {
    rc = batch_windows(b);
  } catch (const std::bad_alloc &) {  // the list of them, on the host
    rc = WDY_ENOMEM;
  }
  if (!rc) return WDY_OK;
  (void)hipGetLastError();  // else the next launch's check finds it
  for (BatchDesc &q : d) q.L = q.nwin = 0;  // from where it is
  const int ru = batch_upload(b);
  return rc == WDY_ENOMEM ? ru : rc;
}

extern "C" {

int wdy_batch_create(int64_t nsims, const int64_t *offsets, const double *x,
                     const double *v, const double *m, const double *totmass,
                     const double *omega2, wdy_batch **out) {
  if (!out) return fail(WDY_EINVAL, "wdy_batch_create: out is NULL");
  *out = nullptr;
  if (nsims < 1 || !offsets || !x || !v || !m || !totmass || !omega2)
    return fail(WDY_EINVAL, "wdy_batch_create: bad arguments");
  if (offsets[0] != 0)
    return fail(WDY_EINVAL, "wdy_batch_create: offsets[0] must be 0");
  for (int64_t k = 0; k < nsims; ++k) {
    if (offsets[k + 1] <= offsets[k])
      return fail(WDY_EINVAL, "wdy_batch_create: simulation %lld is empty or "
                  "offsets decrease", (long long)k);
    if (!std::isfinite(totmass[k]) || !std::isfinite(omega2[k]))
      return fail(WDY_EINVAL, "wdy_batch_create: non-finite totmass/omega2 of "
                  "simulation %lld", (long long)k);
  }
  const int64_t ntot = offsets[nsims];
  if (ntot >= (int64_t(1) << 31))
    return fail(WDY_EINVAL, "wdy_batch_create: %lld sheets in total, limit 2^31",
                (long long)ntot);
  for (int64_t i = 0; i < ntot; ++i)
    if (!std::isfinite(x[i]) || !std::isfinite(v[i]) || !std::isfinite(m[i]) ||
        m[i] < 0.0)
      return fail(WDY_EINVAL, "wdy_batch_create: non-finite or negative input "
                  "at sheet %lld", (long long)i);
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
    return fail(WDY_ENODEV, "wdy_batch_create: no GPU visible");
  wdy_batch *b = new (std::nothrow) wdy_batch();
  if (!b) return fail(WDY_ENOMEM, "wdy_batch_create: host allocation failed");
  int rc = [&]() -> int {
    WDY_HIP(hipGetDevice(&b->device));
    WDY_HIP(hipStreamCreate(&b->stream));
    WDY_HIP(hipEventCreate(&b->ev0));
    WDY_HIP(hipEventCreate(&b->ev1));
    b->nsims = nsims;
    b->ntot = (u64)ntot;
    bool any_unequal = false;
    std::vector<BatchDesc> descs((size_t)nsims);
    for (int64_t k = 0; k < nsims; ++k) {
      BatchDesc &d = descs[(size_t)k];
      batch_desc_fill(d, m + offsets[k], (u32)(offsets[k + 1] - offsets[k]),
                      totmass[k], omega2[k]);
      d.off = (u64)offsets[k];
      d.id0 = (u32)offsets[k];
      any_unequal = any_unequal || !(d.flags & 1u);
    }
    std::stable_sort(descs.begin(), descs.end(),
                     [](const BatchDesc &p, const BatchDesc &q) { return p.n > q.n; });
    for (size_t k = 0; k < descs.size(); ++k) descs[k].eslot = (u32)k;
    b->h_desc = descs;
    b->reach.assign(descs.size(), 1.0);
    const size_t N = (size_t)ntot;
    for (int s = 0; s < 2; ++s) {
      WDY_HIP(hipMalloc(&b->arr.key[s], N * 8));
      WDY_HIP(hipMalloc(&b->arr.vel[s], N * 8));
      WDY_HIP(hipMalloc(&b->arr.idx[s], N * 4));
      if (any_unequal) WDY_HIP(hipMalloc(&b->arr.mass[s], N * 8));
    }
    WDY_HIP(hipMalloc(&b->d_desc, descs.size() * sizeof(BatchDesc)));
    WDY_HIP(hipMalloc(&b->out_x, N * 8));
    WDY_HIP(hipMalloc(&b->out_v, N * 8));
    WDY_HIP(hipMalloc(&b->err, (size_t)nsims * 4));
    WDY_HIP(hipMemsetAsync(b->err, 0, (size_t)nsims * 4, b->stream));
    WDY_HIP(hipMemcpyAsync(b->d_desc, descs.data(), descs.size() * sizeof(BatchDesc),
                           hipMemcpyHostToDevice, b->stream));
    WDY_HIP(hipMemcpyAsync(b->out_x, x, N * 8, hipMemcpyHostToDevice, b->stream));
    WDY_HIP(hipMemcpyAsync(b->arr.vel[0], v, N * 8, hipMemcpyHostToDevice, b->stream));
    if (any_unequal)
      WDY_HIP(hipMemcpyAsync(b->arr.mass[0], m, N * 8, hipMemcpyHostToDevice,
                             b->stream));
    k_batch_init<<<(unsigned)((N + 255) / 256), 256, 0, b->stream>>>(
        (u64)N, b->out_x, b->arr.key[0], b->arr.idx[0], b->arr.idx[1]);
    WDY_CHECK_LAUNCH();
    WDY_HIP(hipStreamSynchronize(b->stream));
    return WDY_OK;
  }();
  if (rc) {
    batch_free(b);
    return rc;
  }
  *out = b;
  return WDY_OK;
}

int wdy_batch_advance(wdy_batch *b, double h, int nleap) {
  if (!b) return fail(WDY_EINVAL, "wdy_batch_advance: batch is NULL");
  if (nleap < 1 || !std::isfinite(h))
    return fail(WDY_EINVAL, "wdy_batch_advance: bad h or nleap");
  WDY_HIP(hipSetDevice(b->device));
  const bool change = h != b->h || nleap != b->nleap;
  // A batch's first interval puts every simulation in order; from the second
  // interval of the same steps on it runs in windows.  (A plan sorts every
  // simulation twice in one workgroup each: with steps that change with every
  // interval, 64 disks of 256 to 32768 sheets took 723 us an interval of one step
  // in windows, 228 without.)  A plan stays until h or nleap changes or a window
  // failed (the reports are the host's to read at any time: they only say when
  // to look again).
  bool plan = change || !b->planned;
  if (!plan && b->shape >= 0)
    for (size_t k = 0; k < b->h_desc.size() && !plan; ++k)
      plan = b->h_desc[k].L != 0 && b->many.intact[k] == 0;
  if (plan)
    if (int rc = batch_plan(b, h, nleap, !change)) return rc;
  WDY_HIP(hipEventRecord(b->ev0, b->stream));
  if (b->shape >= 0)
    for (u32 q = 0; q < b->launches; ++q)
      if (int rc = span_many_launch(b->stream, b->shape, b->d_desc, b->d_list, b->neq,
                                    b->nun, b->arr, b->many, q, b->iv))
        return rc;
  if (int rc = batch_launch(b->stream, b->d_desc, (int)b->nsims, b->arr, b->err,
                            b->shape >= 0 ? &b->many : nullptr, b->iv))
    return rc;
  ++b->iv;
  WDY_HIP(hipEventRecord(b->ev1, b->stream));
  return WDY_OK;
}

int wdy_batch_read(wdy_batch *b, double *x_out, double *v_out,
                   double *seconds_out) {
  if (!b) return fail(WDY_EINVAL, "wdy_batch_read: batch is NULL");
  WDY_HIP(hipSetDevice(b->device));
  const size_t N = (size_t)b->ntot;
  if (x_out || v_out) {
    k_batch_desort<<<(unsigned)b->nsims, 256, 0, b->stream>>>(
        b->d_desc, b->arr, b->iv, b->out_x, b->out_v);
    WDY_CHECK_LAUNCH();
    if (x_out)
      WDY_HIP(hipMemcpyAsync(x_out, b->out_x, N * 8, hipMemcpyDeviceToHost,
                             b->stream));
    if (v_out)
      WDY_HIP(hipMemcpyAsync(v_out, b->out_v, N * 8, hipMemcpyDeviceToHost,
                             b->stream));
  }
  std::vector<u32> errs((size_t)b->nsims);
  WDY_HIP(hipMemcpyAsync(errs.data(), b->err, errs.size() * 4, hipMemcpyDeviceToHost,
                         b->stream));
  WDY_HIP(hipStreamSynchronize(b->stream));
  u32 err = 0;
  for (u32 e : errs) err |= e;
  if (err)
    return fail(WDY_EVERIFY, "wdy_batch_read: a simulation did not sort within "
                "its bound");
  if (seconds_out) {
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, b->ev0, b->ev1) != hipSuccess) {  // none has run yet
      (void)hipGetLastError();  // else the next launch's check finds it
      ms = 0.f;
    }
    *seconds_out = ms * 1e-3;
  }
  return WDY_OK;
}

int wdy_batch_destroy(wdy_batch *b) {
  if (!b) return WDY_OK;
  (void)hipSetDevice(b->device);
  (void)hipStreamSynchronize(b->stream);
  batch_free(b);
  return WDY_OK;
}

}  // extern "C"
