/*
 * reduce_common.h -- block-level reductions, the partials that blocks leave
 * for the next kernel and their folds, shared by the reduction kernels, the
 * fused kernels and the march kernels: the CFL minimum, compensated
 * per-block totals, and exact fixed-point totals.
 */
#pragma once

#include "common.h"
#include "hydro_math.h"

namespace flowhip {

/* Upper bound on blocks of any launch that leaves reduction partials in
 * FkReduce.partials. */
constexpr int kMaxReduceBlocks = 2048;
/* Layout of FkReduce.partials, in doubles: two per block of the kernel that
 * evaluates the CFL candidates (its minimum and its count of undefined
 * candidates), then 14 64-bit words per block of the kernel that leaves the
 * totals (block_limbs; the kernels with plain compensated sums use 4). */
constexpr int kTotalsOffset = 2 * kMaxReduceBlocks;
constexpr int kTotalsWords = 14;
constexpr int kPartialsDoubles = kTotalsOffset + kTotalsWords * kMaxReduceBlocks;

template <int NT>
__device__ __forceinline__ double block_min(double x) {
  __shared__ double red[NT / kWave];
  x = wave_min(x);
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
  __syncthreads();
  if (lane == 0) red[w] = x;
  __syncthreads();
  if (w == 0) {
    x = (lane < NT / kWave) ? red[lane] : red[0];
    x = wave_min(x);
  }
  return x; /* valid in wave 0 */
}

template <int NT>
__device__ __forceinline__ CSum block_csum(CSum v) {
  __shared__ double rs[NT / kWave], rc[NT / kWave];
  v = wave_csum(v);
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
  __syncthreads();
  if (lane == 0) {
    rs[w] = v.s;
    rc[w] = v.c;
  }
  __syncthreads();
  if (w == 0) {
    CSum t{0.0, 0.0};
    if (lane < NT / kWave) t = CSum{rs[lane], rc[lane]};
    v = wave_csum(t);
  }
  return v; /* valid in wave 0 */
}

/* ---- grid reductions ----
 * A block leaves its partial in FkReduce.partials with plain stores and the
 * next kernel on the stream folds them: the kernel boundary orders the two.
 * The single-pass form this replaces (every block fences its partial and
 * takes a ticket, the last one folds) cost 45-60 ns a block on MI355X, one
 * block after the other (each device-scope fence writes back the XCD's L2),
 * at the end of the kernel where nothing overlaps it: the pre-loop
 * set_timestep of a 512^2 mesh (1024 blocks) took 70 us of which 64 were
 * that, the 752-block Lagrangian march of a 1000^2 mesh about 45 of 117. */

/* A block's CFL minimum and its count of undefined candidates. */
template <int NT>
__device__ __forceinline__ void publish_min(double local_min, int nan_count, FkReduce r) {
  __shared__ int s_nan[NT / kWave];
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) nan_count += __shfl_xor(nan_count, off, kWave);
  if (lane == 0) s_nan[w] = nan_count;
  const double bmin = block_min<NT>(local_min);
  if (threadIdx.x == 0) {
    int bad = 0;
    for (int k = 0; k < NT / kWave; ++k) bad += s_nan[k];
    r.partials[2 * blockIdx.x] = bmin;
    r.partials[2 * blockIdx.x + 1] = (double)bad;
  }
}

/* The minimum over parts blocks' partials and max_dt, and the undefined
 * candidates' count; the same in every thread of the block. kSquared: the
 * candidates are squared time steps (the FP32-state form); the minimum's
 * square root is taken once, here. */
template <int NT, bool kSquared>
__device__ __forceinline__ void fold_min(const FkReduce& r, int parts, double max_dt,
                                         double& g_out, double& bad_out) {
  __shared__ double s_min[NT / kWave], s_bad[NT / kWave];
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
  double g = kSquared ? max_dt * max_dt : max_dt, bad = 0.0;
  for (int b = threadIdx.x; b < parts; b += NT) {
    const double2 p = reinterpret_cast<const double2*>(r.partials)[b];
    g = lesser(g, p.x);
    bad += p.y;
  }
  g = wave_min(g);
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) bad += __shfl_xor(bad, off, kWave);
  if (lane == 0) {
    s_min[w] = g;
    s_bad[w] = bad;
  }
  __syncthreads();
  g = s_min[0];
  bad = s_bad[0];
#pragma unroll
  for (int k = 1; k < NT / kWave; ++k) {
    g = lesser(g, s_min[k]);
    bad += s_bad[k];
  }
  g_out = kSquared ? __builtin_sqrt(g) : g;
  bad_out = bad;
}

/* The (dt, dt_h) update of omp3/flow.c:103-105 from the grid minimum g. */
struct DtPair {
  double dt, dt_h;
};
__device__ __forceinline__ DtPair next_pair(double g, double dt_h, int first_step) {
  const double final_min = lesser(g, kCM * dt_h);
  DtPair p;
  p.dt = 0.5 * (kCT * final_min + dt_h);
  p.dt_h = first_step ? p.dt : kCT * final_min;
  return p;
}

/* A block's compensated sums of the mass and energy. */
template <int NT>
__device__ void publish_sums(CSum ms, CSum es, FkReduce r) {
  ms = block_csum<NT>(ms);
  es = block_csum<NT>(es);
  if (threadIdx.x == 0) {
    double* p = r.partials + kTotalsOffset + 4 * blockIdx.x;
    p[0] = ms.s;
    p[1] = ms.c;
    p[2] = es.s;
    p[3] = es.c;
  }
}

/* Exact accumulator for totals: a sum of doubles, each first truncated
 * toward zero to a multiple of 2^-64, held as a 192-bit two's complement
 * integer in units of 2^-64 (w0 the low word). Integer addition is
 * associative, so the sum is the same bits whatever the order or grouping
 * of the additions. Values of magnitude below 2^127 are taken exactly down
 * to 2^-64; a larger or non-finite value marks the sum bad. */
struct FixSum {
  unsigned long long w0, w1, w2;
  unsigned int bad;

  __host__ __device__ void add(double v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned int E = (unsigned int)(u >> 52) & 0x7ffu;
    if (E >= 1023u + 127u) { /* |v| >= 2^127, inf or NaN */
      bad = 1u;
      return;
    }
    const unsigned long long mant = u & 0xfffffffffffffull;
    const unsigned long long M = E ? (mant | (1ull << 52)) : mant;
    /* v = M 2^(s - 64) */
    const int s = (E ? (int)E : 1) - 1075 + 64;
    unsigned long long a0 = 0, a1 = 0, a2 = 0;
    if (s < 0) {
      a0 = s > -64 ? (M >> -s) : 0ull;
    } else if (s < 64) {
      a0 = M << s;
      a1 = s ? (M >> (64 - s)) : 0ull;
    } else if (s < 128) {
      const int t = s - 64;
      a1 = M << t;
      a2 = t ? (M >> (64 - t)) : 0ull;
    } else {
      a2 = M << (s - 128); /* s <= 138: below 2^63 */
    }
    if (u >> 63) {
      const unsigned long long b0 = w0 < a0;
      w0 -= a0;
      const unsigned long long t1 = w1 - a1, b1 = (w1 < a1) + (t1 < b0);
      w1 = t1 - b0;
      w2 -= a2 + b1;
    } else {
      w0 += a0;
      const unsigned long long c0 = w0 < a0;
      const unsigned long long t1 = w1 + a1, c1a = t1 < a1;
      w1 = t1 + c0;
      w2 += a2 + c1a + (w1 < c0);
    }
  }
};

__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long x) {
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) x += __shfl_xor(x, off, kWave);
  return x;
}

/* The double nearest (to within an ulp; the same bits every time) to the
 * fixed-point total held in 6 limb counters t[0..5] (t[k] counts units of
 * 2^(32k - 64), any size below 2^63) and its bad count t[6]. */
__host__ __device__ inline double fixed_total(const unsigned long long* t) {
  if (t[6]) return __builtin_nan("");
  unsigned int d[6];
  unsigned long long c = 0;
  for (int k = 0; k < 6; ++k) {
    const unsigned long long x = t[k] + c;
    d[k] = (unsigned int)x;
    c = x >> 32;
  }
  const bool neg = (d[5] >> 31) != 0;
  if (neg) { /* two's complement negation of the 192-bit value */
    unsigned long long carry = 1;
    for (int k = 0; k < 6; ++k) {
      const unsigned long long x = (unsigned long long)(~d[k]) + carry;
      d[k] = (unsigned int)x;
      carry = x >> 32;
    }
  }
  /* exact parts, largest first, into a compensated sum */
  CSum acc{0.0, 0.0};
  for (int k = 5; k >= 0; --k) acc.add(__builtin_ldexp((double)d[k], 32 * k - 64));
  const double r = acc.s + acc.c;
  return neg ? -r : r;
}

/* Per-lane exact totals (rho in fm, rho * e in fe) -> the block's 14 words:
 * the sums of its lanes' 32-bit limbs (integer sums, in any order) and of
 * the bad marks, mass first. */
template <int NT>
__device__ void publish_limbs(const FixSum& fm, const FixSum& fe, FkReduce r) {
  __shared__ unsigned long long part[NT / kWave][kTotalsWords];
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
  const FixSum* f[2] = {&fm, &fe};
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const unsigned long long limb[7] = {
        f[q]->w0 & 0xffffffffull, f[q]->w0 >> 32, f[q]->w1 & 0xffffffffull,
        f[q]->w1 >> 32,           f[q]->w2 & 0xffffffffull, f[q]->w2 >> 32,
        (unsigned long long)f[q]->bad};
#pragma unroll
    for (int k = 0; k < 7; ++k) {
      const unsigned long long v = wave_sum_u64(limb[k]);
      if (lane == 0) part[w][7 * q + k] = v;
    }
  }
  __syncthreads();
  if (threadIdx.x < kTotalsWords) {
    unsigned long long v = 0;
    for (int b = 0; b < NT / kWave; ++b) v += part[b][threadIdx.x];
    unsigned long long* p = (unsigned long long*)(r.partials + kTotalsOffset);
    p[kTotalsWords * blockIdx.x + threadIdx.x] = v;
  }
}

/* A value of the dt pair (k 0, 1), a total (2, 3) or the undefined
 * candidates (4), for the host. */
__device__ __forceinline__ void post(const FkReduce& r, int k, double v) {
  if (r.mail) r.mail[k] = v;
}

/* The totals of parts blocks' words -> r.sums[0..1], by one block. Thread
 * t < 252 adds word t % 14 of every 18th block, so a wave reads consecutive
 * words. The totals are the same bits whichever waves and blocks added
 * which values. */
template <int NT>
__device__ void fold_limbs(const FkReduce& r, int parts) {
  constexpr int kSlices = NT / kTotalsWords;
  __shared__ unsigned long long s_sum[kSlices][kTotalsWords];
  const unsigned long long* p = (const unsigned long long*)(r.partials + kTotalsOffset);
  const int slice = threadIdx.x / kTotalsWords, word = threadIdx.x % kTotalsWords;
  if (slice < kSlices) {
    unsigned long long v = 0;
#pragma unroll 4
    for (int b = slice; b < parts; b += kSlices) v += p[kTotalsWords * b + word];
    s_sum[slice][word] = v;
  }
  __syncthreads();
  if (threadIdx.x < kTotalsWords) {
    unsigned long long v = 0;
    for (int k = 0; k < kSlices; ++k) v += s_sum[k][threadIdx.x];
    s_sum[0][threadIdx.x] = v;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    const double v = fixed_total(&s_sum[0][7 * threadIdx.x]);
    r.sums[threadIdx.x] = v;
    post(r, 2 + threadIdx.x, v);
  }
}

}  // namespace flowhip
