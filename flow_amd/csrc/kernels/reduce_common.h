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
 * candidates), then 8 64-bit words per block of the kernel that leaves the
 * totals (publish_totals; the kernels with plain compensated sums use 4). */
constexpr int kTotalsOffset = 2 * kMaxReduceBlocks;
constexpr int kTotalsWords = 8;
constexpr int kPartialsDoubles = kTotalsOffset + kTotalsWords * kMaxReduceBlocks;

/* The cells of a local nx x ny array inside its pad, numbered in row-major
 * order; none where the pad leaves none (set_timestep and print_conservation
 * take the sizes from their caller). Unsigned 32-bit numbers: the largest
 * mesh's interior has fewer than 2^31 cells, so a number and a grid's stride
 * past it fit, and a cell costs one 32-bit division. */
struct Interior {
  int pad;
  unsigned int wx, n;
  __host__ __device__ Interior(int nx, int ny, int pad_) : pad(pad_), wx(1), n(0) {
    if (nx <= 2 * pad || ny <= 2 * pad) return;
    wx = (unsigned int)(nx - 2 * pad);
    n = wx * (unsigned int)(ny - 2 * pad);
  }
  __host__ __device__ int row(unsigned int k) const { return pad + (int)(k / wx); }
  __host__ __device__ int col(unsigned int k) const { return pad + (int)(k % wx); }
};

/* (of a block of at most NT threads) */
template <int NT>
__device__ __forceinline__ double block_min(double x, int waves = NT / kWave) {
  __shared__ double red[NT / kWave];
  x = wave_min(x);
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
  __syncthreads();
  if (lane == 0) red[w] = x;
  __syncthreads();
  if (w == 0) {
    x = (lane < waves) ? red[lane] : red[0];
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

/* A block's CFL minimum and its count of undefined candidates (at most NT
 * threads). */
template <int NT>
__device__ __forceinline__ void publish_min(double local_min, int nan_count, FkReduce r,
                                            int waves = NT / kWave) {
  __shared__ int s_nan[NT / kWave];
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
  /* almost always none */
  if (__ballot(nan_count != 0)) nan_count = wave_sum(nan_count);
  if (lane == 0) s_nan[w] = nan_count;
  const double bmin = block_min<NT>(local_min, waves);
  if (threadIdx.x == 0) {
    int bad = 0;
    for (int k = 0; k < waves; ++k) bad += s_nan[k];
    r.partials[2 * blockIdx.x] = bmin;
    r.partials[2 * blockIdx.x + 1] = (double)bad;
  }
}

/* The minimum over parts blocks' partials and max_dt, the same in every thread
 * of the block (at most 16 waves), and their undefined candidates, valid in
 * thread 0. The block shares the loads out: one or two a thread in flight at
 * once, then one barrier. (With each wave folding all of them for itself, the
 * batches of loads took 7800 of the 16100 cycles that a block of the
 * mass/energy kernel runs for on a 512^2 mesh.) kSquared: the candidates are
 * squared time steps (the FP32-state form); the minimum's square root is
 * taken once, here. */
struct MinFold {
  double g;
  int bad;
};
template <bool kSquared>
__device__ __forceinline__ MinFold fold_min(const FkReduce& r, int parts, double max_dt) {
  __shared__ double s_min[16];
  __shared__ int s_bad[16];
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave, waves = blockDim.x / kWave;
  double g = kSquared ? max_dt * max_dt : max_dt;
  int bad = 0;
#pragma unroll 4
  for (int b = threadIdx.x; b < parts; b += blockDim.x) {
    g = lesser(g, r.partials[2 * b]);
    bad += (int)r.partials[2 * b + 1];
  }
  g = wave_min(g);
  if (__ballot(bad != 0)) bad = wave_sum(bad);
  if (lane == 0) {
    s_min[w] = g;
    s_bad[w] = bad;
  }
  __syncthreads();
  g = wave_min(s_min[lane < waves ? lane : 0]);
  if (threadIdx.x == 0)
    for (int k = 1; k < waves; ++k) bad += s_bad[k];
  return MinFold{kSquared ? __builtin_sqrt(g) : g, bad};
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
    const double mag = __builtin_fabs(v);
    unsigned long long a0 = 0, a1 = 0, a2 = 0;
    if (mag < 0x1p62) {
      /* whole part and fraction, each converted exactly (bits of the
       * fraction below 2^-64 are cut off) */
      a1 = (unsigned long long)mag;
      a0 = (unsigned long long)((mag - (double)a1) * 0x1p64);
    } else if (!words(v, a0, a1, a2)) {
      return;
    }
    if (v < 0.0) {
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

  /* |v| >= 2^62 in units of 2^-64; false, and the sum marked bad, if it is
   * out of range */
  __host__ __device__ bool words(double v, unsigned long long& a0, unsigned long long& a1,
                                 unsigned long long& a2) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned int E = (unsigned int)(u >> 52) & 0x7ffu;
    if (E >= 1023u + 127u) { /* |v| >= 2^127, inf or NaN */
      bad = 1u;
      return false;
    }
    const unsigned long long M = (u & 0xfffffffffffffull) | (1ull << 52);
    const int s = (int)E - 1075 + 64; /* |v| = M 2^(s - 64), 73 <= s <= 138 */
    if (s < 128) {
      const int t = s - 64;
      a1 = M << t;
      a2 = M >> (64 - t);
    } else {
      a2 = M << (s - 128);
    }
    return true;
  }
};

/* a += b, modulo 2^192 */
struct Words192 {
  unsigned long long w0, w1, w2;
};
__host__ __device__ __forceinline__ void add192(Words192& a, const Words192& b) {
  a.w0 += b.w0;
  const unsigned long long c0 = a.w0 < b.w0;
  const unsigned long long t = a.w1 + b.w1;
  const unsigned long long c1 = t < b.w1;
  a.w1 = t + c0;
  a.w2 += b.w2 + c1 + (a.w1 < c0);
}

/* The sum over the wave (all lanes active), valid in lane 63. */
__device__ __forceinline__ Words192 wave_sum192(Words192 x) {
#define FLOWHIP_ADD_STEP(ctrl, rows)                                              \
  add192(x, Words192{dpp_step<ctrl, rows>(0ull, x.w0), dpp_step<ctrl, rows>(0ull, x.w1), \
                     dpp_step<ctrl, rows>(0ull, x.w2)});
  FLOWHIP_DPP_STEPS(FLOWHIP_ADD_STEP)
#undef FLOWHIP_ADD_STEP
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

/* Per-lane exact totals (rho in fm, rho * e in fe) -> the block's 8 words:
 * mass, its bad mark, energy, its bad mark. Integer addition is associative,
 * so the totals are the same bits whichever waves and blocks added which
 * values. (As 14 sums of 32-bit limbs through shuffles this took 7800
 * cycles, a quarter of the mass/energy march of a 512^2 mesh.) */
template <int NT>
__device__ void publish_totals(const FixSum& fm, const FixSum& fe, FkReduce r) {
  __shared__ Words192 part[NT / kWave][2];
  __shared__ unsigned int s_bad[NT / kWave][2];
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
  const Words192 m = wave_sum192(Words192{fm.w0, fm.w1, fm.w2});
  const Words192 e = wave_sum192(Words192{fe.w0, fe.w1, fe.w2});
  const bool bm = __ballot(fm.bad != 0u) != 0ull, be = __ballot(fe.bad != 0u) != 0ull;
  if (lane == kWave - 1) {
    part[w][0] = m;
    part[w][1] = e;
    s_bad[w][0] = bm;
    s_bad[w][1] = be;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    Words192 t = part[0][threadIdx.x];
    unsigned int bad = s_bad[0][threadIdx.x];
    for (int k = 1; k < NT / kWave; ++k) {
      add192(t, part[k][threadIdx.x]);
      bad |= s_bad[k][threadIdx.x];
    }
    unsigned long long* p = (unsigned long long*)(r.partials + kTotalsOffset) +
                            kTotalsWords * blockIdx.x + 4 * threadIdx.x;
    p[0] = t.w0;
    p[1] = t.w1;
    p[2] = t.w2;
    p[3] = bad;
  }
}

/* A value of the dt pair (k 0, 1), a total (2, 3) or the undefined
 * candidates (4), for the host. */
__device__ __forceinline__ void post(const FkReduce& r, int k, double v) {
  if (r.mail) r.mail[k] = v;
}

/* The totals of parts blocks' words -> r.sums[0..1], by the first NT threads of
 * one block: the first half the mass, the second the energy. */
template <int NT>
__device__ void fold_totals(const FkReduce& r, int parts) {
  constexpr int kHalf = NT / 2;
  __shared__ Words192 s_sum[NT / kWave];
  __shared__ unsigned int s_bad[NT / kWave];
  const int q = threadIdx.x / kHalf, lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
  const unsigned long long* p =
      (const unsigned long long*)(r.partials + kTotalsOffset) + 4 * q;
  Words192 t{0, 0, 0};
  unsigned long long any = 0;
#pragma unroll 2
  for (int b = threadIdx.x % kHalf; q < 2 && b < parts; b += kHalf) {
    const unsigned long long* v = p + kTotalsWords * b;
    add192(t, Words192{v[0], v[1], v[2]});
    any |= v[3];
  }
  t = wave_sum192(t);
  const bool bad = __ballot(any != 0ull) != 0ull;
  if (q < 2 && lane == kWave - 1) {
    s_sum[w] = t;
    s_bad[w] = bad;
  }
  __syncthreads();
  if (q < 2 && threadIdx.x % kHalf == 0) {
    constexpr int kPer = kHalf / kWave;
    Words192 s = s_sum[q * kPer];
    unsigned int b = s_bad[q * kPer];
    for (int k = 1; k < kPer; ++k) {
      add192(s, s_sum[q * kPer + k]);
      b |= s_bad[q * kPer + k];
    }
    const unsigned long long limb[7] = {
        s.w0 & 0xffffffffull, s.w0 >> 32, s.w1 & 0xffffffffull, s.w1 >> 32,
        s.w2 & 0xffffffffull, s.w2 >> 32, (unsigned long long)b};
    const double v = fixed_total(limb);
    r.sums[q] = v;
    post(r, 2 + q, v);
  }
}

}  // namespace flowhip
