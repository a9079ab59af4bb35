/*
 * common.h -- launch geometry, index helpers and wave64 reductions shared by
 * the hip kernel set's translation units.
 */
#pragma once

#include <hip/hip_runtime.h>

#include "../../../include/flow_hip_kernels.h"

namespace flowhip {

constexpr int kWave = 64;

/* A rectangular loop domain [r0, r1) x [c0, c1) of a 2-D array. */
struct Domain {
  int r0, r1, c0, c1;
  __host__ __device__ int rows() const { return r1 - r0; }
  __host__ __device__ int cols() const { return c1 - c0; }
};

/* Stagewise kernels: 64 x 4 threads, one point per thread. */
constexpr int kSwX = 64;
constexpr int kSwY = 4;

inline dim3 sw_grid(const Domain& d) {
  const int gx = (d.cols() + kSwX - 1) / kSwX;
  const int gy = (d.rows() + kSwY - 1) / kSwY;
  return dim3(gx > 0 ? gx : 1, gy > 0 ? gy : 1, 1);
}

/* One step of a wave64 reduction as DPP moves: lane i of a row of 16 reads
 * lane i - 1, 2, 4, 8 (row_shr), then rows 1 and 3 read lane 15 of the row
 * before, then rows 2 and 3 read lane 31, so lane 63 ends with the whole
 * wave's. A lane without a source reads old. Register moves, a few cycles
 * each; the shuffles they replace go through LDS, 50 cycles and more a step. */
template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned int dpp_step(unsigned int old, unsigned int v) {
  return (unsigned int)__builtin_amdgcn_update_dpp((int)old, (int)v, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned long long dpp_step(unsigned long long old,
                                                       unsigned long long v) {
  const unsigned int lo = dpp_step<CTRL, ROWS>((unsigned int)old, (unsigned int)v);
  const unsigned int hi =
      dpp_step<CTRL, ROWS>((unsigned int)(old >> 32), (unsigned int)(v >> 32));
  return ((unsigned long long)hi << 32) | lo;
}
/* op(control, row mask) for each step of a wave's reduction */
#define FLOWHIP_DPP_STEPS(op) \
  op(0x111, 0xf) op(0x112, 0xf) op(0x114, 0xf) op(0x118, 0xf) op(0x142, 0xa) op(0x143, 0xc)

/* lane 63's value, in every lane */
__device__ __forceinline__ unsigned long long last_lane(unsigned long long v) {
  const unsigned int lo = __builtin_amdgcn_readlane((int)(unsigned int)v, kWave - 1);
  const unsigned int hi = __builtin_amdgcn_readlane((int)(unsigned int)(v >> 32), kWave - 1);
  return ((unsigned long long)hi << 32) | lo;
}

/* The minimum over the wave (all lanes active), in every lane. */
__device__ __forceinline__ double wave_min(double x) {
#define FLOWHIP_MIN_STEP(ctrl, rows)                                                 \
  {                                                                                  \
    const unsigned long long v = __builtin_bit_cast(unsigned long long, x);          \
    const double y = __builtin_bit_cast(double, (dpp_step<ctrl, rows>(v, v)));       \
    x = (y < x) ? y : x;                                                             \
  }
  FLOWHIP_DPP_STEPS(FLOWHIP_MIN_STEP)
#undef FLOWHIP_MIN_STEP
  return __builtin_bit_cast(double, last_lane(__builtin_bit_cast(unsigned long long, x)));
}

/* The sum over the wave (all lanes active), in every lane. */
__device__ __forceinline__ int wave_sum(int x) {
#define FLOWHIP_SUM_STEP(ctrl, rows) x += (int)dpp_step<ctrl, rows>(0u, (unsigned int)x);
  FLOWHIP_DPP_STEPS(FLOWHIP_SUM_STEP)
#undef FLOWHIP_SUM_STEP
  return __builtin_amdgcn_readlane(x, kWave - 1);
}

/* 1/x for a positive power of two x with a normal reciprocal, exactly: 2^-k
 * has biased exponent 2 * bias - (bias + k), so the reciprocal's bits are a
 * constant minus x's bits. */
__host__ __device__ __forceinline__ double recip_pow2(double x) {
  return __builtin_bit_cast(double, 0x7fe0000000000000ull -
                                        __builtin_bit_cast(unsigned long long, x));
}
__host__ __device__ __forceinline__ float recip_pow2(float x) {
  return __builtin_bit_cast(float, 0x7f000000u - __builtin_bit_cast(unsigned int, x));
}

/* Error-free transformation a + b = s + err (Knuth TwoSum). */
__host__ __device__ __forceinline__ void two_sum(double a, double b, double& s,
                                                 double& err) {
  s = a + b;
  const double bp = s - a;
  const double ap = s - bp;
  err = (a - ap) + (b - bp);
}

/* Compensated accumulator (sum, compensation), merged with TwoSum. */
struct CSum {
  double s, c;
  __host__ __device__ void add(double x) {
    double t, e;
    two_sum(s, x, t, e);
    s = t;
    c += e;
  }
  __host__ __device__ void merge(const CSum& o) {
    double t, e;
    two_sum(s, o.s, t, e);
    s = t;
    c += e + o.c;
  }
};

__device__ __forceinline__ CSum wave_csum(CSum v) {
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    CSum o;
    o.s = __shfl_xor(v.s, off, kWave);
    o.c = __shfl_xor(v.c, off, kWave);
    v.merge(o);
  }
  return v;
}

}  // namespace flowhip
