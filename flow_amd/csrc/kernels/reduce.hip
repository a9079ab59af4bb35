/*
 * reduce.hip -- grid reductions of the stagewise schedule: the CFL timestep
 * minimum (omp3/flow.c:77-105) and the conservation totals
 * (omp3/flow.c:973-995).
 *
 * Each block reduces its share across its waves (the minimum by DPP moves, the
 * compensated sums by shuffles) and through LDS, and writes one partial; a
 * one-block launch folds the partials (reduce_common.h says why that beats
 * folding in the last block to finish).
 */
#include "reduce_common.h"

namespace flowhip {
namespace {

constexpr int kRedThreads = 256;
constexpr int kRedBlocks = 1024;

/* Each block's CFL minimum over its share of the interior (k_finish_timestep
 * folds them). min is exact, so the visiting order does not change the result. NaN
 * candidates (cells with negative energy: sqrt of a negative) are left out,
 * as the reference's min(a, b) = a < b ? a : b leaves them out in effect,
 * and counted. */
template <typename M, typename T>
__global__ __launch_bounds__(kRedThreads) void k_timestep(
    M m, const T* __restrict__ Qxx, const T* __restrict__ Qyy,
    const T* __restrict__ rho, const T* __restrict__ e, FkReduce r,
    double max_dt) {
  const Interior in(m.nx, m.ny, m.pad);
  double local = max_dt;
  int bad = 0;
  for (unsigned int k = blockIdx.x * blockDim.x + threadIdx.x; k < in.n;
       k += gridDim.x * blockDim.x) {
    const int i = in.row(k), j = in.col(k);
    const int c = i * m.nx + j;
    const double ec = double(e[c]), qx = double(Qxx[c]), qy = double(Qyy[c]),
                 rc = double(rho[c]), dx = double(m.celldx[j]), dy = double(m.celldy[i]);
    if (cfl_above(ec, qx, qy, rc, dx, dy, local * local)) continue;
    const double cand = cell_timestep(ec, qx, qy, rc, dx, dy);
    if (cand == cand)
      local = lesser(local, cand);
    else
      ++bad;
  }
  publish_min<kRedThreads>(local, bad, r);
}

/* The (dt, dt_h) update from parts blocks' minima. */
__global__ __launch_bounds__(kRedThreads) void k_finish_timestep(FkReduce r, int parts,
                                                           double max_dt, int first_step) {
  const MinFold m = fold_min<false>(r, parts, max_dt);
  const double g = m.g;
  const int bad = m.bad;
  if (threadIdx.x == 0) {
    const DtPair p = next_pair(g, r.dtp[1], first_step);
    r.dtp[0] = p.dt;
    r.dtp[1] = p.dt_h;
    r.sums[2] = g;
    r.status[1] = bad;
    post(r, 0, p.dt);
    post(r, 1, p.dt_h);
    post(r, 4, (double)bad);
  }
}

/* The totals from parts blocks' compensated sums. */
__global__ __launch_bounds__(kRedThreads) void k_finish_sums(FkReduce r, int parts) {
  CSum gm{0.0, 0.0}, ge{0.0, 0.0};
  for (int b = threadIdx.x; b < parts; b += kRedThreads) {
    const double* p = r.partials + kTotalsOffset + 4 * b;
    gm.merge(CSum{p[0], p[1]});
    ge.merge(CSum{p[2], p[3]});
  }
  gm = block_csum<kRedThreads>(gm);
  ge = block_csum<kRedThreads>(ge);
  if (threadIdx.x == 0) {
    r.sums[0] = gm.s + gm.c;
    r.sums[1] = ge.s + ge.c;
    post(r, 2, r.sums[0]);
    post(r, 3, r.sums[1]);
  }
}

/* State of omp3's serial CFL fold over a run of consecutive candidates
 * (row-major order): p is the fold from +inf with min(a, b) = a < b ? a : b,
 * so NaN when the run ends on a NaN candidate and otherwise the minimum
 * over the candidates after the run's last NaN (all of them if none); nan
 * records that the run holds a NaN, any that it holds a candidate. Joining
 * two adjacent runs gives the state of their concatenation, so the grid
 * can fold contiguous ranges independently and join them in order. */
struct SerialFold {
  double p;
  int nan, any;
};

__device__ __forceinline__ SerialFold fold_join(SerialFold a, SerialFold b) {
  if (!b.any) return a;
  if (!a.any) return b;
  /* b's last NaN makes every earlier candidate irrelevant; otherwise b's
   * first candidate replaces a NaN in a's fold and the rest are minima */
  SerialFold o{b.p, a.nan | b.nan, 1};
  if (!b.nan && a.p == a.p) o.p = lesser(a.p, b.p);
  return o;
}

/* The fold of 64 consecutive candidates, one per lane (valid lanes only),
 * the same in every lane. */
__device__ __forceinline__ SerialFold wave_fold(double cand, bool valid) {
  const unsigned long long vmask = __ballot(valid);
  const unsigned long long nmask = __ballot(valid && cand != cand);
  const int lane = threadIdx.x % kWave;
  SerialFold f{__builtin_inf(), nmask != 0ull, vmask != 0ull};
  unsigned long long tail = vmask;
  if (nmask) {
    const int last = 63 - __builtin_clzll(nmask);
    tail = vmask & ~((2ull << last) - 1ull); /* lanes after the last NaN */
  }
  const double x = ((tail >> lane) & 1ull) ? cand : __builtin_inf();
  f.p = wave_min(x);
  if (nmask && !tail) f.p = __builtin_nan("");
  return f;
}

/* omp3/flow.c:77-105 read as one OpenMP thread executes it (see
 * fk_timestep_serial): block b folds a contiguous range of the interior in
 * row-major order, its waves contiguous sub-ranges, 64 cells at a time;
 * k_finish_serial joins the blocks' folds in order. */
template <bool kFromArrays>
__global__ __launch_bounds__(kRedThreads) void k_timestep_serial(
    FkMesh m, const double* __restrict__ cfl, const double* __restrict__ Qxx,
    const double* __restrict__ Qyy, const double* __restrict__ rho,
    const double* __restrict__ e, FkReduce r) {
  constexpr int kWaves = kRedThreads / kWave;
  __shared__ SerialFold s_fold[kWaves];
  __shared__ int s_bad[kWaves];
  const Interior in(m.nx, m.ny, m.pad);
  const long n = in.n;
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
  const long b0 = n * blockIdx.x / gridDim.x, b1 = n * (blockIdx.x + 1) / gridDim.x;
  const long k0 = b0 + (b1 - b0) * w / kWaves, k1 = b0 + (b1 - b0) * (w + 1) / kWaves;
  SerialFold acc{__builtin_inf(), 0, 0};
  int bad = 0;
  for (long base = k0; base < k1; base += kWave) {
    const long k = base + lane;
    const bool valid = k < k1;
    double cand = 0.0;
    if (valid) {
      const int i = in.row((unsigned int)k), j = in.col((unsigned int)k);
      const int c = i * m.nx + j;
      cand = kFromArrays ? cell_timestep(e[c], Qxx[c], Qyy[c], rho[c], m.celldx[j],
                                         m.celldy[i])
                         : cfl[c];
    }
    const SerialFold f = wave_fold(cand, valid);
    if (f.nan) bad += __popcll(__ballot(valid && cand != cand));
    acc = fold_join(acc, f);
  }
  if (lane == 0) {
    s_fold[w] = acc;
    s_bad[w] = bad;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    SerialFold blk = s_fold[0];
    int blk_bad = s_bad[0];
    for (int q = 1; q < kWaves; ++q) {
      blk = fold_join(blk, s_fold[q]);
      blk_bad += s_bad[q];
    }
    double* p = r.partials + 4 * blockIdx.x;
    p[0] = blk.p;
    p[1] = (double)(blk.nan + 2 * blk.any);
    p[2] = (double)blk_bad;
  }
}

/* Joins the folds of parts blocks (at most kRedBlocks) in order, and the
 * (dt, dt_h) update. */
__global__ __launch_bounds__(kRedThreads) void k_finish_serial(FkReduce r, int parts,
                                                               double max_dt,
                                                               int first_step) {
  __shared__ double s_p[kRedBlocks], s_flags[kRedBlocks], s_bad[kRedBlocks];
  for (int b = threadIdx.x; b < parts; b += kRedThreads) {
    s_p[b] = r.partials[4 * b];
    s_flags[b] = r.partials[4 * b + 1];
    s_bad[b] = r.partials[4 * b + 2];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    SerialFold all{__builtin_inf(), 0, 0};
    double bad = 0.0;
    for (int b = 0; b < parts; ++b) {
      const int flags = (int)s_flags[b];
      all = fold_join(all, SerialFold{s_p[b], flags & 1, flags >> 1});
      bad += s_bad[b];
    }
    /* OpenMP's min combiner merges the thread's fold into max_dt: a fold
     * that ends on a NaN leaves max_dt */
    const double g = lesser(all.p, max_dt);
    const DtPair p = next_pair(g, r.dtp[1], first_step);
    r.dtp[0] = p.dt;
    r.dtp[1] = p.dt_h;
    r.sums[2] = g;
    r.status[1] = (int)bad;
    post(r, 0, p.dt);
    post(r, 1, p.dt_h);
    post(r, 4, bad);
  }
}

template <typename M, typename T>
__global__ __launch_bounds__(kRedThreads) void k_conservation(
    M m, const T* __restrict__ rho, const T* __restrict__ e, FkReduce r) {
  const Interior in(m.nx, m.ny, m.pad);
  CSum ms{0.0, 0.0}, es{0.0, 0.0};
  for (unsigned int k = blockIdx.x * blockDim.x + threadIdx.x; k < in.n;
       k += gridDim.x * blockDim.x) {
    const int i = in.row(k), j = in.col(k);
    const int c = i * m.nx + j;
    ms.add(double(rho[c]));
    es.add(double(rho[c]) * double(e[c]));
  }
  publish_sums<kRedThreads>(ms, es, r);
}

template <typename M>
int red_blocks(const M& m) {
  const long n = Interior(m.nx, m.ny, m.pad).n;
  long b = (n + kRedThreads - 1) / kRedThreads;
  if (b > kRedBlocks) b = kRedBlocks;
  return b < 1 ? 1 : (int)b;
}

}  // namespace
}  // namespace flowhip

using namespace flowhip;

extern "C" {

int fk_reduce_blocks(void) { return kPartialsDoubles; }

hipError_t fk_finish_timestep(FkReduce r, int parts, double max_dt, int first_step,
                              hipStream_t s) {
  hipLaunchKernelGGL(k_finish_timestep, dim3(1), dim3(kRedThreads), 0, s, r, parts, max_dt,
                     first_step);
  return hipGetLastError();
}

hipError_t fk_finish_sums(FkReduce r, int parts, hipStream_t s) {
  hipLaunchKernelGGL(k_finish_sums, dim3(1), dim3(kRedThreads), 0, s, r, parts);
  return hipGetLastError();
}

hipError_t fk_timestep(FkMesh m, const double* Qxx, const double* Qyy,
                       const double* rho, const double* e, FkReduce r,
                       double max_dt, int first_step, hipStream_t s) {
  const int grid = red_blocks(m);
  hipLaunchKernelGGL((k_timestep<FkMesh, double>), dim3(grid), dim3(kRedThreads), 0, s, m,
                     Qxx, Qyy, rho, e, r, max_dt);
  return fk_finish_timestep(r, grid, max_dt, first_step, s);
}

hipError_t fk_timestep_serial(FkMesh m, const double* cfl, const double* Qxx,
                              const double* Qyy, const double* rho,
                              const double* e, FkReduce r, double max_dt,
                              int first_step, hipStream_t s) {
  const int grid = red_blocks(m);
  if (cfl)
    hipLaunchKernelGGL(k_timestep_serial<false>, dim3(grid), dim3(kRedThreads), 0, s, m,
                       cfl, Qxx, Qyy, rho, e, r);
  else
    hipLaunchKernelGGL(k_timestep_serial<true>, dim3(grid), dim3(kRedThreads), 0, s, m,
                       cfl, Qxx, Qyy, rho, e, r);
  hipLaunchKernelGGL(k_finish_serial, dim3(1), dim3(kRedThreads), 0, s, r, grid, max_dt,
                     first_step);
  return hipGetLastError();
}

hipError_t fk_conservation(FkMesh m, const double* rho, const double* e,
                           FkReduce r, hipStream_t s) {
  const int grid = red_blocks(m);
  hipLaunchKernelGGL((k_conservation<FkMesh, double>), dim3(grid), dim3(kRedThreads), 0, s,
                     m, rho, e, r);
  return fk_finish_sums(r, grid, s);
}

hipError_t fk_timestep_f32(FkMesh32 m, const float* Qxx, const float* Qyy,
                           const float* rho, const float* e, FkReduce r,
                           double max_dt, int first_step, hipStream_t s) {
  const int grid = red_blocks(m);
  hipLaunchKernelGGL((k_timestep<FkMesh32, float>), dim3(grid), dim3(kRedThreads), 0, s, m,
                     Qxx, Qyy, rho, e, r, max_dt);
  return fk_finish_timestep(r, grid, max_dt, first_step, s);
}

hipError_t fk_conservation_f32(FkMesh32 m, const float* rho, const float* e,
                               FkReduce r, hipStream_t s) {
  const int grid = red_blocks(m);
  hipLaunchKernelGGL((k_conservation<FkMesh32, float>), dim3(grid), dim3(kRedThreads), 0, s,
                     m, rho, e, r);
  return fk_finish_sums(r, grid, s);
}

}  // extern "C"
