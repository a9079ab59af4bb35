/*
 * ensemble.hip -- the batching form: many independent meshes of uneven
 * sizes advanced together, one launch per stage for the whole ensemble.
 *
 * Every instance's interior is cut into the same row-march items (strips
 * of kEnsW columns, chunks of H rows), and one work list holds the items
 * of all instances, in the order the host (or its autotuner) chose. The
 * persistent kernels below walk that list: each wave takes an item, reads
 * its instance's descriptor (geometry, arrays, dt pair) with scalar loads,
 * and runs the same per-item body as the single-mesh march kernels, so a
 * batched instance computes bit for bit what it computes alone.
 *
 * A step is the three march kernels and nothing between them. An instance's CFL
 * minimum (omp3/flow.c:77-105) is one word that the Lagrangian march's items
 * lower; the mass/energy march's items each take the new dt pair from it. The
 * compensated mass and energy totals (omp3/flow.c:973-995) go through per-item
 * partials, indexed by the item's position inside its instance, which blocks at
 * the front of the momentum march combine in item order. Per-step dt pairs and
 * totals are appended to device history buffers at a device-side step counter,
 * so a step can be captured once in a hipGraph and replayed.
 */
#include <cmath>

#include "march.h"

namespace flowhip {

/* Strip width of every ensemble kernel: the narrowest any march kernel
 * allows (the Lagrangian kernel's), so one work list serves all stages.
 * Momentum runs as one fused march or as the x then y marches, a schedule
 * choice of the host (and its autotuner). */
constexpr int kEnsW = kWave - 6;

template <typename T>
__device__ __forceinline__ MGeo<T> ens_geo(const FkEnsInst& in) {
  MGeo<T> g;
  g.nx = in.nx;
  g.ny = in.ny;
  g.edx = (const T*)in.geo[0];
  g.edy = (const T*)in.geo[1];
  g.cdx = (const T*)in.geo[2];
  g.cdy = (const T*)in.geo[3];
  g.iedx = (const T*)in.geo[4];
  g.iedy = (const T*)in.geo[5];
  g.u = uniform_of<T>(in.u);
  return g;
}

template <typename T>
__device__ __forceinline__ T* arr(const FkEnsInst& in, int k) {
  return (T*)in.a[k];
}

/* solve_hydro_2d's array order */
enum { kP, kRho, kRhoOld, kE, kU, kV, kMomX, kMomY, kQxx, kQyy, kFx, kFy,
       kUFx, kUFy, kVFx, kVFy };

__device__ __forceinline__ MarchList ens_list(const FkEnsInst& in, int H) {
  MarchList ml;
  ml.W = kEnsW;
  ml.H = H;
  ml.nstrips = in.nstrips;
  ml.nchunks = in.nchunks;
  ml.nitems = in.nitems;
  ml.inv = in.strip_inv;
  return ml;
}

/* ---- CFL minima, one word per instance ----
 * A double as an unsigned key of the same order (any sign), so that the minimum
 * is an integer atomic whose result does not depend on the order of the items;
 * all ones: no candidate yet. An item whose candidates all lie at or above its
 * seed (cfl_seed: they cannot count) leaves the word alone, which on most steps
 * is nearly every item. */
constexpr unsigned long long kNoCandidate = ~0ull;

__device__ __forceinline__ unsigned long long min_key(double x) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(x);
  return b ^ ((unsigned long long)((long long)b >> 63) | 0x8000000000000000ull);
}
__device__ __forceinline__ double min_value(unsigned long long key) {
  const unsigned long long b = (key >> 63) ? key ^ 0x8000000000000000ull : ~key;
  return __longlong_as_double((long long)b);
}

/* An item's minimum and its undefined candidates, per lane. */
__device__ __forceinline__ void publish_item(const FkEnsPartials& part, int inst, int lane,
                                             double local_min, double seed, int nan_count) {
  local_min = wave_min(local_min);
  if (lane == 0 && local_min < seed) atomicMin(part.min + inst, min_key(local_min));
  if (__ballot(nan_count != 0)) {
    nan_count = wave_sum(nan_count);
    if (lane == 0) atomicAdd(part.nan + inst, nan_count);
  }
}

/* The instance's new pair (omp3/flow.c:103-105). */
template <bool kSquared>
__device__ __forceinline__ DtPair ens_pair(const FkEnsInst& in, unsigned long long key,
                                           int first_step) {
  double g = kSquared ? in.max_dt * in.max_dt : in.max_dt;
  if (key != kNoCandidate) g = lesser(g, min_value(key));
  if (kSquared) g = __builtin_sqrt(g);
  return next_pair(g, in.dtp[1], first_step);
}

/* ---- the stages ---- */

template <typename T, bool P2, bool UNI>
__global__ __launch_bounds__(kMNT, FLOWHIP_MARCH_WAVES) void k_ens_lagrangian(
    const FkEnsInst* __restrict__ insts, const int2* __restrict__ work, int nwork,
    unsigned int* __restrict__ queue,
    int H, FkEnsPartials part, int* __restrict__ counter) {
  const int lane = threadIdx.x % kWave;
  if (blockIdx.x == 0) {
    march_queue_reset(queue, kStageLag);
    if (threadIdx.x == 0) *counter += 1; /* this step's history row */
  }
  MarchQueue<true> mq(queue, kStageLag, nwork, blockIdx.x, gridDim.x);
  for (int w = mq.first(); w < mq.end; w = mq.next()) {
    const int2 wi = work[w];
    const FkEnsInst& in = insts[wi.x];
    const MLagIO<T> io{arr<T>(in, kRho),   arr<T>(in, kE),   arr<T>(in, kMomX),
                       arr<T>(in, kMomY),  arr<T>(in, kQxx), arr<T>(in, kQyy),
                       arr<T>(in, kUFx),   arr<T>(in, kUFy), arr<T>(in, kP),
                       arr<T>(in, kRhoOld)};
    const T dt = T(in.dtp[0]), dt_h = T(in.dtp[1]);
    const double seed = cfl_seed<T>(in.max_dt, in.dtp[1]);
    double local_min = seed;
    int nan_count = 0;
    const MGeo<T> g = ens_geo<T>(in);
    const MarchList ml = ens_list(in, H);
    /* interior items take the straight-line form, as on a single mesh */
    const ItemBox b = item_box(ml, g.nx, g.ny, wi.y);
    if (!box_edge(b, g.nx, g.ny))
      lagrangian_box<T, P2, 0, false, UNI>(g, io, dt, dt_h, b, lane, local_min, nan_count);
    else
      lagrangian_box<T, P2, -1, true, UNI>(g, io, dt, dt_h, b, lane, local_min, nan_count);
    publish_item(part, wi.x, lane, local_min, seed, nan_count);
  }
}

template <typename T, bool P2, bool UNI>
__global__ __launch_bounds__(kMNT, FLOWHIP_MARCH_WAVES) void k_ens_mass(
    const FkEnsInst* __restrict__ insts, const int2* __restrict__ work, int nwork,
    unsigned int* __restrict__ queue,
    int H, int tt, int ninst, FkEnsPartials part, FkEnsHistory hist) {
  const int lane = threadIdx.x % kWave;
  if (blockIdx.x == 0) march_queue_reset(queue, kStageMass);
  MarchQueue<true> mq(queue, kStageMass, nwork, blockIdx.x, gridDim.x);
  for (int w = mq.first(); w < mq.end; w = mq.next()) {
    const int2 wi = work[w];
    const FkEnsInst& in = insts[wi.x];
    const MMassIO<T> io{arr<T>(in, kUFx), arr<T>(in, kUFy), arr<T>(in, kRhoOld),
                        arr<T>(in, kP),   arr<T>(in, kRho), arr<T>(in, kE),
                        arr<T>(in, kFx),  arr<T>(in, kFy)};
    const DtPair pair =
        ens_pair<std::is_same<T, float>::value>(in, part.min[wi.x], tt == 0 ? 1 : 0);
    const T dt = T(pair.dt), dt_h = T(pair.dt_h);
    if (wi.y == 0 && lane == 0) {
      const long h = (long)*hist.counter * ninst + wi.x;
      in.dtp_new[0] = hist.dt[2 * h] = pair.dt;
      in.dtp_new[1] = hist.dt[2 * h + 1] = pair.dt_h;
      hist.nan[h] = part.nan[wi.x];
    }
    CSum ms{0.0, 0.0}, es{0.0, 0.0};
    const MGeo<T> g = ens_geo<T>(in);
    const MarchList ml = ens_list(in, H);
    const ItemBox b = item_box(ml, g.nx, g.ny, wi.y);
    const bool edge = box_edge(b, g.nx, g.ny);
    if (tt % 2 == 0) {
      if (edge)
        mass_xy_box<T, P2, true, UNI>(g, io, dt, dt_h, b, lane, ms, es);
      else
        mass_xy_box<T, P2, false, UNI>(g, io, dt, dt_h, b, lane, ms, es);
    } else {
      if (edge)
        mass_yx_box<T, P2, true, UNI>(g, io, dt, dt_h, b, lane, ms, es);
      else
        mass_yx_box<T, P2, false, UNI>(g, io, dt, dt_h, b, lane, ms, es);
    }
    ms = wave_csum(ms);
    es = wave_csum(es);
    if (lane == 0) {
      double* p = part.sums + 4 * (in.item0 + wi.y);
      p[0] = ms.s;
      p[1] = ms.c;
      p[2] = es.s;
      p[3] = es.c;
    }
  }
}

/* ---- the step's epilogue ----
 * The first ens_epilogue_blocks blocks of the momentum march march nothing: a
 * wave per instance folds the totals' partials in item order, moves the new dt
 * pair to where the next step's Lagrangian march reads it, and clears the CFL
 * words. As kernels of their own (dt pair, totals, counter) these took 15 us of
 * a 150 us step of 24 instances of 64^2 to 464^2 on MI355X and 31 of 750 us for
 * 96 FP32 instances up to 1013^2. */
__host__ __device__ inline int ens_epilogue_blocks(int ninst) { return (ninst + kMWaves - 1) / kMWaves; }

__device__ __forceinline__ void ens_epilogue(const FkEnsInst* __restrict__ insts, int ninst,
                                             const FkEnsPartials& part,
                                             const FkEnsHistory& hist) {
  const int lane = threadIdx.x % kWave;
  const int inst =
      __builtin_amdgcn_readfirstlane(blockIdx.x * kMWaves + threadIdx.x / kWave);
  if (inst >= ninst) return;
  const FkEnsInst& in = insts[inst];
  CSum gm{0.0, 0.0}, ge{0.0, 0.0};
#pragma unroll 4
  for (int k = lane; k < in.nitems; k += kWave) {
    const double* p = part.sums + 4 * (in.item0 + k);
    gm.merge(CSum{p[0], p[1]});
    ge.merge(CSum{p[2], p[3]});
  }
  gm = wave_csum(gm);
  ge = wave_csum(ge);
  if (lane == 0) {
    const long h = (long)*hist.counter * ninst + inst;
    hist.sums[2 * h] = gm.s + gm.c;
    hist.sums[2 * h + 1] = ge.s + ge.c;
    in.dtp[0] = in.dtp_new[0];
    in.dtp[1] = in.dtp_new[1];
    part.min[inst] = kNoCandidate;
    part.nan[inst] = 0;
  }
}

/* ydir 0: x momentum (u0 = uF_x), 1: y momentum (io.u = the u just written) */
template <typename T, bool P2>
__global__ __launch_bounds__(kMNT, FLOWHIP_MARCH_WAVES) void k_ens_momentum(
    const FkEnsInst* __restrict__ insts, const int2* __restrict__ work, int nwork,
    unsigned int* __restrict__ queue,
    int H, int tt, int ydir, int ninst, FkEnsPartials part, FkEnsHistory hist) {
  const int lane = threadIdx.x % kWave;
  const int front = ydir ? 0 : ens_epilogue_blocks(ninst);
  /* the y direction counts in the mass/energy march's set, which the x
   * direction has zeroed */
  const int stage = ydir ? kStageMass : kStageMom;
  if (blockIdx.x == 0) march_queue_reset(queue, stage);
  if ((int)blockIdx.x < front) {
    ens_epilogue(insts, ninst, part, hist);
    return;
  }
  MarchQueue<true> mq(queue, stage, nwork, blockIdx.x - front, gridDim.x - front);
  for (int w = mq.first(); w < mq.end; w = mq.next()) {
    const int2 wi = work[w];
    const FkEnsInst& in = insts[wi.x];
    const T dt = T(in.dtp_new[0]), dt_h = T(in.dtp_new[1]);
    const MGeo<T> g = ens_geo<T>(in);
    const MarchList ml = ens_list(in, H);
    if (!ydir) {
      const MMomIO<T> io{arr<T>(in, kUFx), arr<T>(in, kUFy), arr<T>(in, kFx),
                         arr<T>(in, kFy),  arr<T>(in, kRho), arr<T>(in, kQxx),
                         arr<T>(in, kMomX), arr<T>(in, kU)};
      if (tt % 2)
        momx_xy_item<T, P2>(g, io, dt, dt_h, ml, wi.y, lane);
      else
        momx_yx_item<T, P2>(g, io, dt, dt_h, ml, wi.y, lane);
    } else {
      const MMomIO<T> io{arr<T>(in, kU),   arr<T>(in, kUFy), arr<T>(in, kFx),
                         arr<T>(in, kFy),  arr<T>(in, kRho), arr<T>(in, kQyy),
                         arr<T>(in, kMomY), arr<T>(in, kV)};
      if (tt % 2)
        momy_xy_item<T, P2>(g, io, dt, dt_h, ml, wi.y, lane);
      else
        momy_yx_item<T, P2>(g, io, dt, dt_h, ml, wi.y, lane);
    }
  }
}

/* Both momentum directions in one march (momxy_*_item). */
template <typename T, bool P2, bool UNI>
__global__ __launch_bounds__(kMNT, FLOWHIP_MARCH_WAVES) void k_ens_momentum_xy(
    const FkEnsInst* __restrict__ insts, const int2* __restrict__ work, int nwork,
    unsigned int* __restrict__ queue,
    int H, int tt, int ninst, FkEnsPartials part, FkEnsHistory hist) {
  const int lane = threadIdx.x % kWave;
  const int front = ens_epilogue_blocks(ninst);
  if (blockIdx.x == 0) march_queue_reset(queue, kStageMom);
  if ((int)blockIdx.x < front) {
    ens_epilogue(insts, ninst, part, hist);
    return;
  }
  /* claimed per block, as the single-mesh fused momentum march */
  const int wave = threadIdx.x / kWave;
  MarchBlockQueue mq(queue, kStageMom, nwork, blockIdx.x - front, gridDim.x - front);
  for (int base = mq.first(); base < mq.end; base = mq.next()) {
    const int w = __builtin_amdgcn_readfirstlane(base + wave);
    if (w >= mq.end) continue;
    const int2 wi = work[w];
    const FkEnsInst& in = insts[wi.x];
    const T dt = T(in.dtp_new[0]), dt_h = T(in.dtp_new[1]);
    const MMom2IO<T> io{arr<T>(in, kUFx), arr<T>(in, kUFy), arr<T>(in, kFx),
                        arr<T>(in, kFy),  arr<T>(in, kRho), arr<T>(in, kQxx),
                        arr<T>(in, kQyy), arr<T>(in, kMomX), arr<T>(in, kMomY),
                        arr<T>(in, kU),   arr<T>(in, kV)};
    const MGeo<T> g = ens_geo<T>(in);
    const MarchList ml = ens_list(in, H);
    const ItemBox b = item_box(ml, g.nx, g.ny, wi.y);
    const bool edge = box_edge(b, g.nx, g.ny);
    if (tt % 2) {
      if (edge)
        momxy_xy_box<T, P2, -1, true, UNI>(g, io, dt, dt_h, b, lane);
      else
        momxy_xy_box<T, P2, 0, false, UNI>(g, io, dt, dt_h, b, lane);
    } else {
      if (edge)
        momxy_yx_box<T, P2, -1, true, UNI>(g, io, dt, dt_h, b, lane);
      else
        momxy_yx_box<T, P2, 0, false, UNI>(g, io, dt, dt_h, b, lane);
    }
  }
}

/* CFL candidates of one item's cells (the pre-loop set_timestep). */
template <typename T>
__global__ __launch_bounds__(kMNT) void k_ens_timestep(
    const FkEnsInst* __restrict__ insts, const int2* __restrict__ work, int nwork,
    unsigned int* __restrict__ queue,
    int H, FkEnsPartials part) {
  const int lane = threadIdx.x % kWave;
  MarchQueue<true> mq(queue, kStageLag, nwork, blockIdx.x, gridDim.x);
  for (int w = mq.first(); w < mq.end; w = mq.next()) {
    const int2 wi = work[w];
    const FkEnsInst& in = insts[wi.x];
    const MGeo<T> g = ens_geo<T>(in);
    const int nx = in.nx, ny = in.ny;
    const ItemBox b = item_box(ens_list(in, H), nx, ny, wi.y);
    const int x1 = b.x1, y0 = b.y0, y1 = b.y1;
    const int j = b.x0 + lane;
    const T *e = arr<T>(in, kE), *qxx = arr<T>(in, kQxx), *qyy = arr<T>(in, kQyy),
            *rho = arr<T>(in, kRho);
    double local_min = in.max_dt;
    int nan_count = 0;
    if (j < x1) {
      for (int i = y0; i < y1; ++i) {
        const int c = i * nx + j;
        const double ec = double(e[c]), qx = double(qxx[c]), qy = double(qyy[c]),
                     rc = double(rho[c]), dx = double(g.cdx[j]), dy = double(g.cdy[i]);
        if (cfl_above(ec, qx, qy, rc, dx, dy, local_min * local_min)) continue;
        const double cand = cell_timestep(ec, qx, qy, rc, dx, dy);
        if (cand == cand)
          local_min = lesser(local_min, cand);
        else
          ++nan_count;
      }
    }
    publish_item(part, wi.x, lane, local_min, in.max_dt, nan_count);
  }
}

/* The pre-loop pair of every instance; clears the CFL words and the work-queue
 * counters. */
__global__ __launch_bounds__(kMNT) void k_ens_dt(const FkEnsInst* __restrict__ insts, int ninst,
                                                 FkEnsPartials part,
                                                 unsigned int* __restrict__ queue) {
  if (blockIdx.x == 0) march_queue_reset(queue, -1);
  const int inst = blockIdx.x * kMNT + threadIdx.x;
  if (inst >= ninst) return;
  const FkEnsInst& in = insts[inst];
  const DtPair p = ens_pair<false>(in, part.min[inst], 0);
  in.dtp[0] = p.dt;
  in.dtp[1] = p.dt_h;
  part.min[inst] = kNoCandidate;
  part.nan[inst] = 0;
}

__global__ void k_ens_set_counter(int* counter, int v) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *counter = v;
}

/* ---- launch helpers ---- */

template <typename T, bool P2, bool UNI>
hipError_t ens_step_p(const FkEnsLaunch& L, int tt, hipStream_t s) {
  static int pc_lag = 0, pc_mass = 0, pc_mom = 0;
  const int nw = L.nwork;
  if (nw < 1 || L.ninst < 1 || !L.queue) return hipErrorInvalidValue;
  const int2* work = (const int2*)L.work;
  hipLaunchKernelGGL((k_ens_lagrangian<T, P2, UNI>),
                     dim3(march_grid(k_ens_lagrangian<T, P2, UNI>, pc_lag, nw, kMarchMaxWaves<T>)),
                     dim3(kMNT), 0, s, L.insts, work, nw, L.queue, L.chunk_rows, L.part,
                     L.hist.counter);
  hipLaunchKernelGGL((k_ens_mass<T, P2, UNI>),
                     dim3(march_grid(k_ens_mass<T, P2, UNI>, pc_mass, nw, kMarchMaxWaves<T>)),
                     dim3(kMNT), 0, s, L.insts, work, nw, L.queue, L.chunk_rows, tt, L.ninst,
                     L.part, L.hist);
  const int front = ens_epilogue_blocks(L.ninst);
  if (L.fused_momentum) {
    static int pc_momxy = 0;
    hipLaunchKernelGGL((k_ens_momentum_xy<T, P2, UNI>),
                       dim3(front + march_grid(k_ens_momentum_xy<T, P2, UNI>, pc_momxy, nw,
                                               kMarchMaxWaves<T>)),
                       dim3(kMNT), 0, s, L.insts, work, nw, L.queue, L.chunk_rows, tt, L.ninst,
                       L.part, L.hist);
  } else {
    const int gm = march_grid(k_ens_momentum<T, P2>, pc_mom, nw);
    hipLaunchKernelGGL((k_ens_momentum<T, P2>), dim3(front + gm), dim3(kMNT), 0, s, L.insts,
                       work, nw, L.queue, L.chunk_rows, tt, 0, L.ninst, L.part, L.hist);
    hipLaunchKernelGGL((k_ens_momentum<T, P2>), dim3(gm), dim3(kMNT), 0, s, L.insts, work, nw,
                       L.queue, L.chunk_rows, tt, 1, L.ninst, L.part, L.hist);
  }
  return hipGetLastError();
}

template <typename T>
hipError_t ens_step(const FkEnsLaunch& L, int tt, hipStream_t s) {
  /* every instance's spacings are uniform (width / n): the mass/energy and
   * momentum marches read their row geometry once per item unless
   * FLOWHIP_UNIFORM=0 (the same bits either way) */
  if (L.uniform)
    return L.pow2 ? ens_step_p<T, true, true>(L, tt, s) : ens_step_p<T, false, true>(L, tt, s);
  return L.pow2 ? ens_step_p<T, true, false>(L, tt, s) : ens_step_p<T, false, false>(L, tt, s);
}

template <typename T>
hipError_t ens_timestep(const FkEnsLaunch& L, hipStream_t s) {
  static int pc = 0;
  const int nw = L.nwork;
  if (nw < 1 || L.ninst < 1 || !L.queue) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_ens_timestep<T>, dim3(march_grid(k_ens_timestep<T>, pc, nw)),
                     dim3(kMNT), 0, s, L.insts, (const int2*)L.work, nw, L.queue,
                     L.chunk_rows, L.part);
  hipLaunchKernelGGL(k_ens_dt, dim3((L.ninst + kMNT - 1) / kMNT), dim3(kMNT), 0, s, L.insts,
                     L.ninst, L.part, L.queue);
  return hipGetLastError();
}

}  // namespace flowhip

using namespace flowhip;

extern "C" {

int fk_ens_strip_width(void) { return kEnsW; }

unsigned long long fk_strip_inverse(int nstrips) { return strip_inverse(nstrips); }

/* The single-mesh rule for chunk heights (march.hip) on the cells of the whole
 * ensemble, with one height for all stages (prologue 4.5 rows, at most the 20
 * rows the autotuner picks for the 256-instance ensemble). */
int fk_ens_default_rows(double cells, int fp32) {
  const double slots =
      (double)march_cus() * kMWaves * (fp32 ? kMarchMaxWaves<float> : kMarchMaxWaves<double>);
  const int H = (int)(std::sqrt(4.5 * cells / (kEnsW * slots)) + 0.5);
  return H < 4 ? 4 : H > 20 ? 20 : H;
}

hipError_t fk_ens_step(FkEnsLaunch L, int tt, int fp32, hipStream_t s) {
  if (L.chunk_rows < 4 || L.chunk_rows > kMaxChunkRows) return hipErrorInvalidValue;
  return fp32 ? ens_step<float>(L, tt, s) : ens_step<double>(L, tt, s);
}

hipError_t fk_ens_timestep(FkEnsLaunch L, int fp32, hipStream_t s) {
  if (L.chunk_rows < 4 || L.chunk_rows > kMaxChunkRows) return hipErrorInvalidValue;
  return fp32 ? ens_timestep<float>(L, s) : ens_timestep<double>(L, s);
}

hipError_t fk_ens_set_counter(int* counter, int value, hipStream_t s) {
  hipLaunchKernelGGL(k_ens_set_counter, dim3(1), dim3(1), 0, s, counter, value);
  return hipGetLastError();
}

}  // extern "C"
