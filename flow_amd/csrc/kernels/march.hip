/*
 * march.hip -- launchers of the row-marching kernels on one mesh (FP64 and
 * the FP32-state form). The kernels are in march.h, their row-parallel form for
 * small meshes in rows.h.
 */
#include <cmath>

#include "march.h"
#include "rows.h"

namespace flowhip {

/* Chunk height of a march kernel when none is given. An item costs its H rows
 * and about p more (prologue rows, first loads); C cells in strips of W
 * columns on S waves then take (C / (W H S)) (H + p) row times, and the last
 * items to finish leave the GPU partly idle for about H + p more, which is
 * least at H = sqrt(p C / (W S)). So the height follows the square root of
 * the mesh's cells, up to the height measured fastest at 8192^2, beyond which
 * the rows in flight leave the last-level cache. p is fitted per kernel to
 * sweeps of 2 to 24 rows at 64^2, 300x200, 512^2, 1000^2, 3000x150, 1536^2,
 * 2048^2, 3001x2999 and 4096^2. Measured on MI355X (us a step, FP64; FP32),
 * fixed heights of 24 / 20 / 16 rows (24 / 16 / 16) before and this rule
 * after: 64^2 168 -> 64; 138 -> 52, 512^2 180 -> 83; 144 -> 60, 1000^2 197
 * -> 130; 156 -> 90, 3000x150 195 -> 96; 156 -> 72, 2048^2 323 -> 323; 191 ->
 * 166, 3001x2999 and up within 2%.
 *
 * Where a mass/energy or momentum chunk up to 1.6 times as tall lets the items
 * fit the waves in one round, it is taken: items a little over one round leave
 * the last ones to march alone. Measured (us a kernel, the height above and this
 * one): FP64 momentum 1150^2 35.7 -> 33.0, 1250^2 39.8 -> 36.3, 1400^2 45.3 -> 41.4,
 * mass/energy 1100^2 39.0 -> 36.0, 1400^2 50.7 -> 49.3; FP32 momentum 1250^2 24.0
 * -> 22.1, 1400^2 27.3 -> 24.7, 2500x600 23.6 -> 22.0. Past 1.6 times the longer
 * items cost what the round saves (FP64 momentum 1536^2 with 14 rows for 9: the
 * same). The Lagrangian, whose prologue is short, gained at 900^2 (5 rows for 4:
 * 32 -> 30) and lost at 850^2 (5 for 3: 27.8 -> 29.5); it keeps the root.
 */
struct Rows {
  double p;      /* prologue, in rows */
  int most;      /* height on large meshes */
  double taller; /* how much taller a chunk may be to fit one round */
};
enum { kKLag = 0, kKMass = 1, kKMom = 2 };
template <typename T>
constexpr Rows rows_of(int kernel) {
  return sizeof(T) == 8 ? (kernel == kKLag    ? Rows{2.9, 24, 1.0}
                           : kernel == kKMass ? Rows{5.7, 20, 1.6}
                                              : Rows{6.2, 16, 1.6})
                        : (kernel == kKLag    ? Rows{2.1, 24, 1.0}
                           : kernel == kKMass ? Rows{8.5, 16, 1.6}
                                              : Rows{5.2, 16, 1.6});
}

/* the marches with two columns per lane (12 rows in FP64, measured 8 to 24; 10
 * in FP32, measured 4 to 24) run on large meshes, or where a caller asks */
template <typename T>
constexpr Rows pair_rows() {
  return sizeof(T) == 8 ? Rows{2.9, 12, 1.0} : Rows{2.1, 10, 1.0};
}

inline MarchList march_items(int nx, int ny, int W, int chunk_rows, Rows r, int waves_per_simd,
                             int least = kMinChunkRows) {
  if (chunk_rows > 0)
    return make_march(nx, ny, W, chunk_rows < kMaxChunkRows ? chunk_rows : kMaxChunkRows);
  if (make_march(nx, ny, W, least).nitems < 1) return make_march(nx, ny, W, least);
  const double cells = (double)(nx - 2 * kPad) * (ny - 2 * kPad);
  const int slots = march_cus() * kMWaves * waves_per_simd;
  const double h = std::sqrt(r.p * cells / ((double)W * slots));
  int H = (int)(h + 0.5);
  H = H < least ? least : H > r.most ? r.most : H;
  const int strips = make_march(nx, ny, W, H).nstrips;
  if (strips >= 1 && strips <= slots) {
    const int chunks = slots / strips, one_round = (ny - 2 * kPad + chunks - 1) / chunks;
    if (one_round > H && one_round <= r.taller * h && one_round <= r.most) H = one_round;
  }
  return make_march(nx, ny, W, H);
}

template <typename T, bool P2, bool UNI, bool PAIR = false>
hipError_t launch_march_mass_p(MGeo<T> g, MMassIO<T> io, int tt, FkReduce r, MarchStep st,
                               int* parts, int chunk_rows, hipStream_t s) {
  constexpr int kWaves = PAIR ? kMassPairWaves<T> : kMarchMaxWaves<T>;
  const MarchList ml = march_items(g.nx, g.ny, PAIR ? kMassW2 : kMassW, chunk_rows,
                                   PAIR ? pair_rows<T>() : rows_of<T>(kKMass), kWaves);
  if (ml.nitems < 1 || !r.queue) return hipErrorInvalidValue;
  if (tt % 2 == 0) {
    static int per_cu = 0;
    const int grid = march_grid(k_march_mass_xy<T, P2, UNI, PAIR>, per_cu, ml.nitems,
                                kWaves);
    hipLaunchKernelGGL((k_march_mass_xy<T, P2, UNI, PAIR>), dim3(grid), dim3(kMNT), 0, s,
                       g, io, r, st, ml);
    *parts = grid;
  } else {
    static int per_cu = 0;
    const int grid = march_grid(k_march_mass_yx<T, P2, UNI, PAIR>, per_cu, ml.nitems,
                                kWaves);
    hipLaunchKernelGGL((k_march_mass_yx<T, P2, UNI, PAIR>), dim3(grid), dim3(kMNT), 0, s,
                       g, io, r, st, ml);
    *parts = grid;
  }
  return hipGetLastError();
}

/* Whether the two-column form runs: FkMesh.pairs 2 always, 1 on meshes of
 * at least FK_PAIR_MIN_CELLS interior cells. */
inline bool pairs_wanted(int pairs, int nx, int ny) {
  return pairs == 2 ||
         (pairs == 1 && (long)(nx - 2 * kPad) * (ny - 2 * kPad) >= FK_PAIR_MIN_CELLS);
}

/* Whether a mass/energy march can hold two columns per lane: rows of the cell
 * and y-face arrays it reads or writes as column pairs start on boundaries of
 * two values (nx even, arrays so aligned; strips start at even columns). */
template <typename T>
inline bool pairs_fit(const MGeo<T>& g, const MMassIO<T>& io) {
  const unsigned long long bits =
      (unsigned long long)io.v0 | (unsigned long long)io.rho0 | (unsigned long long)io.e1 |
      (unsigned long long)io.rho | (unsigned long long)io.e | (unsigned long long)io.F_y;
  return g.nx % 2 == 0 && (bits & (2 * sizeof(T) - 1)) == 0;
}

template <typename T, bool P2, bool UNI, bool PAIR = false>
hipError_t launch_march_lagrangian_p(MGeo<T> g, MLagIO<T> io, FkReduce r, double max_dt,
                                     int* parts, int chunk_rows, hipStream_t s) {
  constexpr int kWaves = PAIR ? kLagPairWaves<T> : kLagMaxWaves<T>;
  const MarchList ml = march_items(g.nx, g.ny, PAIR ? kLagW2 : kLagW, chunk_rows,
                                   PAIR ? pair_rows<T>() : rows_of<T>(kKLag), kWaves);
  if (ml.nitems < 1 || !r.queue) return hipErrorInvalidValue;
  static int per_cu = 0;
  const int grid = march_grid(k_march_lagrangian<T, P2, UNI, PAIR>, per_cu, ml.nitems,
                              kWaves);
  hipLaunchKernelGGL((k_march_lagrangian<T, P2, UNI, PAIR>), dim3(grid), dim3(kMNT), 0, s,
                     g, io, r, max_dt, ml);
  *parts = grid;
  return hipGetLastError();
}

/* Whether a Lagrangian march can hold two columns per lane (as pairs_fit,
 * for the arrays it reads or writes in column pairs: aligned to two
 * values). */
template <typename T>
inline bool lag_pairs_fit(const MGeo<T>& g, const MLagIO<T>& io) {
  const unsigned long long bits =
      (unsigned long long)io.rho | (unsigned long long)io.e | (unsigned long long)io.mom_y |
      (unsigned long long)io.my1 | (unsigned long long)io.v0 | (unsigned long long)io.e1 |
      (unsigned long long)io.rho_old;
  return g.nx % 2 == 0 && (bits & (2 * sizeof(T) - 1)) == 0;
}

/* Even-tt x momentum needs faces [x0-2, x1+1] and one lane below them. */
constexpr int kMomXW = kWave - 5;
constexpr int kMomW = kWave - 4;

/* The end of a step whose momentum directions march apart. */
static __global__ __launch_bounds__(kMNT) void k_march_settle(FkReduce red, int parts) {
  step_epilogue(red, parts);
}

template <typename T, bool P2>
hipError_t launch_march_momentum_p(MGeo<T> g, MMomIO<T> io, int tt, int ydir, FkReduce r,
                                   int parts, int chunk_rows, hipStream_t s) {
  const bool odd = (tt % 2) != 0;
  const MarchList ml =
      march_items(g.nx, g.ny, (!ydir && !odd) ? kMomXW : kMomW, chunk_rows,
                  rows_of<T>(kKMom), kMarchMaxWaves<T>, 4);
  if (ml.nitems < 1 || !r.queue) return hipErrorInvalidValue;
  const double* dtp = r.dtp + 2; /* the pair the mass/energy march left */
  if (!ydir && odd) {
    static int per_cu = 0;
    const int grid = march_grid(k_march_momx_xy<T, P2>, per_cu, ml.nitems);
    hipLaunchKernelGGL((k_march_momx_xy<T, P2>), dim3(grid), dim3(kMNT), 0, s, g, io, dtp, ml);
  } else if (!ydir) {
    static int per_cu = 0;
    const int grid = march_grid(k_march_momx_yx<T, P2>, per_cu, ml.nitems);
    hipLaunchKernelGGL((k_march_momx_yx<T, P2>), dim3(grid), dim3(kMNT), 0, s, g, io, dtp, ml);
  } else if (odd) {
    static int per_cu = 0;
    const int grid = march_grid(k_march_momy_xy<T, P2>, per_cu, ml.nitems);
    hipLaunchKernelGGL((k_march_momy_xy<T, P2>), dim3(grid), dim3(kMNT), 0, s, g, io, dtp, ml);
  } else {
    static int per_cu = 0;
    const int grid = march_grid(k_march_momy_yx<T, P2>, per_cu, ml.nitems);
    hipLaunchKernelGGL((k_march_momy_yx<T, P2>), dim3(grid), dim3(kMNT), 0, s, g, io, dtp, ml);
  }
  if (ydir) hipLaunchKernelGGL(k_march_settle, dim3(1), dim3(kMNT), 0, s, r, parts);
  return hipGetLastError();
}


/* both momentum directions in one march: strips of 59 columns */
constexpr int kMomXYW = kWave - 5;

template <typename T, bool P2, bool UNI>
hipError_t launch_march_momxy_p(MGeo<T> g, MMom2IO<T> io, int tt, FkReduce r, int parts,
                                int chunk_rows, hipStream_t s) {
  const MarchList ml = march_items(g.nx, g.ny, kMomXYW, chunk_rows, rows_of<T>(kKMom),
                                   kMarchMaxWaves<T>);
  if (ml.nitems < 1 || !r.queue) return hipErrorInvalidValue;
  /* one block more, for the step's epilogue */
  if (tt % 2) {
    static int per_cu = 0;
    const int grid =
        march_grid(k_march_momxy_xy<T, P2, UNI>, per_cu, ml.nitems, kMarchMaxWaves<T>);
    hipLaunchKernelGGL((k_march_momxy_xy<T, P2, UNI>), dim3(grid + 1), dim3(kMNT), 0, s, g,
                       io, r, parts, ml);
  } else {
    static int per_cu = 0;
    const int grid =
        march_grid(k_march_momxy_yx<T, P2, UNI>, per_cu, ml.nitems, kMarchMaxWaves<T>);
    hipLaunchKernelGGL((k_march_momxy_yx<T, P2, UNI>), dim3(grid + 1), dim3(kMNT), 0, s, g,
                       io, r, parts, ml);
  }
  return hipGetLastError();
}

/* Blocks of a row-parallel kernel (rows.h): waves per block, 0 where the march
 * is the faster form, and the items.
 *
 * The time of such a launch goes with the waves on the fullest CU: blocks of n
 * waves own n - halo rows, so tall blocks compute fewer halo rows twice and low
 * ones divide more evenly. n is the one of 8 to 16 that leaves that CU the
 * fewest waves (6 and 7 were no faster at 64^2). Measured on MI355X (us a
 * step, FP64; FP32), blocks of 16 and then this rule: 64^2 21.9 -> 17.9; 18.3
 * -> 15.9, 300x200 26.5 -> 23.8; 20.2 -> 19.1, 512^2 42.7 -> 40.8; 31.6 -> 30.4.
 *
 * Above 48 waves on that CU the march takes over: its chunks then have rows
 * enough to pay for their prologue, and it computes no halo row twice. Rows
 * against march at 30 to 48 waves (512^2, 3000x150, and mass/energy and
 * momentum at 700^2): 7 to 22% faster; at 56 (the Lagrangian at 700^2) 7%
 * slower in FP64 and 3% faster in FP32; at 75 to 112 (1000^2) 2 to 18% slower.
 * A given chunk height asks for the march. */
constexpr int kRowsMostWaves = 48;

struct RowsGrid {
  int waves;
  MarchList ml;
};
inline RowsGrid rows_grid(int nx, int ny, int chunk_rows, int W, int halo) {
  RowsGrid best{0, {}};
  if (chunk_rows > 0) return best;
  long least = kRowsMostWaves + 1;
  for (int nw = kRowsMinWaves; nw <= kRowsMaxWaves; ++nw) {
    const MarchList ml = make_march(nx, ny, W, nw - halo);
    const long waves = (long)nw * ((ml.nitems + march_cus() - 1) / march_cus());
    if (ml.nitems < 1 || ml.nitems > kMaxReduceBlocks || waves >= least) continue;
    best = RowsGrid{nw, ml};
    least = waves;
  }
  return best;
}

template <typename T, bool P2, bool UNI>
hipError_t launch_rows_lagrangian(const RowsGrid& rg, MGeo<T> g, MLagIO<T> io, FkReduce r,
                                  double max_dt, int* parts, hipStream_t s) {
  if (!r.queue) return hipErrorInvalidValue;
  hipLaunchKernelGGL((k_rows_lagrangian<T, P2, UNI>), dim3(rg.ml.nitems),
                     dim3(rg.waves * kWave), 0, s, g, io, r, max_dt, rg.ml);
  *parts = rg.ml.nitems;
  return hipGetLastError();
}

template <typename T, bool P2, bool UNI>
hipError_t launch_rows_mass(const RowsGrid& rg, MGeo<T> g, MMassIO<T> io, int tt, FkReduce r,
                            MarchStep st, int* parts, hipStream_t s) {
  if (!r.queue) return hipErrorInvalidValue;
  const dim3 grid(rg.ml.nitems), block(rg.waves * kWave);
  if (tt % 2 == 0)
    hipLaunchKernelGGL((k_rows_mass_xy<T, P2, UNI>), grid, block, 0, s, g, io, r, st, rg.ml);
  else
    hipLaunchKernelGGL((k_rows_mass_yx<T, P2, UNI>), grid, block, 0, s, g, io, r, st, rg.ml);
  *parts = rg.ml.nitems;
  return hipGetLastError();
}

template <typename T, bool P2, bool UNI>
hipError_t launch_rows_momxy(const RowsGrid& rg, MGeo<T> g, MMom2IO<T> io, int tt, FkReduce r,
                             int parts, hipStream_t s) {
  if (!r.queue) return hipErrorInvalidValue;
  /* one block more, for the step's epilogue */
  const dim3 grid(rg.ml.nitems + 1), block(rg.waves * kWave);
  if (tt % 2)
    hipLaunchKernelGGL((k_rows_momxy_xy<T, P2, UNI>), grid, block, 0, s, g, io, r, parts, rg.ml);
  else
    hipLaunchKernelGGL((k_rows_momxy_yx<T, P2, UNI>), grid, block, 0, s, g, io, r, parts, rg.ml);
  return hipGetLastError();
}

/* Dispatch on whether every mesh spacing is a power of two (quotients by
 * spacings become products with exact reciprocals) and whether the mesh is
 * uniform (MUni): launch<P2, UNI>. */
template <typename F>
hipError_t by_geometry(int pow2, int uniform, F&& launch) {
  using Yes = std::true_type;
  using No = std::false_type;
  if (uniform) return pow2 ? launch(Yes{}, Yes{}) : launch(No{}, Yes{});
  return pow2 ? launch(Yes{}, No{}) : launch(No{}, No{});
}

template <typename T>
hipError_t launch_march_mass(MGeo<T> g, MMassIO<T> io, int tt, FkReduce r, MarchStep st,
                             int* parts, int chunk_rows, int pow2, int uniform, int pairs,
                             hipStream_t s) {
  if (pairs_wanted(pairs, g.nx, g.ny) && pow2 && uniform && pairs_fit(g, io))
    return launch_march_mass_p<T, true, true, true>(g, io, tt, r, st, parts, chunk_rows, s);
  const RowsGrid rg = rows_grid(g.nx, g.ny, chunk_rows, kMassW,
                                tt % 2 ? kRowsMassYXHalo : kRowsMassXYHalo);
  if (rg.waves)
    return by_geometry(pow2, uniform, [&](auto p2, auto uni) {
      return launch_rows_mass<T, decltype(p2)::value, decltype(uni)::value>(
          rg, g, io, tt, r, st, parts, s);
    });
  return by_geometry(pow2, uniform, [&](auto p2, auto uni) {
    return launch_march_mass_p<T, decltype(p2)::value, decltype(uni)::value>(
        g, io, tt, r, st, parts, chunk_rows, s);
  });
}

template <typename T>
hipError_t launch_march_lagrangian(MGeo<T> g, MLagIO<T> io, FkReduce r, double max_dt,
                                   int* parts, int chunk_rows, int pow2, int uniform,
                                   int pairs, hipStream_t s) {
  if (pairs_wanted(pairs, g.nx, g.ny) && pow2 && uniform && lag_pairs_fit(g, io))
    return launch_march_lagrangian_p<T, true, true, true>(g, io, r, max_dt, parts,
                                                          chunk_rows, s);
  const RowsGrid rg = rows_grid(g.nx, g.ny, chunk_rows, kLagW, kRowsLagHalo);
  if (rg.waves)
    return by_geometry(pow2, uniform, [&](auto p2, auto uni) {
      return launch_rows_lagrangian<T, decltype(p2)::value, decltype(uni)::value>(
          rg, g, io, r, max_dt, parts, s);
    });
  return by_geometry(pow2, uniform, [&](auto p2, auto uni) {
    return launch_march_lagrangian_p<T, decltype(p2)::value, decltype(uni)::value>(
        g, io, r, max_dt, parts, chunk_rows, s);
  });
}

template <typename T>
hipError_t launch_march_momentum(MGeo<T> g, MMomIO<T> io, int tt, int ydir, FkReduce r,
                                 int parts, int chunk_rows, int pow2, hipStream_t s) {
  return pow2 ? launch_march_momentum_p<T, true>(g, io, tt, ydir, r, parts, chunk_rows, s)
              : launch_march_momentum_p<T, false>(g, io, tt, ydir, r, parts, chunk_rows, s);
}

template <typename T>
hipError_t launch_march_momxy(MGeo<T> g, MMom2IO<T> io, int tt, FkReduce r, int parts,
                              int chunk_rows, int pow2, int uniform, hipStream_t s) {
  const RowsGrid rg = rows_grid(g.nx, g.ny, chunk_rows, kMomXYW,
                                tt % 2 ? kRowsMomXYHalo : kRowsMomYXHalo);
  if (rg.waves)
    return by_geometry(pow2, uniform, [&](auto p2, auto uni) {
      return launch_rows_momxy<T, decltype(p2)::value, decltype(uni)::value>(
          rg, g, io, tt, r, parts, s);
    });
  return by_geometry(pow2, uniform, [&](auto p2, auto uni) {
    return launch_march_momxy_p<T, decltype(p2)::value, decltype(uni)::value>(
        g, io, tt, r, parts, chunk_rows, s);
  });
}

}  // namespace flowhip

using namespace flowhip;

static MGeo<double> mgeo64(FkMesh m) {
  MGeo<double> g{m.nx, m.ny, m.edgedx, m.edgedy, m.celldx, m.celldy,
                 m.inv_edgedx, m.inv_edgedy, uniform_of<double>(m.u)};
  return g;
}

extern "C" {

hipError_t fk_march_lagrangian(FkMesh m, const double* rho, const double* e,
                               const double* mom_x, const double* mom_y, double* mx1,
                               double* my1, double* u0, double* v0, double* e1,
                               double* rho_old, FkReduce r, double max_dt, int* parts,
                               int chunk_rows, hipStream_t s) {
  MLagIO<double> io{rho, e, mom_x, mom_y, mx1, my1, u0, v0, e1, rho_old, r.cfl};
  return launch_march_lagrangian<double>(mgeo64(m), io, r, max_dt, parts, chunk_rows, m.pow2,
                                         m.uniform, m.pairs, s);
}

hipError_t fk_march_momentum(FkMesh m, int tt, const double* u0, const double* v0,
                             const double* F_x, const double* F_y, const double* rho,
                             const double* mx1, const double* my1, double* mom_x,
                             double* mom_y, double* u, double* v, FkReduce r,
                             int parts, int chunk_rows, hipStream_t s) {
  MMom2IO<double> io{u0, v0, F_x, F_y, rho, mx1, my1, mom_x, mom_y, u, v};
  return launch_march_momxy<double>(mgeo64(m), io, tt, r, parts, chunk_rows,
                                    m.pow2, m.uniform, s);
}

hipError_t fk_march_momentum_x(FkMesh m, int tt, const double* u0,
                               const double* v0, const double* F_x,
                               const double* F_y, const double* rho,
                               const double* mx1, double* mom_x, double* u,
                               FkReduce r, int chunk_rows, hipStream_t s) {
  MMomIO<double> io{u0, v0, F_x, F_y, rho, mx1, mom_x, u};
  return launch_march_momentum<double>(mgeo64(m), io, tt, 0, r, 0, chunk_rows, m.pow2, s);
}

hipError_t fk_march_momentum_y(FkMesh m, int tt, const double* u1,
                               const double* v0, const double* F_x,
                               const double* F_y, const double* rho,
                               const double* my1, double* mom_y, double* v,
                               FkReduce r, int parts, int chunk_rows, hipStream_t s) {
  MMomIO<double> io{u1, v0, F_x, F_y, rho, my1, mom_y, v};
  return launch_march_momentum<double>(mgeo64(m), io, tt, 1, r, parts, chunk_rows, m.pow2, s);
}

hipError_t fk_march_mass_energy(FkMesh m, int tt, const double* u0,
                                const double* v0, const double* rho0,
                                const double* e1, double* rho, double* e,
                                double* F_x, double* F_y, FkReduce r, double max_dt,
                                int first_step, int lag_parts, int* parts,
                                int chunk_rows, hipStream_t s) {
  MMassIO<double> io{u0, v0, rho0, e1, rho, e, F_x, F_y};
  const MarchStep st{max_dt, first_step, lag_parts};
  return launch_march_mass<double>(mgeo64(m), io, tt, r, st, parts, chunk_rows, m.pow2, m.uniform,
                                   m.pairs, s);
}

static MGeo<float> mgeo32(FkMesh32 m) {
  MGeo<float> g{m.nx, m.ny, m.edgedx, m.edgedy, m.celldx, m.celldy,
                m.inv_edgedx, m.inv_edgedy, uniform_of<float>(m.u)};
  return g;
}

hipError_t fk_march_lagrangian_f32(FkMesh32 m, const float* rho, const float* e,
                                   const float* mom_x, const float* mom_y,
                                   float* mx1, float* my1, float* u0, float* v0,
                                   float* e1, float* rho_old, FkReduce r,
                                   double max_dt, int* parts, int chunk_rows,
                                   hipStream_t s) {
  MLagIO<float> io{rho, e, mom_x, mom_y, mx1, my1, u0, v0, e1, rho_old};
  return launch_march_lagrangian<float>(mgeo32(m), io, r, max_dt, parts, chunk_rows, m.pow2,
                                        m.uniform, m.pairs, s);
}

hipError_t fk_march_mass_energy_f32(FkMesh32 m, int tt, const float* u0,
                                    const float* v0, const float* rho0,
                                    const float* e1, float* rho, float* e,
                                    float* F_x, float* F_y, FkReduce r, double max_dt,
                                    int first_step, int lag_parts, int* parts,
                                    int chunk_rows, hipStream_t s) {
  MMassIO<float> io{u0, v0, rho0, e1, rho, e, F_x, F_y};
  const MarchStep st{max_dt, first_step, lag_parts};
  return launch_march_mass<float>(mgeo32(m), io, tt, r, st, parts, chunk_rows, m.pow2, m.uniform,
                                  m.pairs, s);
}

hipError_t fk_march_momentum_f32(FkMesh32 m, int tt, const float* u0, const float* v0,
                                 const float* F_x, const float* F_y, const float* rho,
                                 const float* mx1, const float* my1, float* mom_x,
                                 float* mom_y, float* u, float* v, FkReduce r,
                                 int parts, int chunk_rows, hipStream_t s) {
  MMom2IO<float> io{u0, v0, F_x, F_y, rho, mx1, my1, mom_x, mom_y, u, v};
  return launch_march_momxy<float>(mgeo32(m), io, tt, r, parts, chunk_rows,
                                   m.pow2, m.uniform, s);
}

hipError_t fk_march_momentum_x_f32(FkMesh32 m, int tt, const float* u0,
                                   const float* v0, const float* F_x,
                                   const float* F_y, const float* rho,
                                   const float* mx1, float* mom_x, float* u,
                                   FkReduce r, int chunk_rows, hipStream_t s) {
  MMomIO<float> io{u0, v0, F_x, F_y, rho, mx1, mom_x, u};
  return launch_march_momentum<float>(mgeo32(m), io, tt, 0, r, 0, chunk_rows, m.pow2, s);
}

hipError_t fk_march_momentum_y_f32(FkMesh32 m, int tt, const float* u1,
                                   const float* v0, const float* F_x,
                                   const float* F_y, const float* rho,
                                   const float* my1, float* mom_y, float* v,
                                   FkReduce r, int parts, int chunk_rows, hipStream_t s) {
  MMomIO<float> io{u1, v0, F_x, F_y, rho, my1, mom_y, v};
  return launch_march_momentum<float>(mgeo32(m), io, tt, 1, r, parts, chunk_rows, m.pow2, s);
}

}  // extern "C"
