/*
 * rows.h -- the three kernels of a march step in row-parallel form, for meshes
 * too small to fill the GPU with marching waves.
 *
 * A march wave takes the rows of its chunk one after the other, and on a
 * small mesh that chain is the kernel's time: 2000 to 3000 cycles a row of
 * dependent arithmetic (a wave alone on its SIMD waits 8 cycles for each
 * result, 70 for a quotient), two to seven rows of it with the prologue, while
 * most of the GPU idles. Here a block takes a strip of columns by R rows with
 * one wave per row, halo rows included: every stage of the step runs on all
 * the block's rows at once, and rows exchange their values through LDS, with
 * a barrier between stages in place of the march's row windows. Along x a
 * wave is as in the marches (columns in lanes, neighbours by DPP moves), and
 * the arithmetic is the same pointwise code in the same order, so the fields
 * are bitwise the march's. A wave whose row lies outside the domain computes
 * the row it mirrors; the waves past a short last chunk compute rows that
 * nothing reads.
 *
 * What bounds a block (cycles of the 8600 to 9500 at 64^2): the first loads
 * 1300 to 2200, the flux and velocity stages about 1500 each, the barriers
 * 100 to 500 each, the folds and sums of the totals about 3000; beside them
 * 1.9 us a launch. At 512^2, with 28 waves a CU, issue slots bound it: FP64
 * operations issue every 4.6 cycles on a SIMD. The halo rows (1 to 5 of 8 to
 * 16) are the price, hence the tall blocks where the mesh has rows enough.
 * Measured on MI355X (us a step, FP64; FP32), marches and then this form:
 * 64^2 29.8 -> 17.3; 26.9 -> 15.5, 300x200 32.3 -> 23.0; 27.1 -> 18.0, 512^2
 * 48.0 -> 37.9; 34.6 -> 29.4, 3000x150 59.1 -> 51.1; 42.3 -> 37.5.
 */
#pragma once

#include "march.h"

namespace flowhip {

constexpr int kRowsMinWaves = 8, kRowsMaxWaves = 16;
/* halo rows: a block of n waves owns n less these */
constexpr int kRowsLagHalo = 5;
constexpr int kRowsMassXYHalo = 4, kRowsMassYXHalo = 1;
constexpr int kRowsMomXYHalo = 5, kRowsMomYXHalo = 2;

/* Spacings at a lane's column q (clamped to where the arrays have a value:
 * 1 .. nx) and of the rows; rcdx and rcdy stand in for quotients on
 * power-of-two meshes. */
template <typename T, bool P2, bool UNI>
struct RowsGeo {
  T edx, edx1, cdx, cdxm, iedx, rcdx;
  RowS<T, UNI> edy, cdy, iedy;
  RowR<T, P2, UNI> rcdy;
  __device__ RowsGeo(const MGeo<T>& g, int q)
      : edy(g.edy, g.u.edy, 0, g.ny, 0),
        cdy(g.cdy, g.u.cdy, 0, g.ny, 0),
        iedy(g.iedy, g.u.iedy, 0, g.ny, 0),
        rcdy(g.cdy, g.u.rcdy, 0, g.ny, 0) {
    const int k = min(max(q, 1), g.nx);
    edx = geo_at<UNI>(g.edx, g.u.edx, k);
    edx1 = geo_at<UNI>(g.edx, g.u.edx, min(k + 1, g.nx));
    cdx = geo_at<UNI>(g.cdx, g.u.cdx, k);
    cdxm = geo_at<UNI>(g.cdx, g.u.cdx, k - 1);
    iedx = geo_at<UNI>(g.iedx, g.u.iedx, k);
    rcdx = UNI ? g.u.rcdx : T(1.0) / cdx;
  }
};

/* one value per column and row of a block */
template <typename T>
using RowsLds = T[kRowsMaxWaves][kWave];

/* ======================================================================= */
/* Lagrangian: lagrangian_box's arithmetic                                   */
/* ======================================================================= */

/* Wave w holds cell row and y face f = y0 - 2 + w: v after pressure
 * acceleration at face f, the x stages of row f, Qyy of row f, v after the
 * viscous step at face f, shock heating of row f. */
template <typename T, bool P2, bool UNI>
__global__ __launch_bounds__(kRowsMaxWaves * kWave) void k_rows_lagrangian(
    MGeo<T> g, MLagIO<T> io, FkReduce red, double max_dt, MarchList ml) {
  __shared__ RowsLds<T> s_v, s_q;
  const T dt = T(red.dtp[0]), dt_h = T(red.dtp[1]);
  if (blockIdx.x == 0) march_queue_reset(red.queue, kStageLag);
  const int nx = g.nx, ny = g.ny, sx = nx + 1;
  const int lane = threadIdx.x % kWave;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const ItemBox box = item_box(ml, nx, ny, blockIdx.x);
  const int x0 = box.x0, x1 = box.x1, y0 = box.y0, y1 = box.y1;
  const bool edge = box_edge(box, nx, ny), xedge = box_xedge(box, nx);
  const bool last_chunk = y1 == ny - kPad;
  double local_min = cfl_seed<T>(max_dt, red.dtp[1]);
  int nan_count = 0;

  const int q = x0 - 3 + lane;
  const RowsGeo<T, P2, UNI> m(g, q);
  const int qf = min(max(q, 0), nx), qc = min(max(q, 0), nx - 1);
  const bool face_ghost = is_ghost(q, sx), cell_ghost = is_ghost(q, nx);
  const int mf_lane = mirror_lane(lane, q, sx), mc_lane = mirror_lane(lane, q, nx);
  const bool own_face = q >= x0 && (q < x1 || (q == x1 && x1 == nx - kPad));
  const bool own = q >= x0 && q < x1;

  const int f = min(y0 - 2 + w, ny);
  const int fm = mirror(f, ny + 1); /* the face itself, or the one it mirrors */
  const bool row = f >= y0 && f < y1;
  const T rk = io.rho[fm * nx + qc], ek = io.e[fm * nx + qc];
  const T rs = io.rho[(fm - 1) * nx + qc], es_ = io.e[(fm - 1) * nx + qc];
  const T my = io.mom_y[fm * nx + qc];
  const T mx = io.mom_x[min(f, ny - 1) * sx + qf];

  /* the copy of rho: the strip's own columns and, beside a wall, the ghost ones
   * there; ghost rows by the waves that hold them */
  if (q >= (x0 == kPad ? 0 : x0) && q < (x1 == nx - kPad ? nx : x1)) {
    if (row)
      io.rho_old[f * nx + q] = rk;
    else if (is_ghost(f, ny) && f < ny)
      io.rho_old[f * nx + q] = io.rho[f * nx + q];
  }

  /* y face f after pressure acceleration; a ghost face is its negated mirror */
  const T Pk = eos_pressure(rk, ek);
  const T pm = accelerate<T, P2>(my, dt, Pk, eos_pressure(rs, es_), m.edy(fm),
                                     m.iedy(fm));
  const T pr = rho_edge_y<T, P2>(rk, rs, m.cdx, m.cdy(fm), m.cdy(fm - 1), m.edy(fm),
                                     T(0.5) * m.rcdx * m.iedy(fm));
  T v = velocity(pm, pr);
  if (fm != f) v = -v;
  s_v[w][lane] = v;

  /* along x on row f */
  T qx = T(0), uav = T(0);
  if (row) {
    const T mx_pa = accelerate<T, P2>(mx, dt, Pk, up(Pk, 1), m.edx, m.iedx);
    const T rex = rho_edge_x<T, P2>(rk, up(rk, 1), m.cdx, m.cdxm, m.cdy(f), m.edx,
                                       T(0.5) * m.iedx * m.rcdy(f));
    T u_pa = velocity(mx_pa, rex);
    u_pa = mirror_fix(xedge, u_pa, mf_lane, face_ghost, T(-1.0));
    qx = viscous_stress(rk, up(u_pa, 1), u_pa, dn(u_pa, 1), dn(u_pa, 2));
    qx = mirror_fix(xedge, qx, mc_lane, cell_ghost, T(1.0));
    const T mx_av = accelerate<T, P2>(mx_pa, dt, qx, up(qx, 1), m.cdx, m.rcdx);
    uav = velocity(mx_av, rex);
    if (own_face) {
      io.mx1[f * sx + q] = mx_av;
      mput_xface(edge, io.u0, nx, ny, f, q, uav, T(-1.0));
    }
  }
  __syncthreads();

  /* Qyy of the interior rows y0-1 .. y1 */
  T qy = T(0);
  if (f >= max(y0 - 1, kPad) && f <= min(y1, ny - kPad - 1)) {
    qy = viscous_stress(rk, s_v[w - 1][lane], v, s_v[w + 1][lane], s_v[w + 2][lane]);
    s_q[w][lane] = qy;
  }
  __syncthreads();

  /* y face f after the viscous acceleration (a ghost row's Qyy is its mirror
   * row's) */
  T vav = T(0);
  if (f >= y0 && f <= y1) {
    const T q_lo = f - 1 < kPad ? qy : s_q[w - 1][lane];
    const T q_hi = f >= ny - kPad ? s_q[w - 1][lane] : qy;
    const T my_av = accelerate<T, P2>(pm, dt, q_hi, q_lo, m.cdy(f), m.rcdy(f));
    vav = velocity(my_av, pr);
    if (own && (f < y1 || last_chunk)) {
      io.my1[f * nx + q] = my_av;
      mput_yface(edge, io.v0, nx, ny, f, q, vav, T(-1.0));
    }
    s_v[w][lane] = vav;
  }
  __syncthreads();

  if (row) {
    const T uav_e = dn(uav, 1), vav_e = s_v[w + 1][lane];
    if (own) {
      const int c = f * nx + q;
      const T es = shock_heating<T, P2>(ek, Pk, rk, qx, qy, uav, uav_e, vav, vav_e, m.cdx,
                                        m.cdy(f), dt_h, m.rcdx, m.rcdy(f));
      mput_cell(edge, io.e1, nx, ny, f, q, es);
      cfl_candidate<T>(io, c, es, qx, qy, rk, m.cdx, m.cdy(f), local_min, nan_count);
    }
  }
  publish_min<kRowsMaxWaves * kWave>(local_min, nan_count, red, blockDim.x / kWave);
}

/* ======================================================================= */
/* mass and energy                                                           */
/* ======================================================================= */

/* The block's totals: the waves leave the cells they own in LDS (zero
 * elsewhere), wave 0 adds up the mass and wave 1 the energy, column by column
 * with a march lane's sums. (Each
 * wave adding its cells into exact accumulators of its own cost 16 wave sums of
 * 192-bit integers a block: at 64^2 the step took 24.1 us for 21.9.)
 * The caller's last reads of s_r and s_e lie before its last barrier. */
template <typename T>
__device__ __forceinline__ void rows_totals(RowsLds<T>& s_r, RowsLds<T>& s_e, T rho, T e,
                                            int lane, int w, int rows, int first, FkReduce red) {
  s_r[w][lane] = rho;
  s_e[w][lane] = e;
  __syncthreads();
  if (w > 1) return;
  ItemSum<T> sum{0.0, 0.0};
#pragma unroll 4
  for (int k = first; k < first + rows; ++k) {
    const double r = double(s_r[k][lane]);
    sum.add(w == 0 ? r : r * double(s_e[k][lane]));
  }
  FixSum f{0, 0, 0, 0};
  f.add(sum.s + sum.c);
  const Words192 t = wave_sum192(Words192{f.w0, f.w1, f.w2});
  const bool bad = __ballot(f.bad != 0u) != 0ull;
  if (lane == kWave - 1) {
    unsigned long long* p = (unsigned long long*)(red.partials + kTotalsOffset) +
                            kTotalsWords * blockIdx.x + 4 * w;
    p[0] = t.w0;
    p[1] = t.w1;
    p[2] = t.w2;
    p[3] = bad;
  }
}

/* x sweep first (mass_xy_box's arithmetic). Wave w holds row and y face r =
 * y0 - 2 + w: the x sweep of row r, the y flux at face r, the y update of
 * row r. */
template <typename T, bool P2, bool UNI>
__global__ __launch_bounds__(kRowsMaxWaves * kWave) void k_rows_mass_xy(
    MGeo<T> g, MMassIO<T> io, FkReduce red, MarchStep st, MarchList ml) {
  __shared__ RowsLds<T> s_r, s_e, s_f, s_ef;
  const int nx = g.nx, ny = g.ny, sx = nx + 1;
  const int lane = threadIdx.x % kWave;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const ItemBox box = item_box(ml, nx, ny, blockIdx.x);
  const int x0 = box.x0, x1 = box.x1, y0 = box.y0, y1 = box.y1;
  const bool edge = box_edge(box, nx, ny);

  const int q = x0 - 2 + lane;
  const RowsGeo<T, P2, UNI> m(g, q);
  const bool face = q >= x0 && q <= x1, own = q >= x0 && q < x1;
  const bool own_face = face && (q < x1 || x1 == nx - kPad);
  const int qc = min(q, nx - 1), qf = min(q, nx);
  const int r = min(y0 - 2 + w, ny - 1);
  const int rm = mirror(r, ny);
  const bool row = r >= y0 && r < y1;
  const T a_r = io.rho0[rm * nx + qc], a_e = io.e1[rm * nx + qc];
  const T a_u = io.u0[rm * sx + qf];
  const T vm = io.v0[max(r - 1, 0) * nx + qc], v = io.v0[r * nx + qc],
          vp = io.v0[(r + 1) * nx + qc];
  const DtPair pair = mass_pair<T>(red, st);
  const T dt = T(pair.dt), dt_h = T(pair.dt_h);

  const T rm2 = up(a_r, 2), rm1 = up(a_r, 1), rp1 = dn(a_r, 1);
  const T em2 = up(a_e, 2), em1 = up(a_e, 1), ep1 = dn(a_e, 1);
  FaceFlux<T> fx = mass_energy_flux<T, false, P2>(up(a_u, 1), a_u, dn(a_u, 1), rm2, rm1, a_r,
                                                  rp1, em2, em1, a_e, ep1, m.iedx, m.cdxm, m.cdx,
                                                  m.edy(rm), dt, dt_h, m.rcdx);
  if (own_face && row) mput_xface(edge, io.F_x, nx, ny, r, q, fx.mass, T(-1.0));
  const T f_hi = dn(fx.mass, 1), ef_hi = dn(fx.energy, 1);
  const CellState<T> xs = sweep_update<T, P2>(a_r, a_r, a_e, fx.mass, f_hi, fx.energy, ef_hi,
                                              m.edy(rm), m.edy(rm + 1), m.cdx, m.cdy(rm), dt_h,
                                              true, m.rcdx * m.rcdy(rm));
  s_r[w][lane] = xs.rho;
  s_e[w][lane] = xs.e;
  __syncthreads();

  FaceFlux<T> fy{T(0), T(0)};
  if (r >= y0 && r <= y1) {
    fy = mass_energy_flux<T, true, P2>(vm, v, vp, s_r[w - 2][lane], s_r[w - 1][lane], xs.rho,
                                       s_r[w + 1][lane], s_e[w - 2][lane], s_e[w - 1][lane],
                                       xs.e, s_e[w + 1][lane], m.iedy(r), m.cdy(r - 1), m.cdy(r), m.edx, dt,
                                       dt_h, m.rcdy(r));
    if (own && (r < y1 || y1 == ny - kPad))
      mput_yface(edge, io.F_y, nx, ny, r, q, fy.mass, T(-1.0));
    s_f[w][lane] = fy.mass;
    s_ef[w][lane] = fy.energy;
  }
  __syncthreads();

  T out_r = T(0), out_e = T(0);
  if (row && own) {
    const CellState<T> ys =
        sweep_update<T, P2>(xs.rho, a_r, xs.e, fy.mass, s_f[w + 1][lane], fy.energy,
                            s_ef[w + 1][lane], m.edx, m.edx1, m.cdx, m.cdy(r), dt_h, false,
                            m.rcdx * m.rcdy(r));
    mput_cell(edge, io.rho, nx, ny, r, q, ys.rho);
    mput_cell(edge, io.e, nx, ny, r, q, ys.e);
    out_r = ys.rho;
    out_e = ys.e;
  }
  rows_totals<T>(s_r, s_e, out_r, out_e, lane, w, y1 - y0, 2, red);
}

/* y sweep first (mass_yx_box's arithmetic). Wave w holds y face and row r =
 * y0 + w: the y flux at face r, then the y update and the x sweep of row r. */
template <typename T, bool P2, bool UNI>
__global__ __launch_bounds__(kRowsMaxWaves * kWave) void k_rows_mass_yx(
    MGeo<T> g, MMassIO<T> io, FkReduce red, MarchStep st, MarchList ml) {
  __shared__ RowsLds<T> s_f, s_ef, s_r, s_e;
  const int nx = g.nx, ny = g.ny, sx = nx + 1;
  const int lane = threadIdx.x % kWave;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const ItemBox box = item_box(ml, nx, ny, blockIdx.x);
  const int x0 = box.x0, x1 = box.x1, y0 = box.y0, y1 = box.y1;
  const bool edge = box_edge(box, nx, ny);

  const int q = x0 - 2 + lane;
  const bool inq = q < nx;
  const bool face = q >= x0 && q <= x1, own = q >= x0 && q < x1;
  const bool own_face = face && (q < x1 || x1 == nx - kPad);
  /* the y sweep of a ghost column is that of its mirror column */
  const int qm = inq ? mirror(q, nx) : nx - kPad - 1;
  const int qc = min(q, nx - 1), qf = min(q, nx);
  const RowsGeo<T, P2, UNI> m(g, q);
  const RowsGeo<T, P2, UNI> mm(g, qm);
  const int r = min(y0 + w, y1);
  const bool row = y0 + w < y1;
  T wr[4], we[4], wv[3];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    wr[k] = io.rho0[(r - 2 + k) * nx + qm];
    we[k] = io.e1[(r - 2 + k) * nx + qm];
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) wv[k] = io.v0[(r - 1 + k) * nx + qm];
  const T c_u = io.u0[r * sx + qf], c_r0 = io.rho0[r * nx + qc];
  const DtPair pair = mass_pair<T>(red, st);
  const T dt = T(pair.dt), dt_h = T(pair.dt_h);

  const FaceFlux<T> fy = mass_energy_flux<T, true, P2>(wv[0], wv[1], wv[2], wr[0], wr[1],
                                                       wr[2], wr[3], we[0], we[1], we[2], we[3],
                                                       m.iedy(r), m.cdy(r - 1), m.cdy(r), mm.edx, dt, dt_h,
                                                       m.rcdy(r));
  if (own && q == qm && (row || (y0 + w == y1 && y1 == ny - kPad)))
    mput_yface(edge, io.F_y, nx, ny, r, q, fy.mass, T(-1.0));
  s_f[w][lane] = fy.mass;
  s_ef[w][lane] = fy.energy;
  __syncthreads();

  T out_r = T(0), out_e = T(0);
  if (row) {
    const CellState<T> ys =
        sweep_update<T, P2>(wr[2], wr[2], we[2], fy.mass, s_f[w + 1][lane], fy.energy,
                            s_ef[w + 1][lane], mm.edx, mm.edx1, mm.cdx, m.cdy(r), dt_h, true,
                            mm.rcdx * m.rcdy(r));
    const T rm2 = up(ys.rho, 2), rm1 = up(ys.rho, 1), rp1 = dn(ys.rho, 1);
    const T em2 = up(ys.e, 2), em1 = up(ys.e, 1), ep1 = dn(ys.e, 1);
    const FaceFlux<T> fx = mass_energy_flux<T, false, P2>(up(c_u, 1), c_u, dn(c_u, 1), rm2, rm1,
                                                          ys.rho, rp1, em2, em1, ys.e, ep1,
                                                          m.iedx, m.cdxm, m.cdx, m.edy(r), dt, dt_h,
                                                          m.rcdx);
    if (own_face) mput_xface(edge, io.F_x, nx, ny, r, q, fx.mass, T(-1.0));
    const T f_hi = dn(fx.mass, 1), ef_hi = dn(fx.energy, 1);
    if (own) {
      const CellState<T> xs =
          sweep_update<T, P2>(ys.rho, c_r0, ys.e, fx.mass, f_hi, fx.energy, ef_hi, m.edy(r),
                              m.edy(r + 1), m.cdx, m.cdy(r), dt_h, false, m.rcdx * m.rcdy(r));
      mput_cell(edge, io.rho, nx, ny, r, q, xs.rho);
      mput_cell(edge, io.e, nx, ny, r, q, xs.e);
      out_r = xs.rho;
      out_e = xs.e;
    }
  }
  rows_totals<T>(s_r, s_e, out_r, out_e, lane, w, y1 - y0, 0, red);
}

/* ======================================================================= */
/* momentum                                                                  */
/* ======================================================================= */

/* Odd tt (momxy_xy_box's arithmetic). Wave w holds row and y face k = y0 - 3 +
 * w: u after the x flux in x of row k, v after the y flux in x of face k and
 * the corner flux of row k, then the two remaining fluxes' updates. */
template <typename T, bool P2, bool UNI>
__global__ __launch_bounds__(kRowsMaxWaves * kWave) void k_rows_momxy_xy(
    MGeo<T> g, MMom2IO<T> io, FkReduce red, int parts, MarchList ml) {
  if (blockIdx.x == 0) {
    step_epilogue(red, parts);
    return;
  }
  __shared__ RowsLds<T> s_u, s_v, s_uf, s_vf;
  const T dt_h = T(red.dtp[3]);
  const int nx = g.nx, ny = g.ny, sx = nx + 1;
  const int lane = threadIdx.x % kWave;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const ItemBox box = item_box(ml, nx, ny, blockIdx.x - 1);
  const int x0 = box.x0, x1 = box.x1, y0 = box.y0, y1 = box.y1;
  const bool edge = box_edge(box, nx, ny), xedge = box_xedge(box, nx);
  const int gend = y1 == ny - kPad ? y1 + 1 : y1;

  const int q = x0 - 2 + lane;
  const RowsGeo<T, P2, UNI> m(g, q);
  const int qf = min(q, nx), qc = min(q, nx - 1);
  const bool cell_ghost = is_ghost(q, nx);
  const int mc_lane = mirror_lane(lane, q, nx);
  const bool own_x = q >= x0 && (q < x1 || (q == x1 && x1 == nx - kPad));
  const bool own_y = q >= x0 && q < x1;

  const int k0 = y0 - 3, k = k0 + w;
  /* cell rows k and k - 1, as the boundary copies them */
  const int i = mirror(min(max(k, 0), ny - 1), ny);
  const int ip = mirror(min(max(k - 1, 0), ny - 1), ny);
  const int kf = min(max(k, 0), ny), kf1 = min(kf + 1, ny);
  const T a_u = io.u0[i * sx + qf], a_fx = io.F_x[i * sx + qf], a_mx = io.mx1[i * sx + qf];
  const T a_r = io.rho[i * nx + qc];
  const T p_fx = io.F_x[ip * sx + qf], p_r = io.rho[ip * nx + qc];
  const T a_v = io.v0[kf * nx + qc], a_my = io.my1[kf * nx + qc];
  const T a_fy = io.F_y[kf * nx + qc], n_fy = io.F_y[kf1 * nx + qc];

  /* x stage: u1 and m1 of cell row k */
  T m1x, u1;
  {
    const T up1 = dn(a_u, 1);
    T ufx = momentum_flux(m.edy(i), a_fx, dn(a_fx, 1), up(a_u, 1), a_u, up1, dn(a_u, 2), m.iedx,
                          T(0.5) * (a_u + up1), m.cdxm, m.cdx, dt_h);
    ufx = mirror_fix(xedge, ufx, mc_lane, cell_ghost, T(1.0));
    m1x = advect_update<T, P2>(a_mx, dt_h, ufx, up(ufx, 1), m.edx, m.cdy(i),
                                m.iedx * m.rcdy(i));
    const T rex = rho_edge_x<T, P2>(a_r, up(a_r, 1), m.cdx, m.cdxm, m.cdy(i), m.edx,
                                       T(0.5) * m.iedx * m.rcdy(i));
    u1 = velocity(m1x, rex);
  }
  s_u[w][lane] = u1;
  __syncthreads();

  /* y stage: v1 and m1 of the interior faces k in [y0-2, y1+1]; x stage: the
   * x flux in y at corner rows y0 .. y1 */
  T m1y = T(0), v1 = T(0), uf = T(0);
  if (k >= max(y0 - 2, kPad) && k <= min(y1 + 1, ny - kPad)) {
    const T vfx = momentum_flux(m.cdy(k), a_fx, p_fx, up(a_v, 2), up(a_v, 1), a_v, dn(a_v, 1),
                                m.iedx, T(0.5) * (u1 + s_u[w - 1][lane]), m.cdxm, m.cdx, dt_h);
    m1y = advect_update<T, P2>(a_my, dt_h, dn(vfx, 1), vfx, m.edx, m.cdy(k),
                                m.iedx * m.rcdy(k));
    const T rey = rho_edge_y<T, P2>(a_r, p_r, m.cdx, m.cdy(k), m.cdy(k - 1), m.edy(k),
                                       T(0.5) * m.rcdx * m.iedy(k));
    v1 = velocity(m1y, rey);
    s_v[w][lane] = v1;
  }
  if (k >= y0 && k <= y1) {
    uf = momentum_flux(m.edx, a_fy, up(a_fy, 1), s_u[w - 2][lane], s_u[w - 1][lane], u1,
                       s_u[w + 1][lane], m.iedy(k), T(0.5) * (up(a_v, 1) + a_v), m.cdy(k - 1),
                       m.cdy(k), dt_h);
    s_uf[w][lane] = uf;
  }
  __syncthreads();

  /* x stage: the second update of row k; y stage: the y flux in y of the
   * interior cell rows y0-1 .. y1-1 (a ghost face's v1 is the negated mirror) */
  if (k >= y0 && k < y1) {
    const T uf_hi = s_uf[w + 1][lane];
    if (own_x) {
      io.mom_x[k * sx + q] = advect_update<T, P2>(m1x, dt_h, uf_hi, uf, m.cdx, m.edy(k),
                                                    m.rcdx * m.iedy(k));
      mput_xface(edge, io.u, nx, ny, k, q, u1, T(-1.0));
    }
  }
  T vfy = T(0);
  if (k >= max(y0 - 1, kPad) && k < y1) {
    auto face = [&](int j) {
      const int jm = mirror(j, ny + 1);
      const T t = s_v[jm - k0][lane];
      return jm == j ? t : -t;
    };
    const T w2 = face(k + 1);
    vfy = momentum_flux(m.cdx, a_fy, n_fy, face(k - 1), v1, w2, face(k + 2), m.iedy(k),
                        T(0.5) * (v1 + w2), m.cdy(k - 1), m.cdy(k), dt_h);
    s_vf[w][lane] = vfy;
  }
  __syncthreads();

  /* y stage: the second update of face k (a ghost row's flux is its mirror
   * row's) */
  if (k >= y0 && k < gend) {
    const T hi = k >= ny - kPad ? s_vf[w - 1][lane] : vfy;
    const T lo = k - 1 < kPad ? vfy : s_vf[w - 1][lane];
    if (own_y) {
      io.mom_y[k * nx + q] = advect_update<T, P2>(m1y, dt_h, hi, lo, m.cdx, m.edy(k),
                                                  m.rcdx * m.iedy(k));
      mput_yface(edge, io.v, nx, ny, k, q, v1, T(-1.0));
    }
  }
}

/* Even tt (momxy_yx_box's arithmetic). Wave w holds row and y face k = y0 - 1 +
 * w: the corner flux of row k and the y flux in y of row k, then u and v
 * after them, then the fluxes in x and the second updates. */
template <typename T, bool P2, bool UNI>
__global__ __launch_bounds__(kRowsMaxWaves * kWave) void k_rows_momxy_yx(
    MGeo<T> g, MMom2IO<T> io, FkReduce red, int parts, MarchList ml) {
  if (blockIdx.x == 0) {
    step_epilogue(red, parts);
    return;
  }
  __shared__ RowsLds<T> s_u, s_uf, s_vf;
  const T dt_h = T(red.dtp[3]);
  const int nx = g.nx, ny = g.ny, sx = nx + 1;
  const int lane = threadIdx.x % kWave;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const ItemBox box = item_box(ml, nx, ny, blockIdx.x - 1);
  const int x0 = box.x0, x1 = box.x1, y0 = box.y0, y1 = box.y1;
  const bool edge = box_edge(box, nx, ny), xedge = box_xedge(box, nx);
  const int gend = y1 == ny - kPad ? y1 + 1 : y1;

  const int q = x0 - 3 + lane;
  const RowsGeo<T, P2, UNI> m(g, q);
  const int qf = min(max(q, 0), nx), qc = min(max(q, 0), nx - 1);
  const bool face_ghost = is_ghost(q, sx), cell_ghost = is_ghost(q, nx);
  const int mf_lane = mirror_lane(lane, q, sx), mc_lane = mirror_lane(lane, q, nx);
  const bool own_x = q >= x0 && (q < x1 || (q == x1 && x1 == nx - kPad));
  const bool own_y = q >= x0 && q < x1;

  const int k = y0 - 1 + w;
  const int kr = min(k, ny - 1), kp = kr - 1;
  const int kf = min(k, ny);
  /* u0 rows k-2 .. k+1 and v0 faces k-1 .. k+2 (their ghosts are in memory) */
  T wu[4], wv[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    wu[s] = io.u0[min(max(k - 2 + s, 0), ny - 1) * sx + qf];
    wv[s] = io.v0[min(max(k - 1 + s, 0), ny) * nx + qc];
  }
  const T a_fy = io.F_y[kf * nx + qc], n_fy = io.F_y[min(k + 1, ny) * nx + qc];
  const T a_mx = io.mx1[kr * sx + qf], a_my = io.my1[kf * nx + qc];
  const T a_r = io.rho[kr * nx + qc], p_r = io.rho[kp * nx + qc];
  const T a_fx = io.F_x[kr * sx + qf], p_fx = io.F_x[kp * sx + qf];

  /* x stage: x flux in y at corner row k; y stage: y flux in y of row k */
  const T uf = momentum_flux(m.edx, a_fy, up(a_fy, 1), wu[0], wu[1], wu[2], wu[3], m.iedy(k),
                             T(0.5) * (up(wv[1], 1) + wv[1]), m.cdy(k - 1), m.cdy(k), dt_h);
  const T vfy = momentum_flux(m.cdx, a_fy, n_fy, wv[0], wv[1], wv[2], wv[3], m.iedy(k),
                              T(0.5) * (wv[1] + wv[2]), m.cdy(k - 1), m.cdy(k), dt_h);
  s_uf[w][lane] = uf;
  s_vf[w][lane] = vfy;
  __syncthreads();

  /* x stage: u1 of the interior rows y0-1 .. y1-1, and the second update of
   * rows y0 .. y1-1 */
  T u1 = T(0);
  if (k >= max(y0 - 1, kPad) && k < y1) {
    const T m1 = advect_update<T, P2>(a_mx, dt_h, s_uf[w + 1][lane], uf, m.cdx, m.edy(k),
                                      m.rcdx * m.iedy(k));
    const T rex = rho_edge_x<T, P2>(a_r, up(a_r, 1), m.cdx, m.cdxm, m.cdy(k), m.edx,
                                       T(0.5) * m.iedx * m.rcdy(k));
    u1 = velocity(m1, rex);
    u1 = mirror_fix(xedge, u1, mf_lane, face_ghost, T(-1.0));
    s_u[w][lane] = u1;
    if (k >= y0) {
      const T up1 = dn(u1, 1);
      T ufx = momentum_flux(m.edy(k), a_fx, dn(a_fx, 1), up(u1, 1), u1, up1, dn(u1, 2), m.iedx,
                            T(0.5) * (u1 + up1), m.cdxm, m.cdx, dt_h);
      ufx = mirror_fix(xedge, ufx, mc_lane, cell_ghost, T(1.0));
      const T ufx_lo = up(ufx, 1);
      if (own_x) {
        io.mom_x[k * sx + q] = advect_update<T, P2>(m1, dt_h, ufx, ufx_lo, m.edx, m.cdy(k),
                                                    m.iedx * m.rcdy(k));
        mput_xface(edge, io.u, nx, ny, k, q, u1, T(-1.0));
      }
    }
  }
  /* y stage: v1 of faces y0 .. (a ghost row's flux is its mirror row's) */
  T m1y = T(0), v1 = T(0);
  if (k >= y0 && k < gend) {
    const T hi = k >= ny - kPad ? s_vf[w - 1][lane] : vfy;
    const T lo = k - 1 < kPad ? vfy : s_vf[w - 1][lane];
    m1y = advect_update<T, P2>(a_my, dt_h, hi, lo, m.cdx, m.edy(k), m.rcdx * m.iedy(k));
    const T rey = rho_edge_y<T, P2>(a_r, p_r, m.cdx, m.cdy(k), m.cdy(k - 1), m.edy(k),
                                       T(0.5) * m.rcdx * m.iedy(k));
    v1 = velocity(m1y, rey);
    v1 = mirror_fix(xedge, v1, mc_lane, cell_ghost, T(1.0));
  }
  __syncthreads();

  /* y stage: y flux in x and the second update of face k (a ghost row's u is
   * its mirror row's) */
  if (k >= y0 && k < gend) {
    const T u_hi = k < ny - kPad ? u1 : s_u[w - 1][lane];
    const T u_lo = k - 1 < kPad ? u1 : s_u[w - 1][lane];
    const T vm1 = up(v1, 1);
    const T vfx = momentum_flux(m.cdy(k), a_fx, p_fx, up(v1, 2), vm1, v1, dn(v1, 1), m.iedx,
                                T(0.5) * (u_hi + u_lo), m.cdxm, m.cdx, dt_h);
    const T vfx_hi = dn(vfx, 1);
    if (own_y) {
      io.mom_y[k * nx + q] = advect_update<T, P2>(m1y, dt_h, vfx_hi, vfx, m.edx, m.cdy(k),
                                                  m.iedx * m.rcdy(k));
      mput_yface(edge, io.v, nx, ny, k, q, v1, T(-1.0));
    }
  }
}

}  // namespace flowhip
