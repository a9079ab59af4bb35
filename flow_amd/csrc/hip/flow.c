/*
 * flow.c -- the hip kernel set's implementation of flow_interface.h.
 *
 * C host code that drives hand-written HIP kernels through the thin C ABI of
 * flow_hip_kernels.h. Every array stays in device memory; the timestep pair
 * lives on the device between kernels. The kernels that settle the scalars
 * the caller reads (mesh->dt and mesh->dt_h, as main.c:95 requires, and the
 * totals) write them to pinned host memory too, so a call ends with one wait
 * and no transfer, and print_conservation after a step has nothing to wait
 * for.
 */
#include <stdio.h>
#include <string.h>

#include "../../../include/flow_interface.h"
#include "flowhip_ctx.h"
#include "schedules.h"

static const char* const kWho = "hip kernel set";

void flowhip_check_size(const Mesh* mesh) {
  /* a pad-2 reflection needs two interior cells to mirror along each axis */
  if (mesh->local_nx - 2 * mesh->pad < 2 || mesh->local_ny - 2 * mesh->pad < 2)
    TERMINATE("solve_hydro_2d: the mesh needs at least 2x2 interior cells "
              "(got %dx%d)", mesh->local_nx - 2 * mesh->pad,
              mesh->local_ny - 2 * mesh->pad);
}

FlowHipStep flowhip_step_of(Mesh* mesh, int tt, double** a) {
  FlowHipStep st;
  st.m = flowhip_fkmesh(mesh);
  st.tt = tt;
  st.max_dt = mesh->max_dt;
  st.P = a[0];
  st.rho = a[1];
  st.rho_old = a[2];
  st.e = a[3];
  st.u = a[4];
  st.v = a[5];
  st.mom_x = a[6];
  st.mom_y = a[7];
  st.Qxx = a[8];
  st.Qyy = a[9];
  st.F_x = a[10];
  st.F_y = a[11];
  st.uF_x = a[12];
  st.uF_y = a[13];
  st.vF_x = a[14];
  st.vF_y = a[15];
  return st;
}

/* omp3/flow.c:10-52 */
void solve_hydro_2d(Mesh* mesh, int tt, double* P, double* rho,
                    double* rho_old, double* e, double* u, double* v,
                    double* rho_u, double* rho_v, double* Qxx, double* Qyy,
                    double* F_x, double* F_y, double* uF_x, double* uF_y,
                    double* vF_x, double* vF_y, double* reduce_array) {
  (void)reduce_array;
  FlowHipCtx* h = flowhip_ctx(mesh);
  flowhip_check_size(mesh);
  if (mesh->rank == MASTER && mesh->verbose)
    printf("Timestep:        %.12e\n", mesh->dt);

  double* a[16] = {P,   rho, rho_old, e,   u,   v,    rho_u, rho_v,
                   Qxx, Qyy, F_x,     F_y, uF_x, uF_y, vF_x,  vF_y};
  const FlowHipStep st = flowhip_step_of(mesh, tt, a);
  flowhip_post_to(h, 0);
  h->sums_valid = 0; /* until this step leaves totals of its own */
  flowhip_push_pair(h, mesh);
  flowhip_enqueue_step(h, &st);
  flowhip_wait(h);
  flowhip_take_pair(h, mesh, 0, kWho);
}

/* omp3/flow.c:73-106 (reduce_all_min is the identity on one GPU) */
void flowhip_enqueue_timestep(FlowHipCtx* h, FkMesh m, const double* Qxx, const double* Qyy,
                              const double* rho, const double* e, double max_dt,
                              int first_step) {
  if (h->cfl_rule == FLOWHIP_CFL_OMP3_SERIAL)
    FK_LAUNCH(h, "timestep_serial",
              fk_timestep_serial(m, NULL, Qxx, Qyy, rho, e, h->red, max_dt, first_step,
                                 h->stream));
  else
    FK_LAUNCH(h, "timestep",
              fk_timestep(m, Qxx, Qyy, rho, e, h->red, max_dt, first_step, h->stream));
}

void set_timestep(const int nx, const int ny, double* Qxx, double* Qyy,
                  const double* rho, const double* e, Mesh* mesh,
                  double* reduce_array, const int first_step,
                  const double* celldx, const double* celldy) {
  (void)reduce_array;
  FlowHipCtx* h = flowhip_ctx(mesh);
  FkMesh m = flowhip_fkmesh(mesh);
  m.nx = nx;
  m.ny = ny;
  m.celldx = celldx;
  m.celldy = celldy;
  flowhip_post_to(h, 0);
  flowhip_push_pair(h, mesh);
  flowhip_enqueue_timestep(h, m, Qxx, Qyy, rho, e, mesh->max_dt, first_step);
  flowhip_wait(h);
  flowhip_take_pair(h, mesh, 0, kWho);
}

/* omp3/flow.c:973-995 (reduce_to_master is the identity on one GPU) */
void print_conservation(const int nx, const int ny, double* rho, double* e,
                        double* reduce_array, Mesh* mesh) {
  (void)reduce_array;
  FlowHipCtx* h = flowhip_ctx(mesh);
  if (!(h->sums_valid && h->sums_rho == rho && h->sums_e == e &&
        nx == mesh->local_nx && ny == mesh->local_ny)) {
    FkMesh m = flowhip_fkmesh(mesh);
    m.nx = nx;
    m.ny = ny;
    flowhip_post_to(h, 0);
    FK_LAUNCH(h, "conservation",
              fk_conservation(m, rho, e, h->red, h->stream));
    flowhip_wait(h);
  }
  /* posted by the launch above or, while sums_valid, by the last step */
  memcpy(h->totals, h->mail + 2, sizeof(h->totals));
  h->sums_valid = 0; /* a step's totals are used at most once */
  if (mesh->rank == MASTER && mesh->verbose) {
    printf("Total mass:      %.12e\n", h->totals[0]);
    printf("Total energy:    %.12e\n", h->totals[1]);
  }
}

/* Totals from the last print_conservation or step of flowhip_run. */
void flowhip_last_sums(Mesh* mesh, double* mass, double* energy) {
  FlowHipCtx* h = flowhip_ctx(mesh);
  *mass = h->totals[0];
  *energy = h->totals[1];
}
