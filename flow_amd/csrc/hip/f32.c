/*
 * f32.c -- the FP32-state precision form of the timestep.
 *
 * The 16 arrays of solve_hydro_2d are held as FP32 device arrays and the
 * march kernels run on them in FP32. Three things stay FP64: the CFL
 * candidates and the dt min-reduction (omp3/flow.c:77-105; the state is
 * widened before the sound speed is formed), the mass and energy totals
 * (omp3/flow.c:973-995; compensated FP64 sums of the widened state), and
 * the EOS pressure of near-vacuum cells (rho < 1e-6). The dt pair stays on
 * the device in FP64 and is rounded to FP32 inside each kernel.
 */
#include "schedules.h"

int flowhip_f32_alloc(float** buf, size_t len) {
  if (!buf) return -1;
  HIPCHECK(hipMalloc((void**)buf, sizeof(float) * (len ? len : 1)));
  HIPCHECK(hipMemset(*buf, 0, sizeof(float) * (len ? len : 1)));
  return 0;
}

void flowhip_f32_free(float* buf) {
  if (buf) HIPCHECK(hipFree(buf));
}

int flowhip_f32_zero(float* buf, size_t len) {
  HIPCHECK(hipMemset(buf, 0, sizeof(float) * len));
  return 0;
}

int flowhip_f32_copy(float* dev, float* host, size_t len, int dir) {
  HIPCHECK(hipDeviceSynchronize());
  if (dir == SEND)
    HIPCHECK(hipMemcpy(dev, host, sizeof(float) * len, hipMemcpyHostToDevice));
  else
    HIPCHECK(hipMemcpy(host, dev, sizeof(float) * len, hipMemcpyDeviceToHost));
  return 0;
}

int flowhip_f32_narrow(float* dst, const double* src, size_t len) {
  HIPCHECK(fk_narrow((long)len, dst, src, 0));
  HIPCHECK(hipDeviceSynchronize());
  return 0;
}

int flowhip_f32_widen(double* dst, const float* src, size_t len) {
  HIPCHECK(fk_widen((long)len, dst, src, 0));
  HIPCHECK(hipDeviceSynchronize());
  return 0;
}

int flowhip_f32_boundary(Mesh* mesh, float* arr, int nxp, int nyp, int invert) {
  FlowHipCtx* h = flowhip_ctx(mesh);
  HIPCHECK(fk_boundary_f32(nxp, nyp, mesh->pad, arr, invert, h->stream));
  HIPCHECK(hipStreamSynchronize(h->stream));
  return 0;
}

/* One step of omp3/flow.c:10-52 on FP32 state, in the march schedule's three
 * kernels (the same ping-pong use of P, Qxx, Qyy, uF_x, uF_y as the FP64
 * fused schedule). */
static void step_f32(FlowHipCtx* h, Mesh* mesh, FkMesh32 m, int tt, float** a) {
  float *P = a[0], *rho = a[1], *rho_old = a[2], *e = a[3], *u = a[4],
        *v = a[5], *mom_x = a[6], *mom_y = a[7], *Qxx = a[8], *Qyy = a[9],
        *F_x = a[10], *F_y = a[11], *uF_x = a[12], *uF_y = a[13];
  hipStream_t s = h->stream;
  int lag_parts = 0, parts = 0;
  FK_LAUNCH(h, "lagrangian_f32",
            fk_march_lagrangian_f32(m, rho, e, mom_x, mom_y, Qxx, Qyy, uF_x,
                                    uF_y, P, rho_old, h->red, mesh->max_dt, &lag_parts,
                                    flowhip_rows(h, FLOWHIP_K_LAGRANGIAN, 1), s));
  FK_LAUNCH(h, "advect_mass_energy_f32",
            fk_march_mass_energy_f32(m, tt, uF_x, uF_y, rho_old, P, rho, e,
                                     F_x, F_y, h->red, mesh->max_dt, tt == 0, lag_parts,
                                     &parts, flowhip_rows(h, FLOWHIP_K_MASS, 1), s));
  FK_LAUNCH(h, "advect_momentum_f32",
            fk_march_momentum_f32(m, tt, uF_x, uF_y, F_x, F_y, rho, Qxx, Qyy,
                                  mom_x, mom_y, u, v, h->red, parts,
                                  flowhip_rows(h, FLOWHIP_K_MOMENTUM, 1), s));
}

typedef struct RunArgs32 {
  FlowHipCtx* h;
  Mesh* mesh;
  float** a;
  FkMesh32 m;
} RunArgs32;

static void enqueue_pre_f32(void* arg) {
  RunArgs32* r = (RunArgs32*)arg;
  FlowHipCtx* h = r->h;
  FK_LAUNCH(h, "timestep_f32",
            fk_timestep_f32(r->m, r->a[8], r->a[9], r->a[1], r->a[3], h->red,
                            r->mesh->max_dt, 0, h->stream));
}

static void enqueue_step_f32(void* arg, int tt) {
  RunArgs32* r = (RunArgs32*)arg;
  step_f32(r->h, r->mesh, r->m, tt, r->a);
}

/* main.c:64-115 on FP32 state; the arguments mean what flowhip_run's do. */
int flowhip_run_f32(Mesh* mesh, float** a, int niters, int tt0,
                    int pre_timestep, double* dt_pairs, double* mass,
                    double* energy, double* wall_seconds, int* undefined) {
  if (niters < 0 || !a) return -1;
  if (mesh->local_nx - 2 * mesh->pad < 2 || mesh->local_ny - 2 * mesh->pad < 2)
    TERMINATE("flowhip_run_f32: the mesh needs at least 2x2 interior cells");
  RunArgs32 r = {flowhip_ctx(mesh), mesh, a, {0}};
  r.m = flowhip_fkmesh32(mesh);
  r.h->sums_valid = 0;
  return flowhip_run_loop(r.h, mesh, enqueue_pre_f32, enqueue_step_f32, &r,
                          "hip kernel set (FP32 state)", niters, tt0, pre_timestep, dt_pairs,
                          mass, energy, wall_seconds, undefined);
}
