/*
 * run.c -- flow_hip.h: schedule and graph controls, the restated driver
 * loop, and small device helpers for callers that hold their own buffers.
 */
#include <stdio.h>
#include <string.h>
#include <time.h>

#include "../../../include/flow_interface.h"
#include "flowhip_ctx.h"
#include "schedules.h"

int flowhip_set_schedule(Mesh* mesh, int schedule) {
  if (schedule != FLOWHIP_STAGEWISE && schedule != FLOWHIP_FUSED &&
      schedule != FLOWHIP_MARCH)
    return -1;
  flowhip_ctx(mesh)->schedule = schedule;
  return 0;
}

int flowhip_get_schedule(Mesh* mesh) { return flowhip_ctx(mesh)->schedule; }

int flowhip_set_march_rows(Mesh* mesh, int rows) {
  if (rows != 0 && (rows < 4 || rows > 120)) return -1;
  flowhip_ctx(mesh)->march_rows = rows;
  return 0;
}

int flowhip_set_graphs(Mesh* mesh, int on) {
  flowhip_ctx(mesh)->use_graphs = on ? 1 : 0;
  return 0;
}

static double now_seconds(void) {
  struct timespec ts;
  clock_gettime(CLOCK_MONOTONIC, &ts);
  return (double)ts.tv_sec + 1e-9 * (double)ts.tv_nsec;
}

/* How many of the next `most` steps can be enqueued before the host knows
 * their dt: none but the last of them may be the one after which elapsed
 * reaches sim_end. set_timestep's update gives dt = (C_T m + dt_h) / 2 and
 * dt_h' = C_T m or (first step) dt with m <= min(max_dt, C_M dt_h), which
 * grow with dt_h, so the largest values bound every later step's dt. */
static int steps_ahead(const Mesh* mesh, double elapsed, int most) {
  double dt_h = mesh->dt_h;
  int n = 0;
  while (n < most) {
    const double m = C_T * min(mesh->max_dt, C_M * dt_h);
    const double dt = 0.5 * (m + dt_h);
    elapsed += dt * (1.0 + 1.0e-9);
    dt_h = max(m, dt) * (1.0 + 1.0e-9);
    ++n;
    if (elapsed >= mesh->sim_end) break;
  }
  return n;
}

int flowhip_run_loop(FlowHipCtx* h, Mesh* mesh, void (*pre)(void*), void (*step)(void*, int),
                     void* arg, const char* who, int niters, int tt0, int pre_timestep,
                     double* dt_pairs, double* mass, double* energy, double* wall_seconds,
                     int* undefined) {
  /* replayed graphs post to the slot they were captured with; printed steps
   * wait their turn */
  const int alone = h->use_graphs || (mesh->rank == MASTER && mesh->verbose);
  double wall = 0.0, elapsed = 0.0;
  int k = 0;
  /* with nothing to run the pair stays where it is: no wait would follow */
  if (pre_timestep || niters > 0) flowhip_push_pair(h, mesh);
  if (pre_timestep) {
    flowhip_post_to(h, 0);
    pre(arg);
    flowhip_wait(h);
    flowhip_take_pair(h, mesh, 0, who);
  }
  if (dt_pairs) {
    dt_pairs[0] = mesh->dt;
    dt_pairs[1] = mesh->dt_h;
  }
  if (undefined) undefined[0] = pre_timestep ? h->undefined : 0;
  while (k < niters) {
    const int left = min(niters - k, FLOWHIP_AHEAD);
    const int n = alone ? 1 : steps_ahead(mesh, elapsed, left);
    const double w0 = now_seconds();
    for (int q = 0; q < n; ++q) {
      flowhip_post_to(h, q);
      step(arg, tt0 + k + q);
    }
    flowhip_wait(h);
    wall += now_seconds() - w0;
    for (int q = 0; q < n; ++q, ++k) {
      flowhip_take_pair(h, mesh, q, who);
      const double* m = h->mail + (size_t)q * FK_MAIL_WORDS;
      memcpy(h->totals, m + 2, sizeof(h->totals));
      if (mesh->rank == MASTER && mesh->verbose) {
        printf("\nIteration %d\n", tt0 + k + 1);
        printf("Total mass:      %.12e\n", h->totals[0]);
        printf("Total energy:    %.12e\n", h->totals[1]);
      }
      if (dt_pairs) {
        dt_pairs[2 * (k + 1)] = mesh->dt;
        dt_pairs[2 * (k + 1) + 1] = mesh->dt_h;
      }
      if (mass) mass[k] = h->totals[0];
      if (energy) energy[k] = h->totals[1];
      if (undefined) undefined[k + 1] = h->undefined;
      elapsed += mesh->dt;
      if (elapsed >= mesh->sim_end) {
        ++k;
        niters = k;
        break;
      }
    }
  }
  flowhip_post_to(h, 0);
  if (wall_seconds) *wall_seconds = wall;
  return k;
}

typedef struct RunArgs {
  FlowHipCtx* h;
  FlowHipStep st;
} RunArgs;

static void enqueue_pre_f64(void* arg) {
  const RunArgs* r = (const RunArgs*)arg;
  const FlowHipStep* st = &r->st;
  flowhip_enqueue_timestep(r->h, st->m, st->Qxx, st->Qyy, st->rho, st->e, st->max_dt, 0);
}

static void enqueue_step_f64(void* arg, int tt) {
  RunArgs* r = (RunArgs*)arg;
  FlowHipCtx* h = r->h;
  FlowHipStep* st = &r->st;
  st->tt = tt;
  h->sums_valid = 0;
  flowhip_enqueue_step(h, st);
  if (!h->sums_valid)
    FK_LAUNCH(h, "conservation", fk_conservation(st->m, st->rho, st->e, h->red, h->stream));
  h->sums_valid = 0; /* posted: print_conservation computes its own again */
}

/* main.c:64-115 */
int flowhip_run(Mesh* mesh, double** a, int niters, int tt0, int pre_timestep,
                double* dt_pairs, double* mass, double* energy,
                double* wall_seconds, int* undefined) {
  if (niters < 0 || !a) return -1;
  if (!(mesh->rank == MASTER && mesh->verbose)) {
    RunArgs r;
    r.h = flowhip_ctx(mesh);
    r.st = flowhip_step_of(mesh, tt0, a);
    if (niters > 0) flowhip_check_size(mesh);
    return flowhip_run_loop(r.h, mesh, enqueue_pre_f64, enqueue_step_f64, &r, "hip kernel set",
                            niters, tt0, pre_timestep, dt_pairs, mass, energy, wall_seconds,
                            undefined);
  }
  /* the calls main.c makes, with their prints */
  const int nx = mesh->local_nx, ny = mesh->local_ny;
  double wall = 0.0, elapsed = 0.0;
  if (pre_timestep)
    set_timestep(nx, ny, a[8], a[9], a[1], a[3], mesh, NULL, 0, mesh->celldx,
                 mesh->celldy);
  if (dt_pairs) {
    dt_pairs[0] = mesh->dt;
    dt_pairs[1] = mesh->dt_h;
  }
  if (undefined) undefined[0] = pre_timestep ? flowhip_undefined_candidates(mesh) : 0;
  int k;
  for (k = 0; k < niters; ++k) {
    const int tt = tt0 + k;
    printf("\nIteration %d\n", tt + 1);
    const double w0 = now_seconds();
    solve_hydro_2d(mesh, tt, a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], a[8], a[9],
                   a[10], a[11], a[12], a[13], a[14], a[15], NULL);
    print_conservation(nx, ny, a[1], a[3], NULL, mesh);
    wall += now_seconds() - w0;
    if (dt_pairs) {
      dt_pairs[2 * (k + 1)] = mesh->dt;
      dt_pairs[2 * (k + 1) + 1] = mesh->dt_h;
    }
    if (undefined) undefined[k + 1] = flowhip_undefined_candidates(mesh);
    double ms, es;
    flowhip_last_sums(mesh, &ms, &es);
    if (mass) mass[k] = ms;
    if (energy) energy[k] = es;
    elapsed += mesh->dt;
    if (elapsed >= mesh->sim_end) {
      ++k;
      break;
    }
  }
  if (wall_seconds) *wall_seconds = wall;
  return k;
}

int flowhip_device_sync(void) {
  HIPCHECK(hipDeviceSynchronize());
  return 0;
}

int flowhip_memset_zero(double* dev, size_t len) {
  HIPCHECK(hipMemset(dev, 0, sizeof(double) * len));
  return 0;
}

int flowhip_copy(double* dev, double* host, size_t len, int dir) {
  HIPCHECK(hipDeviceSynchronize());
  if (dir == SEND)
    HIPCHECK(hipMemcpy(dev, host, sizeof(double) * len, hipMemcpyHostToDevice));
  else
    HIPCHECK(hipMemcpy(host, dev, sizeof(double) * len, hipMemcpyDeviceToHost));
  return 0;
}

int flowhip_device_name(char* name, int name_len) {
  int dev = 0;
  hipDeviceProp_t prop;
  HIPCHECK(hipGetDevice(&dev));
  HIPCHECK(hipGetDeviceProperties(&prop, dev));
  snprintf(name, (size_t)name_len, "%s (%s, %d CUs)", prop.name,
           prop.gcnArchName, prop.multiProcessorCount);
  return 0;
}

int flowhip_mesh_size_ok(int global_nx, int global_ny) {
  return global_nx >= 2 && global_ny >= 2 && global_nx <= FLOWHIP_MAX_CELLS_SIDE &&
         global_ny <= FLOWHIP_MAX_CELLS_SIDE;
}

Mesh* flowhip_mesh_new(int global_nx, int global_ny, double width,
                       double height, double max_dt, double sim_end,
                       double dt_param) {
  if (!flowhip_mesh_size_ok(global_nx, global_ny)) return NULL;
  Mesh* m = (Mesh*)calloc(1, sizeof(Mesh));
  if (!m) return NULL;
  m->global_nx = global_nx;
  m->global_ny = global_ny;
  m->pad = 2;
  m->local_nx = global_nx + 2 * m->pad;
  m->local_ny = global_ny + 2 * m->pad;
  m->width = width;
  m->height = height;
  m->max_dt = max_dt;
  m->sim_end = sim_end;
  m->dt = C_T * dt_param;
  m->dt_h = m->dt;
  initialise_mpi(0, NULL, &m->rank, &m->nranks);
  initialise_comms(m);
  initialise_mesh_2d(m);
  return m;
}

void flowhip_mesh_delete(Mesh* mesh) {
  if (!mesh) return;
  finalise_mesh(mesh);
  free(mesh);
}
