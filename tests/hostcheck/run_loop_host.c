/*
 * run_loop_host.c -- flowhip_run_loop (run.c) over stand-ins for the calls it
 * makes, which write the order of those calls into a log: P the dt pair put on
 * its way to the device, W a wait for the stream, B the pre-loop time step, S a
 * step, T a step's results taken. Every step advances dt by its number.
 */
#include <stdlib.h>
#include <string.h>

#include "../../flow_amd/csrc/hip/run.c"

static char g_log[4096];
static size_t g_len;
static void note(char c) {
  if (g_len + 1 < sizeof(g_log)) g_log[g_len++] = c;
}

void flowhip_push_pair(FlowHipCtx* h, const Mesh* mesh) {
  (void)h;
  (void)mesh;
  note('P');
}
void flowhip_post_to(FlowHipCtx* h, int slot) {
  (void)h;
  (void)slot;
}
void flowhip_wait(FlowHipCtx* h) {
  (void)h;
  note('W');
}
void flowhip_take_pair(FlowHipCtx* h, Mesh* mesh, int slot, const char* what) {
  (void)h;
  (void)mesh;
  (void)slot;
  (void)what;
  note('T');
}
static void pre(void* arg) {
  (void)arg;
  note('B');
}
static void step(void* arg, int tt) {
  (void)arg;
  (void)tt;
  note('S');
}

/* the calls of one run, as a string */
const char* run_log(int niters, int tt0, int pre_timestep) {
  FlowHipCtx* h = (FlowHipCtx*)calloc(1, sizeof(FlowHipCtx));
  Mesh mesh;
  memset(&mesh, 0, sizeof(mesh));
  mesh.dt = mesh.dt_h = 1.0e-4;
  mesh.max_dt = mesh.sim_end = 1.0e30;
  h->mail = (double*)calloc(FK_MAIL_WORDS * FLOWHIP_AHEAD, sizeof(double));
  g_len = 0;
  memset(g_log, 0, sizeof(g_log));
  flowhip_run_loop(h, &mesh, pre, step, NULL, "test", niters, tt0, pre_timestep, NULL, NULL,
                   NULL, NULL, NULL);
  free(h->mail);
  free(h);
  return g_log;
}
