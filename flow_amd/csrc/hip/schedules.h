/*
 * schedules.h -- the kernel sequences that make up one solve_hydro_2d step.
 */
#ifndef FLOWHIP_SCHEDULES_H
#define FLOWHIP_SCHEDULES_H

#include "flowhip_ctx.h"

/* Enqueue one step on h->stream (device dt pair already current); with
 * graphs on, replayed from the step graph of its kind. */
void flowhip_enqueue_step(FlowHipCtx* h, const FlowHipStep* st);

/* The two schedules. */
void flowhip_step_stagewise(FlowHipCtx* h, const FlowHipStep* st);
void flowhip_step_fused(FlowHipCtx* h, const FlowHipStep* st);

void flowhip_last_sums(Mesh* mesh, double* mass, double* energy);

/* A mesh without two interior cells a side is fatal. */
void flowhip_check_size(const Mesh* mesh);
/* The launch arguments of step tt on solve_hydro_2d's 16 arrays. */
FlowHipStep flowhip_step_of(Mesh* mesh, int tt, double** a);
void flowhip_enqueue_timestep(FlowHipCtx* h, FkMesh m, const double* Qxx, const double* Qyy,
                              const double* rho, const double* e, double max_dt,
                              int first_step);

/* main.c:64-115's loop for flowhip_run and flowhip_run_f32: pre(arg) puts the
 * pre-loop set_timestep on the stream, step(arg, tt) step tt (any number) and
 * its totals. The other arguments are flowhip_run's. */
int flowhip_run_loop(FlowHipCtx* h, Mesh* mesh, void (*pre)(void*), void (*step)(void*, int),
                     void* arg, const char* who, int niters, int tt0, int pre_timestep,
                     double* dt_pairs, double* mass, double* energy, double* wall_seconds,
                     int* undefined);

#endif
