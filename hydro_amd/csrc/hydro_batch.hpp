// Internal interface of the batched kernels (hydro_batch.hip).
#pragma once
#include "hydro_kernels.hpp"
#include "hydro_numerics.hpp"

namespace hydro {

constexpr int kInstSlots = 64;        // CFL max slots per instance
constexpr int kBoundaryChunk = 1024;  // (line, var) ghost fills per boundary task

// One instance as the batched kernels see it (device array, rebuilt by the
// host whenever the set of instances changes).
template <typename S>
struct InstDev {
  GridGeom g;
  Phys<S> ph;
  double dx, cf, smallc;  // dt = cf*dx / max(cx, cy, smallc)
  GridView<S> buf[2];     // state in buf[0] between steps; with march, after step n0
                          // (RunCtl::nstep) and every other one from there
  RunCtl* ctl;
  uint64_t* cour;         // 2 * kInstSlots
  int bl, br, bd, bu;     // boundary types
  int fold;               // the sweeps form the ghosts (else k_batch_boundary does)
  int nseg;               // 60-cell segments per row
  int yseg;               // rows each wave marches in this instance's y tasks
  int march, n0;          // whole steps, and their rows a wave; 0: the two sweeps
};

// One workgroup's work: kind 1 = x (a = first segment), 2 = y (a = 64-column
// block, b = row-segment group), 3 = whole steps (a = 60-column block, b = row
// segment); for ghost fills kind is the direction.
struct BTask {
  int inst, kind, a, b;
};

// An instance's share of one task list: `count` tasks from tasks[first] on;
// task k has a = k * per, b = 0, or with ncb > 0 a = k % ncb, b = k / ncb.
struct BList {
  int inst, kind, first, count, per, ncb;
};

struct BatchTune {
  int waves;  // waves per workgroup (1..4)
  int xiter;  // segments each wave walks in an x task; 0: by the load
  int yseg;   // at most this many rows per wave in a y task (each instance
              // splits its rows evenly into row groups of waves x yseg); 0:
              // by the load
};

// kind 1: x tasks, 2: y tasks (a phase launches both, on their own tables).
// The first nst1 tasks belong to instances with slope_type == 1.  ghosts: the
// ghost values formed on the way are stored in buffer 0.  waves per
// workgroup, xiter segments per wave in x tasks.
template <typename S>
void launch_batch_sweep(int kind, const InstDev<S>* inst, const BTask* tasks, int ntask,
                        int nst1, int phase, bool ghosts, int waves, int xiter, hipStream_t st);
// Whole steps (fast and mixed forms), on a table of kind 3: of instances with
// march > 0, from the buffer their state is in into the other.
void launch_batch_march(const InstDev<float>* inst, const BTask* tasks, int ntask, int nst1,
                        hipStream_t st);
void launch_batch_march_fast(const InstDev<double>* inst, const BTask* tasks, int ntask, int nst1,
                             hipStream_t st);
template <typename S>
void launch_batch_boundary(const InstDev<S>* inst, const BTask* tasks, int ntask, int phase,
                           hipStream_t st);
template <typename S>
void launch_batch_courant(const InstDev<S>* inst, const int* ids, int nids, hipStream_t st);
template <typename S>
void launch_batch_ctl(const InstDev<S>* inst, const int* ids, int nids, bool begin,
                      hipStream_t st);
void launch_batch_tasks(const BList* lists, int n, BTask* tasks, hipStream_t st);

void launch_batch_set_ctl(RunCtl* c, double t, double dt, double tend, int nstep, int nstepmax,
                          int active, hipStream_t st);
void launch_zero_u64(uint64_t* p, long n, hipStream_t st);
// The FP64 fast form's batched sweeps (hydro_batch.hip, fast unit): as
// launch_batch_sweep for double, with the kFast arithmetic.
void launch_batch_sweep_fast(int kind, const InstDev<double>* inst, const BTask* tasks,
                             int ntask, int nst1, int phase, bool ghosts, int waves, int xiter,
                             hipStream_t st);

}  // namespace hydro
