// Batched kernels: many independent grids (instances) of uneven sizes advanced
// per launch.  The arithmetic per cell is the single-grid code
// (hydro_sweeps.hpp), so every instance's result is bit-identical to running
// it alone.
//
// A step is two phases.  In each phase every instance does one sweep, x or y
// depending on its own step parity (even steps x then y, odd steps y then x,
// HydroC99_2DMpi/Src/main.c:285-291), so a phase's task table mixes x tasks
// of some instances with y tasks of others (the x and y tasks run as separate
// launches, and each list as two: instances with slope_type == 1 first, in
// the specialised variant).  One workgroup takes one task, handed out by the
// hardware's dispatcher: resident workgroups that drew task indices from an
// atomic counter got at most 86 M of them a second (one address), which held
// up every launch of small tasks (60 grids of 64-1024 a side, a step: FP64 701
// against 788 us, fast 434 against 495, mixed 294 against 330 at the same task
// shapes) and made tasks small enough to balance the load a loss.  A
// task is one workgroup's worth of one instance:
//   x task: wpb * xiter consecutive 60-cell row segments (each wave walks xiter)
//   y task: 64 columns x (wpb * yseg) rows (each wave marches yseg rows; the
//           instance's yseg evens its rows out over its row groups)
//   whole steps (large loads of the fast and mixed forms; one launch a step for
//           every parity): 60 columns x the instance's march rows, one wave
// so the CFL reduction of a task never mixes instances.  Run control (t, dt,
// nstep, active) and CFL slots are per instance, on the device.
//
// Compiled three times, as hydro_kernels.hip: the FP64 unit
// (-ffp-contract=off), the mixed-precision unit (HYDRO_MIXED_UNIT,
// -ffp-contract=on) with only the FP32-storage sweeps and CFL kernels, and
// the fast unit (HYDRO_FAST_UNIT, -ffp-contract=on) with only the FP64
// fast-form sweeps.
#include "hydro_batch.hpp"
#include "hydro_sweeps.hpp"

namespace hydro {

// The ghosts of one instance's sweep in direction idim (GhostFill).
template <typename S>
__device__ __forceinline__ GhostFill inst_ghosts(const InstDev<S>& d, int idim, int phase,
                                                 int ghosts) {
  if (!d.fold) return GhostFill{0, 0, 0};
  const int to = ghosts ? 1 + phase : 0;  // buffer 0: read in phase 0, written in phase 1
  return idim == 1 ? GhostFill{d.bl, d.br, to} : GhostFill{d.bd, d.bu, to};
}

// x tasks of one phase (every task's kind is 1).  ST1: every listed
// instance has slope_type == 1 (the host splits each phase's lists), so the
// limiter's multiply/divide by slope_type is compiled out as in single grids.
// FD: the arithmetic form (a batch keeps the SIMDs busy, so the FP64 batches
// take the range-gated divisions, kGated, for every instance).
// Built for 5 waves per SIMD, as the single-grid x sweep (the per-task state
// would otherwise take it to 98 VGPRs and 4 waves; one register spills).
template <typename S, bool ST1, int FD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) void k_batch_sweep_x(
    const InstDev<S>* __restrict__ inst, const BTask* __restrict__ tasks, int phase, int ghosts,
    int xiter) {
  const int wpb = blockDim.x >> 6;
  const BTask tk = tasks[blockIdx.x];
  const InstDev<S>& d = inst[tk.inst];
  if (!d.ctl->active) return;  // workgroup-uniform
  const double dtdx = d.ctl->dt / d.dx;
  const TraceK<S> tr = make_tracek<S>((S) dtdx, d.ph.scheme);
  const GridView<S> in = d.buf[phase], out = d.buf[1 - phase];
  const GhostFill gf = inst_ghosts(d, 1, phase, ghosts);
  // the second sweep of an odd step is an x sweep; it produces the CFL
  // maxima the next (even) step's dt needs
  const bool cour = phase == 1;
  double cx = 0.0, cy = 0.0;
  // segments tk.a + it * wpb + wave, it = 0 .. xiter-1
  SegWalk w(tk.a + wave_id(), d.nseg);
  for (int it = 0; it < xiter && w.row < d.g.ny; it++) {
    if (cour)
      x_segment<S, ST1, true, FD>(d.g, d.ph, tr, dtdx, in, out, gf, w.row, w.seg, cx, cy);
    else
      x_segment<S, ST1, false, FD>(d.g, d.ph, tr, dtdx, in, out, gf, w.row, w.seg, cx, cy);
    w.advance(wpb, d.nseg);
  }
  if (cour) commit_courant(cx, cy, d.cour, kInstSlots, blockIdx.x % kInstSlots);
}

// y tasks of one phase (every task's kind is 2); y sweeps never end a step
// whose successor needs dt, so they fold no CFL maxima.
template <typename S, bool ST1, int FD>
__global__ __launch_bounds__(256) void k_batch_sweep_y(const InstDev<S>* __restrict__ inst,
                                                       const BTask* __restrict__ tasks, int phase,
                                                       int ghosts) {
  const int wpb = blockDim.x >> 6;
  const int wave = wave_id();
  const BTask tk = tasks[blockIdx.x];
  const InstDev<S>& d = inst[tk.inst];
  if (!d.ctl->active) return;
  const double dtdx = d.ctl->dt / d.dx;
  const TraceK<S> tr = make_tracek<S>((S) dtdx, d.ph.scheme);
  const GridView<S> in = d.buf[phase], out = d.buf[1 - phase];
  const int col = tk.a * 64 + (threadIdx.x & 63);
  const bool colok = col < d.g.nx;
  const long i = 2 + (colok ? col : d.g.nx - 1);
  const int j0 = 2 + (tk.b * wpb + wave) * d.yseg;
  double cx = 0.0, cy = 0.0;
  if (j0 < d.g.ny + 2) {  // wave-uniform
    const int j1 = min(j0 + d.yseg, d.g.ny + 2);
    extern __shared__ __attribute__((aligned(16))) unsigned char ylds[];
    YStash<S>* ys = reinterpret_cast<YStash<S>*>(ylds) + wave;
    y_march<S, ST1, false, FD>(d.g, d.ph, tr, dtdx, in, out, inst_ghosts(d, 2, phase, ghosts),
                               colok, i, j0, j1, ys, cx, cy);
  }
}

// The buffer an instance's state is in between steps.
template <typename S>
__device__ __forceinline__ int state_buf(const InstDev<S>& d) {
  return d.march ? (d.ctl->nstep - d.n0) & 1 : 0;
}

#if defined(HYDRO_FAST_UNIT) || defined(HYDRO_MIXED_UNIT)
// Whole steps (step_march): of even steps x first, of odd ones y first with the
// CFL maxima of the new state.
template <typename S, bool ST1, int FD>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(
    sizeof(S) == 4 ? 5 : 4))) void k_batch_march(const InstDev<S>* __restrict__ inst,
                                                 const BTask* __restrict__ tasks) {
  const BTask tk = tasks[blockIdx.x];
  const InstDev<S>& d = inst[tk.inst];
  if (!d.ctl->active) return;  // workgroup-uniform
  const double dtdx = d.ctl->dt / d.dx;
  const TraceK<S> tr = make_tracek<S>((S) dtdx, d.ph.scheme);
  const int cur = state_buf(d);
  const GridView<S> in = d.buf[cur], out = d.buf[1 - cur];
  __shared__ YStash<S> ys;
  const int j0 = 2 + tk.b * d.march, j1 = min(j0 + d.march, d.g.ny + 2);
  double cx = 0.0, cy = 0.0;
  if (d.ctl->nstep % 2 == 0) {
    step_march<S, ST1, false, true, FD>(d.g, d.ph, tr, dtdx, in, out, d.bl, d.br, d.bd, d.bu, tk.a,
                                        j0, j1, &ys, cx, cy);
  } else {
    step_march<S, ST1, true, false, FD>(d.g, d.ph, tr, dtdx, in, out, d.bl, d.br, d.bd, d.bu, tk.a,
                                        j0, j1, &ys, cx, cy);
    commit_courant_wave(cx, cy, d.cour, kInstSlots, blockIdx.x % kInstSlots);
  }
}

template <typename S, int FD>
static void launch_march_fd(const InstDev<S>* inst, const BTask* tasks, int ntask, int nst1,
                            hipStream_t st) {
  if (nst1 > 0)
    hipLaunchKernelGGL((k_batch_march<S, true, FD>), dim3(nst1), dim3(64), 0, st, inst, tasks);
  if (ntask > nst1)
    hipLaunchKernelGGL((k_batch_march<S, false, FD>), dim3(ntask - nst1), dim3(64), 0, st, inst,
                       tasks + nst1);
}
#endif
#ifdef HYDRO_FAST_UNIT
void launch_batch_march_fast(const InstDev<double>* inst, const BTask* tasks, int ntask, int nst1,
                             hipStream_t st) {
  launch_march_fd<double, kFast>(inst, tasks, ntask, nst1, st);
}
#endif
#ifdef HYDRO_MIXED_UNIT
void launch_batch_march(const InstDev<float>* inst, const BTask* tasks, int ntask, int nst1,
                        hipStream_t st) {
  launch_march_fd<float, kIeee>(inst, tasks, ntask, nst1, st);
}
#endif

// Ghost fills of the instances too narrow for the sweeps to form theirs
// (kind = direction): of (line, var) pairs [a, a + kBoundaryChunk)
// of one instance per task, from buffer `phase` into both buffers.
template <typename S>
__global__ __launch_bounds__(256) void k_batch_boundary(const InstDev<S>* inst,
                                                        const BTask* tasks, int phase) {
  const BTask tk = tasks[blockIdx.x];
  const InstDev<S>& d = inst[tk.inst];
  if (!d.ctl->active) return;
  const int idim = tk.kind;
  const int nl = (idim == 1) ? d.g.ny : d.g.nx;
  const GridView<S> src = d.buf[phase], dst = d.buf[1 - phase];
  const int kend = min(tk.a + kBoundaryChunk, 4 * nl);
  for (int k = tk.a + threadIdx.x; k < kend; k += blockDim.x) {
    const int line = k % nl, v = k / nl;
    boundary_line<S>(idim, d.g, d.bl, d.br, d.bd, d.bu, src.p[v], dst.p[v], v, line);
  }
}

// CFL maxima of the listed instances' states (admission / step 0).
template <typename S>
__global__ __launch_bounds__(256) void k_batch_courant(const InstDev<S>* inst, const int* ids,
                                                       int nids) {
  for (int t = blockIdx.x; t < nids * 64; t += gridDim.x) {
    const InstDev<S>& d = inst[ids[t / 64]];
    const int part = t % 64;
    const GridView<S> u = d.buf[state_buf(d)];
    const long n = (long) d.g.nx * d.g.ny;
    double cx = 0.0, cy = 0.0;
    for (long c = (long) part * blockDim.x + threadIdx.x; c < n; c += 64L * blockDim.x) {
      const long jj = c / d.g.nx, ii = c - jj * d.g.nx;
      const long o = (jj + 2) * d.g.pitch + ii + 2;
      S ax, ay;
      courant_cell<S>(u.p[0][o], u.p[1][o], u.p[2][o], u.p[3][o], d.ph, ax, ay);
      cx = maxm(cx, (double) ax);
      cy = maxm(cy, (double) ay);
    }
    commit_courant(cx, cy, d.cour, kInstSlots, part % kInstSlots);
  }
}

// main.c:297-298 and 244-260 for every listed instance, one wave each: closes
// the step that is open (so that only the last step of a run needs
// k_batch_ctl_end: one launch of 4.3 us a step less), opens the next.  A batch
// also stops an instance at its first dt that is not positive and finite
// (the reference would go on; this only differs for runs that have already
// broken down) and flags it, so one bad run cannot stall the others.
template <typename S>
__global__ __launch_bounds__(64) void k_batch_ctl_begin(const InstDev<S>* inst, const int* ids,
                                                        int nids) {
  for (int k = blockIdx.x; k < nids; k += gridDim.x) {
    const InstDev<S>& d = inst[ids[k]];
    RunCtl* c = d.ctl;
    const int open = c->active;
    const double t = open ? c->t + c->dt : c->t, tend = c->tend;
    const int nstep = c->nstep + (open ? 1 : 0), nstepmax = c->nstepmax;
    bool act = (t < tend) && (nstep < nstepmax) && !c->fault;
    bool bad = false;
    if (act && (nstep % 2) == 0) {
      double dt = wave_reduce_dt<kInstSlots>(d.cour, d.cf, d.dx, d.smallc);
      if (nstep == 0) dt = dt / 2.0;
      bad = !(dt > 0.0) || !__builtin_isfinite(dt);
      if (threadIdx.x == 0 && !bad) c->dt = dt;
    }
    if (threadIdx.x == 0) {
      c->t = t;
      c->nstep = nstep;
      if (bad) c->fault = 1;
      c->active = (act && !bad) ? 1 : 0;
    }
  }
}

// main.c:297-298 for the last step of a run
template <typename S>
__global__ void k_batch_ctl_end(const InstDev<S>* inst, const int* ids, int nids) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nids) return;
  RunCtl* c = inst[ids[k]].ctl;
  if (!c->active) return;
  c->nstep += 1;
  c->t += c->dt;
  c->active = 0;
}

[[maybe_unused]] static inline unsigned cdivu(long a, long b) {
  return (unsigned) ((a + b - 1) / b);
}

#ifdef HYDRO_BASE_UNIT
__global__ void k_batch_set_ctl(RunCtl* c, double t, double dt, double tend, int nstep,
                                int nstepmax, int active) {
  if (threadIdx.x != 0) return;
  c->t = t;
  c->dt = dt;
  c->tend = tend;
  c->nstep = nstep;
  c->nstepmax = nstepmax;
  c->active = active;
  c->log = nullptr;
  c->log_cap = 0;
  c->log_base = 0;
  c->fault = 0;
}

// The tasks of one list entry (an instance's share of a phase) per blockIdx.x.
__global__ __launch_bounds__(256) void k_batch_tasks(const BList* __restrict__ lists,
                                                     BTask* __restrict__ tasks) {
  const BList l = lists[blockIdx.x];
  for (int k = blockIdx.y * 256 + threadIdx.x; k < l.count; k += 256 * gridDim.y)
    tasks[l.first + k] = l.ncb > 0 ? BTask{l.inst, l.kind, k % l.ncb, k / l.ncb}
                                   : BTask{l.inst, l.kind, k * l.per, 0};
}

void launch_batch_tasks(const BList* lists, int n, BTask* tasks, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_batch_tasks, dim3(n, 8), dim3(256), 0, st, lists, tasks);
}

__global__ void k_fill_u64(uint64_t* p, long n) {
  for (long k = (long) blockIdx.x * blockDim.x + threadIdx.x; k < n;
       k += (long) gridDim.x * blockDim.x)
    p[k] = 0;
}

void launch_batch_set_ctl(RunCtl* c, double t, double dt, double tend, int nstep, int nstepmax,
                          int active, hipStream_t st) {
  hipLaunchKernelGGL(k_batch_set_ctl, dim3(1), dim3(64), 0, st, c, t, dt, tend, nstep, nstepmax,
                     active);
}

void launch_zero_u64(uint64_t* p, long n, hipStream_t st) {
  if (n <= 0) return;
  long nb = (n + 255) / 256;
  if (nb > 1024) nb = 1024;
  hipLaunchKernelGGL(k_fill_u64, dim3((unsigned) nb), dim3(256), 0, st, p, n);
}
#endif  // HYDRO_BASE_UNIT

// The arithmetic form of this unit's batched sweeps.
template <typename S>
constexpr int unit_form() {
#ifdef HYDRO_FAST_UNIT
  return kFast;
#else
  return sizeof(S) == 8 ? kGated : kIeee;
#endif
}

template <typename S, bool ST1, int FD>
static void launch_sweep_part(int kind, const InstDev<S>* inst, const BTask* tasks, int ntask,
                              int phase, bool ghosts, int waves, int xiter, hipStream_t st) {
  if (ntask <= 0) return;
  if (kind == 1)
    hipLaunchKernelGGL((k_batch_sweep_x<S, ST1, FD>), dim3(ntask), dim3(64 * waves), 0, st, inst,
                       tasks, phase, (int) ghosts, xiter);
  else
    hipLaunchKernelGGL((k_batch_sweep_y<S, ST1, FD>), dim3(ntask), dim3(64 * waves),
                       waves * sizeof(YStash<S>), st, inst, tasks, phase, (int) ghosts);
}

template <typename S, int FD>
static void launch_batch_sweep_fd(int kind, const InstDev<S>* inst, const BTask* tasks,
                                  int ntask, int nst1, int phase, bool ghosts, int waves,
                                  int xiter, hipStream_t st) {
  launch_sweep_part<S, true, FD>(kind, inst, tasks, nst1, phase, ghosts, waves, xiter, st);
  launch_sweep_part<S, false, FD>(kind, inst, tasks + nst1, ntask - nst1, phase, ghosts, waves,
                                  xiter, st);
}

#ifndef HYDRO_FAST_UNIT
template <typename S>
void launch_batch_sweep(int kind, const InstDev<S>* inst, const BTask* tasks, int ntask,
                        int nst1, int phase, bool ghosts, int waves, int xiter, hipStream_t st) {
  launch_batch_sweep_fd<S, unit_form<S>()>(kind, inst, tasks, ntask, nst1, phase, ghosts, waves,
                                           xiter, st);
}
#else
void launch_batch_sweep_fast(int kind, const InstDev<double>* inst, const BTask* tasks,
                             int ntask, int nst1, int phase, bool ghosts, int waves, int xiter,
                             hipStream_t st) {
  launch_batch_sweep_fd<double, kFast>(kind, inst, tasks, ntask, nst1, phase, ghosts, waves, xiter,
                                       st);
}
#endif

template <typename S>
void launch_batch_boundary(const InstDev<S>* inst, const BTask* tasks, int ntask, int phase,
                           hipStream_t st) {
  if (ntask <= 0) return;
  hipLaunchKernelGGL(k_batch_boundary<S>, dim3(ntask), dim3(256), 0, st, inst, tasks, phase);
}

template <typename S>
void launch_batch_courant(const InstDev<S>* inst, const int* ids, int nids, hipStream_t st) {
  if (nids <= 0) return;
  long nb = 64L * nids;
  if (nb > 4096) nb = 4096;
  hipLaunchKernelGGL(k_batch_courant<S>, dim3((unsigned) nb), dim3(256), 0, st, inst, ids, nids);
}

template <typename S>
void launch_batch_ctl(const InstDev<S>* inst, const int* ids, int nids, bool begin,
                      hipStream_t st) {
  if (nids <= 0) return;
  if (begin) {
    const int nb = nids < 1024 ? nids : 1024;
    hipLaunchKernelGGL(k_batch_ctl_begin<S>, dim3(nb), dim3(64), 0, st, inst, ids, nids);
  } else {
    hipLaunchKernelGGL(k_batch_ctl_end<S>, dim3(cdivu(nids, 256)), dim3(256), 0, st, inst, ids,
                       nids);
  }
}

#define INST_ARITH(S)                                                                            \
  template void launch_batch_sweep<S>(int, const InstDev<S>*, const BTask*, int, int, int, bool, \
                                      int, int, hipStream_t);                                    \
  template void launch_batch_courant<S>(const InstDev<S>*, const int*, int, hipStream_t);
#define INST_MOVE(S)                                                                             \
  template void launch_batch_boundary<S>(const InstDev<S>*, const BTask*, int, int, hipStream_t); \
  template void launch_batch_ctl<S>(const InstDev<S>*, const int*, int, bool, hipStream_t);
#if defined(HYDRO_BASE_UNIT)
INST_ARITH(double)
INST_MOVE(double)
INST_MOVE(float)
#elif defined(HYDRO_MIXED_UNIT)
INST_ARITH(float)
#endif
#undef INST_ARITH
#undef INST_MOVE

}  // namespace hydro
