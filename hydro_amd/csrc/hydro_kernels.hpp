// Internal (C++) interface between the C-ABI layer and the HIP kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// The kernel files (hydro_kernels.hip, hydro_batch.hip) are compiled once per
// arithmetic unit: HYDRO_MIXED_UNIT (FP32-storage sweeps), HYDRO_FAST_UNIT
// (FP64 fast-form sweeps) or neither (everything else, FP64 bitwise).
#if !defined(HYDRO_MIXED_UNIT) && !defined(HYDRO_FAST_UNIT)
#define HYDRO_BASE_UNIT 1
#endif

namespace hydro {

// Device-resident time-loop state (HydroC99_2DMpi/Src/main.c:244-298 moved
// onto the GPU so whole runs can be queued or graph-captured without host
// round trips).  A grid has two, one for its even steps and one for its odd
// ones, so that a sweep can read the open step's while one workgroup of it
// already writes the next step's.
struct RunCtl {
  double t, dt, tend;
  int nstep, nstepmax;
  int active;    // 1 while the current step runs (t < tend && nstep < nstepmax)
  int log_base;  // dt of step n goes to log[n - log_base] when in range
  int log_cap;
  int fault;     // batches: set when a computed dt was not positive and finite
  double* log;
};

// One grid as the kernels see it.  Element (i, j, v) of a state buffer lives
// at plane[v][j * pitch + i], i in [0, nx+4), j in [0, ny+4) (padded indices
// with two ghost layers, as in the reference).
template <typename S>
struct GridView {
  S* p[4];
};

struct GridGeom {
  int nx, ny;
  long pitch;
};

// The ghost cells of one sweep's direction: the boundary types of its low and
// high side (<= 0: the ghosts in memory), and where the ghost values go --
// 1 the buffer that the sweep reads, 2 the one it writes, 0 nowhere.
struct GhostFill {
  int lo, hi, to;
};

struct PhysArgs {
  double gamma, smallr, smallc, slope_type, courant_factor, dx;
  int niter, iorder, scheme;
  int bl, br, bd, bu;  // boundary types left/right/down/up
};

// Number of CFL max-slots (spread the atomics over many addresses).
constexpr int kCourSlots = 1024;
// x sweep: one 64-lane wave updates 60 cells of a row.
constexpr int kXSeg = 60;

// Narrowest grid whose ghosts' sources are all interior cells (but for the
// high-x source nx+2 of the absorbing type, which nothing rewrites), so that
// each ghost can be formed on its own.
constexpr int kGhostMin = 3;

struct SweepTune {
  int yseg;     // rows per y-sweep thread (column march length); 0: by the grid's size
  int ywaves;   // waves per y-sweep workgroup (1..4)
  int xwaves;   // waves per x-sweep workgroup (1..4); 0: by the grid's size
  int xiter;    // row segments each x-sweep wave walks; 0: by the grid's size
  int step;     // whole steps in one launch: a tile's rows (8, 16), or (fast and mixed
                // forms) kMarch + the rows of a march; 0: the two sweep kernels; -1: by
                // the grid's size
};
constexpr int kMarch = 32;
// Widest grid of the march (its lanes' offsets in a row are 32 bits of bytes).
constexpr int kMarchWidest = 1 << 28;
constexpr int kSimds = 1024;  // of the GPU: 256 CUs of 4

// ---- launchers (hydro_kernels.hip) -----------------------------------------
// Ghost cells: launch_sweep fills those of its direction itself (fill_ghosts
// says where to: 1 the input, 2 the output, 0 nowhere; -1: the ghosts are in
// memory already, put there by launch_boundary).  It may be asked to on grids
// of at least kGhostMin cells each way.
// dt handling: if ctl != nullptr the kernels read dt and the active flag from
// it; otherwise dt_val is used.  nxt (x sweeps that open an even step): the
// sweep also closes the step in *nxt, which becomes the odd step's control.
// cour (2*kCourSlots uint64, zeroed) receives
// the CFL maxima of the written state when non-null.
template <typename S>
void launch_boundary(int idim, const GridGeom& g, const PhysArgs& ph, GridView<S> src,
                     GridView<S> dst2, const RunCtl* ctl, hipStream_t st);

template <typename S>
void launch_sweep(int idim, const GridGeom& g, const PhysArgs& ph, GridView<S> in,
                  GridView<S> out, double dt_val, const RunCtl* ctl, RunCtl* nxt,
                  uint64_t* cour, const SweepTune& tune, int fill_ghosts, hipStream_t st);

// The FP64 fast form's sweeps (hydro_kernels.hip, fast unit): as
// launch_sweep, with the kFast arithmetic.
void launch_sweep_fast(int idim, const GridGeom& g, const PhysArgs& ph, GridView<double> in,
                       GridView<double> out, double dt_val, const RunCtl* ctl, RunCtl* nxt,
                       uint64_t* cour, const SweepTune& tune, int fill_ghosts, hipStream_t st);

// Both sweeps of a step in one launch, x first (idim 1) or y first (idim 2,
// which folds the CFL maxima when cour is non-null), from one state buffer
// into the other with every ghost cell formed and stored; the rest as
// launch_sweep.  rows: SweepTune::step, positive (tiles of 8 rows, in the mixed
// form or 16; marches in the fast and mixed forms).  For grids of at least
// kGhostMin cells each way.
template <typename S>
void launch_step(int idim, const GridGeom& g, const PhysArgs& ph, GridView<S> in, GridView<S> out,
                 double dt_val, const RunCtl* ctl, RunCtl* nxt, uint64_t* cour, int rows,
                 hipStream_t st);
void launch_step_fast(int idim, const GridGeom& g, const PhysArgs& ph, GridView<double> in,
                      GridView<double> out, double dt_val, const RunCtl* ctl, RunCtl* nxt,
                      uint64_t* cour, int rows, hipStream_t st);

template <typename S>
void launch_courant(const GridGeom& g, const PhysArgs& ph, GridView<S> in, uint64_t* cour,
                    const RunCtl* ctl, hipStream_t st);

// dt_finalize reduces the CFL slots (clearing them) into
// dt = cfl*dx / max(cx, cy, smallc) at *dt_out.  The device time loop's
// control, ctl[0] for even steps and ctl[1] for odd ones: ctl_begin closes the
// odd step before (if one is open) and opens an even step, active = (t < tend
// && nstep < nstepmax), dt from the slots (halved at step 0); the even step's
// x sweep closes it and opens the odd one (launch_sweep's nxt); ctl_end closes
// the last step of a run and leaves the outcome in ctl[0].  Closing a step
// logs dt and advances nstep and t.
void launch_dt_finalize(uint64_t* cour, double cf, double dx, double smallc, double* dt_out,
                        hipStream_t st);
void launch_ctl_begin(RunCtl* ctl, uint64_t* cour, double cf, double dx, double smallc,
                      hipStream_t st);
void launch_ctl_end(RunCtl* ctl, bool odd, hipStream_t st);
void launch_clear_slots(uint64_t* cour, hipStream_t st);

// Initial state (hydro_funcs.c:79-146): interior rho=1, u=v=0, E=1e-5, ghosts
// 0, then E=e_blast at padded cells (bx, by) for by in [by0, by1).  Fills
// both buffers when b is non-null.
template <typename S>
void launch_init(const GridGeom& g, GridView<S> a, GridView<S> b, int bx, int by0, int by1,
                 double e_blast, hipStream_t st);

void launch_copy_probe(const double* a, double* b, long n, hipStream_t st);
struct StreamProbe4 {
  const double* in[4];
  double* out[4];
};
void launch_stream_probe(const StreamProbe4& p, long n, hipStream_t st);

// Density image (hydro_image.hip): clears *key, reduces the maximum density
// of the padded plane `rho` into it, then writes w*h RGB pixels (3 bytes
// each, row cy = 0 first) sampled every `shrink` interior cells.
template <typename S>
void launch_image(const GridGeom& g, const S* rho, int shrink, int w, int h,
                  unsigned long long* key, unsigned char* rgb, hipStream_t st);

// Pitched device rows -> contiguous host rows through pinned staging buffers
// (hydro_stage.cpp); dst_esz == src_esz, or 8 with src_esz == 4 (widening).
int stage_d2h(void* dst, int dst_esz, const void* src, int src_esz, long src_pitch, long width,
              long rows, hipStream_t st);
// Contiguous host rows -> pitched device rows; dst_esz == src_esz, or 4 with
// src_esz == 8 (rounding).
int stage_h2d(void* dst, int dst_esz, long dst_pitch, const void* src, int src_esz, long width,
              long rows, hipStream_t st);
// Host memory to host memory, converting (4 <-> 8 bytes an element).
void host_copy(void* dst, int dst_esz, const void* src, int src_esz, size_t n);

}  // namespace hydro
