// HIP kernels for gfx950 (MI355X), one grid per launch: fused x / y sweeps of
// HydroC99's split Godunov/MUSCL step, ghost fill, CFL reduction, initial
// state and the device-side time-loop control.  The per-task bodies live in
// hydro_sweeps.hpp (shared with the batched kernels).
//
// The file is compiled three times.  The FP64 unit (the default,
// HYDRO_BASE_UNIT) holds everything except the FP32-storage and FP64 fast
// sweeps and is built with -ffp-contract=off, so the FP64 path is op-for-op
// the reference's.  The mixed-precision unit (HYDRO_MIXED_UNIT) holds only
// the FP32-storage sweeps and CFL kernels, and the fast unit
// (HYDRO_FAST_UNIT) only the FP64 fast-form sweeps; both are built with
// -ffp-contract=on: those forms carry no bitwise contract with the
// reference, and multiply-adds fused within each source expression cut their
// VALU instruction counts while keeping the single-grid and batched kernels
// (same source) bit-identical.
#include "hydro_kernels.hpp"
#include "hydro_sweeps.hpp"

namespace hydro {

// ---- run control ---------------------------------------------------------------

// main.c:297-298: the step of c is done (if it ran at all).  Called by one thread.
__device__ __forceinline__ void close_step(RunCtl& c) {
  if (!c.active) return;
  const int k = c.nstep - c.log_base;
  if (c.log && k >= 0 && k < c.log_cap) c.log[k] = c.dt;
  c.nstep += 1;
  c.t += c.dt;
  c.active = 0;
}

// The even step's x sweep, workgroup 0: the odd step that follows takes the
// same dt, so its control is known before the step has run.  Nothing reads
// *nxt in this launch.  (In a kernel of their own, closing a step and opening
// the next one took 4.3 + 4.5 us a step, 2 x 5 launches in the two-step graph
// beside its sweeps; now 1 launch.)
__device__ __forceinline__ void open_odd_step(const RunCtl* ctl, RunCtl* nxt) {
  if (!nxt || blockIdx.x != 0 || threadIdx.x != 0) return;
  RunCtl c = *ctl;
  if (c.active) {
    close_step(c);
    c.active = (c.t < c.tend) && (c.nstep < c.nstepmax);
  }
  *nxt = c;
}

// ---- x sweep ---------------------------------------------------------------

// A workgroup walks wpb * xiter consecutive row segments, wpb at a time.
template <typename S, bool ST1, bool COUR, int FD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) void k_sweep_x(GridGeom g, Phys<S> ph, double dx,
                                                 double dt_val, const RunCtl* ctl,
                                                 RunCtl* nxt, GridView<S> in, GridView<S> out,
                                                 GhostFill gf, uint64_t* cour, int nseg, int xiter) {
  double dt = dt_val;
  if (ctl) {
    open_odd_step(ctl, nxt);
    if (!ctl->active) return;  // grid-uniform
    dt = ctl->dt;
  }
  const double dtdx = dt / dx;  // hydro_godunov.c:101
  const TraceK<S> tk = make_tracek<S>((S) dtdx, ph.scheme);
  const int wpb = blockDim.x >> 6;
  double cx = 0.0, cy = 0.0;
  // segments (blockIdx.x * xiter + it) * wpb + wave, it = 0 .. xiter-1
  SegWalk w((int) blockIdx.x * xiter * wpb + wave_id(), nseg);
  for (int it = 0; it < xiter && w.row < g.ny; it++) {
    x_segment<S, ST1, COUR, FD>(g, ph, tk, dtdx, in, out, gf, w.row, w.seg, cx, cy);
    w.advance(wpb, nseg);
  }
  if (COUR) commit_courant(cx, cy, cour, kCourSlots, blockIdx.x % kCourSlots);
}

// Workgroup form (W = 2 or 4 waves): a workgroup walks xiter consecutive
// row pieces of 64*W - 4 updated cells, neighbours through LDS (x_blocks).
template <typename S, bool ST1, bool COUR, int W, int FD>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(5))) void k_sweep_xb(GridGeom g, Phys<S> ph, double dx,
                                                     double dt_val, const RunCtl* ctl,
                                                     RunCtl* nxt, GridView<S> in,
                                                     GridView<S> out, GhostFill gf, uint64_t* cour, int nseg,
                                                     int xiter) {
  __shared__ XLds<S, W> sh;
  double dt = dt_val;
  if (ctl) {
    open_odd_step(ctl, nxt);
    if (!ctl->active) return;  // grid-uniform
    dt = ctl->dt;
  }
  const double dtdx = dt / dx;  // hydro_godunov.c:101
  const TraceK<S> tk = make_tracek<S>((S) dtdx, ph.scheme);
  double cx = 0.0, cy = 0.0;
  x_blocks<S, ST1, COUR, W, FD>(g, ph, tk, dtdx, in, out, gf, (int) blockIdx.x * xiter, xiter,
                                nseg, sh, cx, cy);
  if (COUR) commit_courant(cx, cy, cour, kCourSlots, blockIdx.x % kCourSlots);
}

// ---- y sweep ---------------------------------------------------------------

// A workgroup covers 64 columns; its waves take consecutive row segments of
// yseg rows each.
template <typename S, bool ST1, bool COUR, int FD>
__global__ __launch_bounds__(256) void k_sweep_y(GridGeom g, Phys<S> ph, double dx,
                                                 double dt_val, const RunCtl* ctl,
                                                 GridView<S> in, GridView<S> out, GhostFill gf,
                                                 uint64_t* cour, int yseg, int ncolblk) {
  double dt = dt_val;
  if (ctl) {
    if (!ctl->active) return;
    dt = ctl->dt;
  }
  const double dtdx = dt / dx;
  const TraceK<S> tk = make_tracek<S>((S) dtdx, ph.scheme);
  const int cb = blockIdx.x % ncolblk;
  const int sgi = (blockIdx.x / ncolblk) * (blockDim.x >> 6) + wave_id();
  const int col = cb * 64 + (threadIdx.x & 63);
  const bool colok = col < g.nx;
  const long i = 2 + (colok ? col : g.nx - 1);
  const int j0 = 2 + sgi * yseg;
  double cx = 0.0, cy = 0.0;
  if (j0 < g.ny + 2) {  // wave-uniform
    const int j1 = min(j0 + yseg, g.ny + 2);  // rows [j0, j1) are updated
    extern __shared__ __attribute__((aligned(16))) unsigned char ylds[];
    YStash<S>* ys = reinterpret_cast<YStash<S>*>(ylds) + wave_id();
    y_march<S, ST1, COUR, FD>(g, ph, tk, dtdx, in, out, gf, colok, i, j0, j1, ys, cx, cy);
  }
  if (COUR) commit_courant(cx, cy, cour, kCourSlots, blockIdx.x % kCourSlots);
}

// ---- whole step ----------------------------------------------------------------

// Both sweeps of one tile per workgroup (tile_step), from one state buffer
// into the other.
template <typename S, bool ST1, bool XY, int W, int FD>
__global__ __launch_bounds__(64 * W) void k_step(GridGeom g, Phys<S> ph, double dx,
                                                 double dt_val, const RunCtl* ctl, RunCtl* nxt,
                                                 GridView<S> in, GridView<S> out, int bl, int br,
                                                 int bd, int bu, uint64_t* cour, int nct) {
  __shared__ TileLds<S, W> sh;
  const int w = wave_id(), lane = threadIdx.x & 63;
  // (the cells' loads are on their way before the control is read)
  const TPlace<S> p = tile_load<S>(g, in, bl, br, bd, bu, 60 * (blockIdx.x % nct) + lane,
                                   (W - 4) * (blockIdx.x / nct) + w);
  double dt = dt_val;
  if (ctl) {
    open_odd_step(ctl, nxt);
    if (!ctl->active) return;  // grid-uniform
    dt = ctl->dt;
  }
  const double dtdx = dt / dx;
  const TraceK<S> tk = make_tracek<S>((S) dtdx, ph.scheme);
  double cx = 0.0, cy = 0.0;
  // (odd steps, y first, fold the CFL maxima that the next step's dt needs)
  tile_step<S, ST1, !XY, XY, W, FD>(g, ph, tk, dtdx, p, out, w, lane, sh, cx, cy);
  if (!XY && cour) commit_courant(cx, cy, cour, kCourSlots, blockIdx.x % kCourSlots);
}

#if defined(HYDRO_FAST_UNIT) || defined(HYDRO_MIXED_UNIT)
// Both sweeps of a large grid's step, one wave a workgroup (step_march): built for
// the waves that the march's LDS slots leave room for, 4 a SIMD, in FP32 5.
template <typename S, bool ST1, bool XY, int FD>
__global__ __launch_bounds__(64) __attribute__((
    amdgpu_waves_per_eu(sizeof(S) == 4 ? 5 : 4))) void k_step_march(GridGeom g, Phys<S> ph,
                                                                    double dx, double dt_val,
                                                                    const RunCtl* ctl, RunCtl* nxt,
                                                                    GridView<S> in,
                                                                    GridView<S> out, int bl,
                                                                    int br, int bd, int bu,
                                                                    uint64_t* cour, int nct,
                                                                    int len) {
  double dt = dt_val;
  if (ctl) {
    open_odd_step(ctl, nxt);
    if (!ctl->active) return;  // grid-uniform
    dt = ctl->dt;
  }
  const double dtdx = dt / dx;
  const TraceK<S> tk = make_tracek<S>((S) dtdx, ph.scheme);
  __shared__ YStash<S> ys;
  const int j0 = 2 + (blockIdx.x / nct) * len, j1 = min(j0 + len, g.ny + 2);
  double cx = 0.0, cy = 0.0;
  step_march<S, ST1, !XY, XY, FD>(g, ph, tk, dtdx, in, out, bl, br, bd, bu, blockIdx.x % nct, j0,
                                  j1, &ys, cx, cy);
  if (!XY && cour) commit_courant_wave(cx, cy, cour, kCourSlots, blockIdx.x % kCourSlots);
}
#endif

// ---- standalone CFL maximum -------------------------------------------------

// CFL maxima over a thread's cells: a wave takes 64 columns of a row, the
// workgroup's waves consecutive rows, from row blockIdx.y * 4 + wave in strides
// of 4 * gridDim.y (by rows and columns: with one running cell index a 64-bit
// division per cell cost as much as the cell's arithmetic).
template <typename S>
__device__ __forceinline__ void courant_cells(const GridGeom& g, const Phys<S>& ph,
                                              const GridView<S>& in, double& cx, double& cy) {
  const int i = (int) blockIdx.x * 64 + (threadIdx.x & 63);
  if (i >= g.nx) return;
  const int step = 4 * gridDim.y;
  for (int j = (int) blockIdx.y * 4 + wave_id(); j < g.ny; j += step) {
    const long o = (j + 2L) * g.pitch + i + 2;
    S ax, ay;
    courant_cell<S>(in.p[0][o], in.p[1][o], in.p[2][o], in.p[3][o], ph, ax, ay);
    cx = maxm(cx, (double) ax);
    cy = maxm(cy, (double) ay);
  }
}

template <typename S>
__global__ __launch_bounds__(256) void k_courant(GridGeom g, Phys<S> ph, GridView<S> in,
                                                 uint64_t* cour, const RunCtl* ctl) {
  if (ctl && !ctl->active) return;
  double cx = 0.0, cy = 0.0;
  courant_cells<S>(g, ph, in, cx, cy);
  commit_courant(cx, cy, cour, kCourSlots,
                 (blockIdx.y * gridDim.x + blockIdx.x) % kCourSlots);
}

// ---- ghost cells -------------------------------------------------------------

// One thread per (line, variable); see boundary_line.
template <typename S>
__global__ __launch_bounds__(256) void k_boundary(int idim, GridGeom g, int bl, int br, int bd,
                                                  int bu, GridView<S> src, GridView<S> dst2,
                                                  int has_dst2, const RunCtl* ctl) {
  if (ctl && !ctl->active) return;
  const int nl = (idim == 1) ? g.ny : g.nx;
  const long t = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 4L * nl) return;
  const int k = (int) (t % nl);
  const int v = (int) (t / nl);
  boundary_line<S>(idim, g, bl, br, bd, bu, src.p[v], has_dst2 ? dst2.p[v] : nullptr, v, k);
}

#ifdef HYDRO_BASE_UNIT
// ---- dt and run control ------------------------------------------------------

__global__ __launch_bounds__(64) void k_dt_finalize(uint64_t* cour, double cf, double dx,
                                                    double smallc, double* dt_out) {
  const double dt = wave_reduce_dt<kCourSlots>(cour, cf, dx, smallc);
  if (threadIdx.x == 0) *dt_out = dt;
}

// main.c:244-260: open an even step (ctl[0]), after closing the odd one before
// it if that is open (ctl[1], which holds the run's latest state either way).
__global__ __launch_bounds__(64) void k_ctl_begin(RunCtl* ctl, uint64_t* cour, double cf,
                                                  double dx, double smallc) {
  RunCtl c = ctl[1];
  if (threadIdx.x != 0) c.log = nullptr;  // one thread logs
  close_step(c);
  if ((c.t < c.tend) && (c.nstep < c.nstepmax)) {  // wave-uniform
    c.dt = wave_reduce_dt<kCourSlots>(cour, cf, dx, smallc);
    if (c.nstep == 0) c.dt = c.dt / 2.0;
    c.active = 1;
  }
  if (threadIdx.x == 0) ctl[0] = c;
}

// The run's last step was odd (open in ctl[1]) or even (closed by its x sweep,
// an odd step opened in ctl[1] that will not run now): the outcome to ctl[0].
__global__ void k_ctl_end(RunCtl* ctl, int odd) {
  if (threadIdx.x != 0) return;
  RunCtl c = ctl[1];
  if (odd) close_step(c);
  c.active = 0;
  ctl[0] = c;
  ctl[1].active = 0;
}

__global__ void k_clear_slots(uint64_t* cour) {
  for (int s = threadIdx.x; s < 2 * kCourSlots; s += blockDim.x) cour[s] = 0;
}
#endif  // HYDRO_BASE_UNIT

template <typename S>
__global__ __launch_bounds__(256) void k_init(GridGeom g, GridView<S> a, GridView<S> b, int bx,
                                              int by0, int by1, S eb) {
  const long t = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long) (g.nx + 4) * (g.ny + 4)) return;
  init_cell<S>(g, a, b, t, bx, by0, by1, eb);
}

#ifdef HYDRO_BASE_UNIT
// ---- plain copy (measurement reference) ---------------------------------------

// Streams n doubles from a to b; used to calibrate HBM byte counters and as
// the achievable-copy-bandwidth reference.
__global__ __launch_bounds__(256) void k_copy_probe(const double* __restrict__ a,
                                                    double* __restrict__ b, long n) {
  for (long k = (long) blockIdx.x * blockDim.x + threadIdx.x; k < n;
       k += (long) gridDim.x * blockDim.x)
    b[k] = a[k];
}

void launch_copy_probe(const double* a, double* b, long n, hipStream_t st) {
  hipLaunchKernelGGL(k_copy_probe, dim3(8192), dim3(256), 0, st, a, b, n);
}

// The sweeps' access shape as a plain copy: four arrays of n doubles in, four
// out, one cell per thread, non-temporal loads and stores (the fastest such
// copy measured: 5.7-6.2 TB/s on MI355X for 8196^2 cells, 5.5 TB/s without
// the hints).  Its rate is the bandwidth of the sweeps' bytes with no
// arithmetic and a linear access pattern.
__global__ __launch_bounds__(256) void k_stream_probe(StreamProbe4 p, long n) {
  const long i = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double v[4];
#pragma unroll
  for (int k = 0; k < 4; k++) v[k] = __builtin_nontemporal_load(&p.in[k][i]);
#pragma unroll
  for (int k = 0; k < 4; k++) __builtin_nontemporal_store(v[k], &p.out[k][i]);
}

void launch_stream_probe(const StreamProbe4& p, long n, hipStream_t st) {
  hipLaunchKernelGGL(k_stream_probe, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, st, p, n);
}
#endif  // HYDRO_BASE_UNIT

// ---- launchers -----------------------------------------------------------------

static inline unsigned cdiv(long a, long b) { return (unsigned) ((a + b - 1) / b); }

template <typename S>
void launch_boundary(int idim, const GridGeom& g, const PhysArgs& ph, GridView<S> src,
                     GridView<S> dst2, const RunCtl* ctl, hipStream_t st) {
  const int nl = (idim == 1) ? g.ny : g.nx;
  const long n = 4L * nl;
  const int has2 = dst2.p[0] != nullptr;
  hipLaunchKernelGGL(k_boundary<S>, dim3(cdiv(n, 256)), dim3(256), 0, st, idim, g, ph.bl, ph.br,
                     ph.bd, ph.bu, src, dst2, has2, ctl);
}

// Rows each y-sweep wave marches when the caller has not said.  A wave of n
// rows starts with work worth about one more row (four rows' loads and
// primitives, one flux), so long segments waste less; but the launch lasts as
// long as its longest wave, and a wave's rows follow one another, so short
// ones end earlier and spread more evenly.  With W = column blocks x rows wave
// rows on a fixed number of SIMDs the two costs, W / n and n, balance at n
// proportional to sqrt(W); the measured best lengths lie at sqrt(W) / 32 from
// 250x125 (1 row) to 8192x8192 (32).  Time of a step, FP64 / fast / mixed
// forms, against the 64 rows (16 on small grids) that every size took before:
// 250x125 34 / 28 / 25 us against 85 / 52 / 46; 1021x767 84 / 57 / 46 against
// 108 / 71 / 59; 4099x3001 595 / 376 / 227 against 653 / 382 / 263.  Past
// `most` rows nothing is won: 8192x8192, fast form, 1.81-1.83 ms at 32 rows,
// 1.83-1.85 at 64; 16384x12000, FP64 form, 8.13 at 32, 8.09 at 64, 8.16 at 128.
static int y_rows(long ncolblk, long ny, int most) {
  int n = 1;
  while (n < most && 1024L * (n + 1) * (n + 1) <= ncolblk * ny) n++;
  const long nseg = cdiv(ny, n);  // even segments: none ends the launch alone
  return (int) cdiv(ny, nseg);
}

// The x sweep's form and the row pieces that a workgroup walks, when the caller
// has not said.  The one-wave form (64-cell pieces) is the faster one in FP64
// at every size (8192x8192: 1.45 against 1.48 ms a sweep, 2048x1536: 200
// against 212 us a step) and in the other forms on small and middle grids
// (2048x1536: fast 119 against 123 us a step, mixed 85 against 88; 1021x767:
// 68 / 71, 57 / 59; these and the four-wave form's figures are of two sweeps a
// step, which such sizes take in a profile, with a given shape or in the mixed
// form below its line in default_step); the four-wave form, with fewer halo cells, where there are
// enough of its pieces to fill the GPU many times over (8192x1024, 33800
// pieces: 285 / 288; 8192x8192 1.83 / 1.88 ms).  The number of pieces goes by
// the square root, as y_rows; the best measured, one wave: 1 at 1021x767, 3 at
// 2048x1536, 4 at 4099x3001, 8-16 at 8192x8192, 16-32 at 16384x12000; four
// waves: 6 at 8192x1024, 6-8 at 4099x3001 and 8192x8192, 16-32 at 16384x12000.
template <typename S, int FD>
static int x_waves(const GridGeom& g) {
  if (sizeof(S) == 8 && FD != kFast) return 1;
  return (long) cdiv(g.nx, 64 * 4 - 4) * g.ny >= 24000 ? 4 : 1;
}
static int x_pieces(long n, int by, int most) {
  int k = 1;
  while (k < most && (long) by * by * (k + 1) * (k + 1) <= n) k++;
  return k;
}

// The sweep launch for one arithmetic form FD (shapes as in launch_sweep).
template <typename S, int FD>
static void launch_sweep_fd(int idim, const GridGeom& g, const Phys<S>& ph, double dx,
                            GridView<S> in, GridView<S> out, const GhostFill& gf, double dt_val,
                            const RunCtl* ctl, RunCtl* nxt, uint64_t* cour,
                            const SweepTune& tune, bool st1, hipStream_t st) {
  const bool c = cour != nullptr;
#define DISPATCH(F)                         \
  do {                                      \
    if (st1) {                              \
      if (c) F(true, true); else F(true, false);    \
    } else {                                \
      if (c) F(false, true); else F(false, false);  \
    }                                       \
  } while (0)
  int xwaves = tune.xwaves;
  if (xwaves <= 0) xwaves = x_waves<S, FD>(g);
  if (idim == 1 && (xwaves == 2 || xwaves == 4)) {
    const int W = xwaves;
    const int nseg = (int) cdiv(g.nx, 64 * W - 4);
    const long pieces = (long) nseg * g.ny;
    int xiter = tune.xiter;
    if (xiter <= 0) xiter = x_pieces(pieces, 32, 16);
    else while (xiter > 1 && cdiv(pieces, xiter) < 1024) xiter >>= 1;
    const dim3 grid(cdiv(pieces, xiter)), blk(64 * W);
#define HXB(A, B, WW) \
  hipLaunchKernelGGL((k_sweep_xb<S, A, B, WW, FD>), grid, blk, 0, st, g, ph, dx, dt_val, ctl, \
                     nxt, in, out, gf, cour, nseg, xiter)
#define HXW(A, B) do { if (W == 2) HXB(A, B, 2); else HXB(A, B, 4); } while (0)
    DISPATCH(HXW);
#undef HXW
#undef HXB
  } else if (idim == 1) {
    const int nseg = (int) cdiv(g.nx, kXSeg);
    const long waves = (long) nseg * g.ny;
    const int xw = xwaves;
    int xiter = tune.xiter;
    if (xiter <= 0) xiter = x_pieces(waves, 100, 32);
    // (given: keep at least ~4 workgroups per CU before walking several segments)
    else while (xiter > 1 && cdiv(waves, (long) xw * xiter) < 1024) xiter >>= 1;
    const dim3 grid(cdiv(waves, (long) xw * xiter)), blk(64 * xw);
#define HX(A, B) \
  hipLaunchKernelGGL((k_sweep_x<S, A, B, FD>), grid, blk, 0, st, g, ph, dx, dt_val, ctl, nxt, \
                     in, out, gf, cour, nseg, xiter)
    DISPATCH(HX);
#undef HX
  } else {
    const int yw = tune.ywaves > 0 ? tune.ywaves : 1;
    const int ncolblk = (int) cdiv(g.nx, 64);
    int yseg = tune.yseg;
    if (yseg <= 0) {
      yseg = y_rows(ncolblk, g.ny, FD == kFast ? 32 : 64);
    } else {
      // a given length: shortened (down to 16 rows) until there are about two
      // waves per SIMD, rather than leave most of the GPU idle
      while (yseg > 16 && (long) ncolblk * cdiv(g.ny, yseg) < 2048) yseg >>= 1;
    }
    const int nsg = (int) cdiv(g.ny, (long) yseg * yw);
#define HY(A, B)                                                                             \
  hipLaunchKernelGGL((k_sweep_y<S, A, B, FD>), dim3((unsigned) ncolblk * nsg), dim3(64 * yw), \
                     yw * sizeof(YStash<S>), st, g, ph, dx, dt_val, ctl, in, out, gf, cour,    \
                     yseg, ncolblk)
    DISPATCH(HY);
#undef HY
  }
#undef DISPATCH
}

// The whole-step launch for one arithmetic form (see launch_step).
template <typename S, int FD>
static void launch_step_fd(bool xy, const GridGeom& g, const Phys<S>& ph, const PhysArgs& pa,
                           GridView<S> in, GridView<S> out, double dt_val, const RunCtl* ctl,
                           RunCtl* nxt, uint64_t* cour, int rows, hipStream_t st) {
  const bool st1 = pa.slope_type == 1.0;
  const int nct = (int) cdiv(g.nx, 60);
#if defined(HYDRO_FAST_UNIT) || defined(HYDRO_MIXED_UNIT)
  if (rows > kMarch) {
    const int nseg = (int) cdiv(g.ny, rows - kMarch), len = (int) cdiv(g.ny, nseg);
#define HM(A, B)                                                                               \
  hipLaunchKernelGGL((k_step_march<S, A, B, FD>), dim3((unsigned) nct * cdiv(g.ny, len)),      \
                     dim3(64), 0, st, g, ph, pa.dx, dt_val, ctl, nxt, in, out, pa.bl, pa.br,   \
                     pa.bd, pa.bu, cour, nct, len)
    if (st1) {
      if (xy) HM(true, true); else HM(true, false);
    } else {
      if (xy) HM(false, true); else HM(false, false);
    }
#undef HM
    return;
  }
#endif
#define HS(A, B, W)                                                                              \
  hipLaunchKernelGGL((k_step<S, A, B, W, FD>), dim3((unsigned) nct * cdiv(g.ny, W - 4)),         \
                     dim3(64 * W), 0, st, g, ph, pa.dx, dt_val, ctl, nxt, in, out, pa.bl, pa.br, \
                     pa.bd, pa.bu, cour, nct)
#define HSW(A, B)                                             \
  do {                                                        \
    if constexpr (sizeof(S) == 4) {                           \
      if (rows == 16) HS(A, B, 16); else HS(A, B, 8);         \
    } else {                                                  \
      HS(A, B, 8);                                            \
    }                                                         \
  } while (0)
  if (st1) {
    if (xy) HSW(true, true); else HSW(true, false);
  } else {
    if (xy) HSW(false, true); else HSW(false, false);
  }
#undef HSW
#undef HS
}

// The ghosts of one sweep: formed by it (fill 0..2, see GhostFill::to), or in
// memory already (fill < 0).
static GhostFill ghost_fill(int idim, const PhysArgs& pa, int fill) {
  if (fill < 0) return GhostFill{0, 0, 0};
  return idim == 1 ? GhostFill{pa.bl, pa.br, fill} : GhostFill{pa.bd, pa.bu, fill};
}

#ifndef HYDRO_FAST_UNIT
template <typename S>
void launch_sweep(int idim, const GridGeom& g, const PhysArgs& pa, GridView<S> in,
                  GridView<S> out, double dt_val, const RunCtl* ctl, RunCtl* nxt,
                  uint64_t* cour, const SweepTune& tune, int fill, hipStream_t st) {
  const GhostFill gf = ghost_fill(idim, pa, fill);
  const Phys<S> ph = make_phys<S>(pa.gamma, pa.smallr, pa.smallc, pa.slope_type, pa.niter,
                                  pa.iorder, pa.scheme);
  const bool st1 = pa.slope_type == 1.0;
  // The range-gated FP64 divisions (the kGated kernels) pay when the launch
  // keeps the SIMDs busy.  A sweep of a small grid has too few waves for
  // that: each wave's march is latency-bound, and the gates' wave-wide
  // tests, branches and larger code lengthen it, so such launches run the
  // kIeee kernels (the results are the same bits either way).  A step of a flow
  // that moves everywhere (of a blast), every sweep gated / every sweep IEEE:
  // 250x125 22.1 / 21.6 us (26.9 / 23.7), 500x500 45.8 / 49.3 (41.2 / 40.7), 777x600
  // 59.9 / 66.9 (52.2 / 52.2), 1531x1200 151 / 167 (122 / 126), 2048x1536 232 / 265
  // (178 / 188); x gated and y IEEE, as the line has it, 777x600 62.4 (51.8),
  // 1021x767 (4096 y waves) 82.9 (67.4) against 80.6 (67.7) all gated: a lower line
  // would gain 3 % on moving flows there and lose 1 % on blasts.
  constexpr long kFastDivWaves = 4096;  // 4 waves per SIMD on 256 CUs
  if constexpr (sizeof(S) == 8) {
    const long ncb = cdiv(g.nx, 64);
    const long rows = tune.yseg > 0 ? 16 : y_rows(ncb, g.ny, 64);
    const bool fd = ph.fastdiv && (idim == 1 ? (long) cdiv(g.nx, kXSeg) * g.ny >= kFastDivWaves
                                             : ncb * cdiv(g.ny, rows) > kFastDivWaves);
    if (fd)
      launch_sweep_fd<S, kGated>(idim, g, ph, pa.dx, in, out, gf, dt_val, ctl, nxt, cour, tune,
                                 st1, st);
    else
      launch_sweep_fd<S, kIeee>(idim, g, ph, pa.dx, in, out, gf, dt_val, ctl, nxt, cour, tune,
                                 st1, st);
  } else {
    launch_sweep_fd<S, kIeee>(idim, g, ph, pa.dx, in, out, gf, dt_val, ctl, nxt, cour, tune,
                                 st1, st);
  }
}

template <typename S>
void launch_step(int idim, const GridGeom& g, const PhysArgs& pa, GridView<S> in, GridView<S> out,
                 double dt_val, const RunCtl* ctl, RunCtl* nxt, uint64_t* cour, int rows,
                 hipStream_t st) {
  const Phys<S> ph = make_phys<S>(pa.gamma, pa.smallr, pa.smallc, pa.slope_type, pa.niter,
                                  pa.iorder, pa.scheme);
  // (FP64: the IEEE code, as in every launch that does not fill the SIMDs)
  launch_step_fd<S, kIeee>(idim == 1, g, ph, pa, in, out, dt_val, ctl, nxt, cour, rows, st);
}
#else
void launch_step_fast(int idim, const GridGeom& g, const PhysArgs& pa, GridView<double> in,
                      GridView<double> out, double dt_val, const RunCtl* ctl, RunCtl* nxt,
                      uint64_t* cour, int rows, hipStream_t st) {
  const Phys<double> ph = make_phys<double>(pa.gamma, pa.smallr, pa.smallc, pa.slope_type,
                                            pa.niter, pa.iorder, pa.scheme);
  launch_step_fd<double, kFast>(idim == 1, g, ph, pa, in, out, dt_val, ctl, nxt, cour, rows, st);
}

void launch_sweep_fast(int idim, const GridGeom& g, const PhysArgs& pa, GridView<double> in,
                       GridView<double> out, double dt_val, const RunCtl* ctl, RunCtl* nxt,
                       uint64_t* cour, const SweepTune& tune, int fill, hipStream_t st) {
  const Phys<double> ph = make_phys<double>(pa.gamma, pa.smallr, pa.smallc, pa.slope_type,
                                            pa.niter, pa.iorder, pa.scheme);
  launch_sweep_fd<double, kFast>(idim, g, ph, pa.dx, in, out, ghost_fill(idim, pa, fill), dt_val,
                                 ctl, nxt, cour, tune, pa.slope_type == 1.0, st);
}
#endif

// Workgroups of a CFL pass: 64 columns x 4 rows each, the rows strided over at
// most about 2048 of them (8 waves a SIMD).
[[maybe_unused]] static dim3 courant_grid(const GridGeom& g) {
  const unsigned ncb = cdiv(g.nx, 64);
  const unsigned rows = cdiv(g.ny, 4), most = ncb < 2048 ? 2048 / ncb : 1;
  return dim3(ncb, rows < most ? rows : most);
}

template <typename S>
void launch_courant(const GridGeom& g, const PhysArgs& pa, GridView<S> in, uint64_t* cour,
                    const RunCtl* ctl, hipStream_t st) {
  const Phys<S> ph = make_phys<S>(pa.gamma, pa.smallr, pa.smallc, pa.slope_type, pa.niter,
                                  pa.iorder, pa.scheme);
  hipLaunchKernelGGL(k_courant<S>, courant_grid(g), dim3(256), 0, st, g, ph, in, cour, ctl);
}

#ifdef HYDRO_BASE_UNIT
void launch_dt_finalize(uint64_t* cour, double cf, double dx, double smallc, double* dt_out,
                        hipStream_t st) {
  hipLaunchKernelGGL(k_dt_finalize, dim3(1), dim3(64), 0, st, cour, cf, dx, smallc, dt_out);
}

void launch_ctl_begin(RunCtl* ctl, uint64_t* cour, double cf, double dx, double smallc,
                      hipStream_t st) {
  hipLaunchKernelGGL(k_ctl_begin, dim3(1), dim3(64), 0, st, ctl, cour, cf, dx, smallc);
}

void launch_ctl_end(RunCtl* ctl, bool odd, hipStream_t st) {
  hipLaunchKernelGGL(k_ctl_end, dim3(1), dim3(64), 0, st, ctl, (int) odd);
}

void launch_clear_slots(uint64_t* cour, hipStream_t st) {
  hipLaunchKernelGGL(k_clear_slots, dim3(1), dim3(256), 0, st, cour);
}
#endif  // HYDRO_BASE_UNIT

template <typename S>
void launch_init(const GridGeom& g, GridView<S> a, GridView<S> b, int bx, int by0, int by1,
                 double e_blast, hipStream_t st) {
  const long n = (long) (g.nx + 4) * (g.ny + 4);
  hipLaunchKernelGGL(k_init<S>, dim3(cdiv(n, 256)), dim3(256), 0, st, g, a, b, bx, by0, by1,
                     (S) e_blast);
}
#ifdef HYDRO_BASE_UNIT
template void launch_init<double>(const GridGeom&, GridView<double>, GridView<double>, int, int,
                                  int, double, hipStream_t);
template void launch_init<float>(const GridGeom&, GridView<float>, GridView<float>, int, int,
                                 int, double, hipStream_t);
template void launch_boundary<double>(int, const GridGeom&, const PhysArgs&, GridView<double>,
                                      GridView<double>, const RunCtl*, hipStream_t);
template void launch_boundary<float>(int, const GridGeom&, const PhysArgs&, GridView<float>,
                                     GridView<float>, const RunCtl*, hipStream_t);
template void launch_sweep<double>(int, const GridGeom&, const PhysArgs&, GridView<double>,
                                   GridView<double>, double, const RunCtl*, RunCtl*, uint64_t*,
                                   const SweepTune&, int, hipStream_t);
template void launch_step<double>(int, const GridGeom&, const PhysArgs&, GridView<double>,
                                  GridView<double>, double, const RunCtl*, RunCtl*, uint64_t*, int,
                                  hipStream_t);
template void launch_courant<double>(const GridGeom&, const PhysArgs&, GridView<double>,
                                     uint64_t*, const RunCtl*, hipStream_t);
#elif defined(HYDRO_MIXED_UNIT)
template void launch_sweep<float>(int, const GridGeom&, const PhysArgs&, GridView<float>,
                                  GridView<float>, double, const RunCtl*, RunCtl*, uint64_t*,
                                  const SweepTune&, int, hipStream_t);
template void launch_step<float>(int, const GridGeom&, const PhysArgs&, GridView<float>,
                                  GridView<float>, double, const RunCtl*, RunCtl*, uint64_t*, int,
                                  hipStream_t);
template void launch_courant<float>(const GridGeom&, const PhysArgs&, GridView<float>,
                                    uint64_t*, const RunCtl*, hipStream_t);
#endif

}  // namespace hydro
