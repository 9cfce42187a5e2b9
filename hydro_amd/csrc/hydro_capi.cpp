// C ABI of libhydro_amd: the handle API of include/hydro_amd.h and the
// HydroC99_2DMpi call surface of include/hydro_surface.h, mapped onto GPU
// grids.  Host-side bookkeeping only; all arithmetic is in hydro_kernels.hip.
#include <hip/hip_runtime.h>

#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/hydro_amd.h"
#include "hydro_kernels.hpp"

using namespace hydro;

// ---- errors ----------------------------------------------------------------------

static thread_local std::string g_err;

static int fail(const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_err = buf;
  return -1;
}

#define HIPCHK(call)                                                                  \
  do {                                                                                \
    hipError_t e_ = (call);                                                           \
    if (e_ != hipSuccess) return fail("%s: %s", #call, hipGetErrorString(e_));        \
  } while (0)

extern "C" const char* hydro_amd_last_error(void) { return g_err.c_str(); }

// For the other translation units of the library (hydro_batch.cpp, the C99
// host files, ...); C linkage so the C files can call it.
extern "C" int hydro_amd_set_error(const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_err = buf;
  return -1;
}

// ---- grid ------------------------------------------------------------------------

// Row pitch is a multiple of 32 elements and rows start 30 elements into the
// allocation, so the first interior cell (i = 2) of every row sits on a
// 256-byte boundary (y-sweep waves then read whole cache lines).
static constexpr long kOrigin = 30;

struct hydro_amd_grid {
  hydro_amd_params p;
  GridGeom geom;
  PhysArgs ph;
  int prec;
  size_t esz;
  long plane;  // elements per variable plane
  void* mem[2] = {nullptr, nullptr};
  GridView<double> vd[2];
  GridView<float> vf[2];
  uint64_t* cour = nullptr;
  RunCtl* ctl = nullptr;    // [2]: even and odd steps (hydro_kernels.hpp)
  RunCtl* hctl = nullptr;   // [2], pinned host copy: every RunCtl / dt transfer goes through it
  double* dlog = nullptr;
  int dlog_cap = 0;
  hipStream_t st = nullptr;
  int cur = 0;           // the buffer that holds the state
  long state_ver = 1;
  long cour_ver = 0;     // state version whose CFL maxima the slots hold (0: none)
  bool cour_dirty = false;
  SweepTune tune = {0, 1, 0, 0, -1};  // set by precision at creation
  // host mirror of the run control, valid between calls
  double t = 0, dt = 0;
  int nstep = 0;
  bool queued = false;  // steps were queued that the mirror does not show yet
  bool flips = false;   // each of them moves the state to the other buffer
  // cached two-step graphs, by the buffer that the even step reads
  hipGraphExec_t gexec[2] = {nullptr, nullptr};
  // kernel timing: events around each sweep / boundary launch (graphs off)
  bool prof = false;
  std::vector<hipEvent_t> ev_pool;
  std::vector<std::pair<int, int>> ev_pending;  // (kind, first event index)
  int ev_used = 0;
  double prof_ms[4] = {0, 0, 0, 0};             // x sweep, y sweep, boundary, courant
  long prof_n[4] = {0, 0, 0, 0};
};

// FP64 storage (the FP64 and FP64 fast forms) rather than FP32.
static bool dbl(const hydro_amd_grid* g) { return g->prec != HYDRO_AMD_MIXED; }

static int ev_pair(hydro_amd_grid* g) {
  if (g->ev_used + 2 > (int) g->ev_pool.size()) {
    for (int k = 0; k < 64; k++) {
      hipEvent_t e;
      if (hipEventCreate(&e) != hipSuccess) return -1;
      g->ev_pool.push_back(e);
    }
  }
  const int i = g->ev_used;
  g->ev_used += 2;
  return i;
}

// Collect finished timings (the stream must be idle).
static void prof_collect(hydro_amd_grid* g) {
  for (auto& pe : g->ev_pending) {
    float ms = 0;
    if (hipEventElapsedTime(&ms, g->ev_pool[pe.second], g->ev_pool[pe.second + 1]) == hipSuccess) {
      g->prof_ms[pe.first] += ms;
      g->prof_n[pe.first]++;
    }
  }
  g->ev_pending.clear();
  g->ev_used = 0;
}

// Wraps one launch in events when profiling; kind 0 x sweep, 1 y sweep,
// 2 boundary, 3 courant.
template <typename F>
static void timed(hydro_amd_grid* g, int kind, F&& launch) {
  int i = -1;
  if (g->prof && (i = ev_pair(g)) >= 0) (void) hipEventRecord(g->ev_pool[i], g->st);
  launch();
  if (i >= 0) {
    (void) hipEventRecord(g->ev_pool[i + 1], g->st);
    g->ev_pending.push_back({kind, i});
  }
}

static PhysArgs phys_of(const hydro_amd_params& p) {
  PhysArgs a;
  a.gamma = p.gamma;
  a.smallr = p.smallr;
  a.smallc = p.smallc;
  a.slope_type = p.slope_type;
  a.courant_factor = p.courant_factor;
  a.dx = p.dx;
  a.niter = p.niter_riemann;
  a.iorder = p.iorder;
  a.scheme = p.scheme;
  a.bl = p.boundary_left;
  a.br = p.boundary_right;
  a.bd = p.boundary_down;
  a.bu = p.boundary_up;
  return a;
}

extern "C" void hydro_amd_params_default(hydro_amd_params* p) {
  // HydroC99_2DMpi/Src/parametres.c:64-109
  memset(p, 0, sizeof(*p));
  p->nx = 20;
  p->ny = 20;
  p->dx = 1.0;
  p->gamma = 1.4;
  p->courant_factor = 0.5;
  p->smallc = 1e-10;
  p->smallr = 1e-10;
  p->slope_type = 1.0;
  p->niter_riemann = 10;
  p->iorder = 2;
  p->scheme = HSCHEME_MUSCL;
  p->boundary_left = p->boundary_right = p->boundary_down = p->boundary_up = 1;
  p->tend = 0.0;
  p->nstepmax = 0x7fffffff;
  p->precision = HYDRO_AMD_FP64;
}

extern "C" void hydro_amd_params_from_surface(const hydroparam_t* H, hydro_amd_params* p) {
  hydro_amd_params_default(p);
  p->nx = H->nx;
  p->ny = H->ny;
  p->dx = H->dx;
  p->gamma = H->gamma;
  p->courant_factor = H->courant_factor;
  p->smallc = H->smallc;
  p->smallr = H->smallr;
  p->slope_type = H->slope_type;
  p->niter_riemann = H->niter_riemann;
  p->iorder = H->iorder;
  p->scheme = H->scheme;
  p->boundary_left = H->boundary_left;
  p->boundary_right = H->boundary_right;
  p->boundary_down = H->boundary_down;
  p->boundary_up = H->boundary_up;
  p->tend = H->tend;
  p->nstepmax = H->nstepmax;
}

static void drop_graph(hydro_amd_grid* g) {
  for (auto& e : g->gexec)
    if (e) {
      (void) hipGraphExecDestroy(e);
      e = nullptr;
    }
}

extern "C" void hydro_amd_grid_destroy(hydro_amd_grid* g) {
  if (!g) return;
  if (g->st) (void) hipStreamSynchronize(g->st);
  drop_graph(g);
  for (auto e : g->ev_pool) (void) hipEventDestroy(e);
  for (int k = 0; k < 2; k++)
    if (g->mem[k]) (void) hipFree(g->mem[k]);
  if (g->cour) (void) hipFree(g->cour);
  if (g->ctl) (void) hipFree(g->ctl);
  if (g->dlog) (void) hipFree(g->dlog);
  if (g->hctl) (void) hipHostFree(g->hctl);
  if (g->st) (void) hipStreamDestroy(g->st);
  delete g;
}

static int alloc_buffer(hydro_amd_grid* g, int k) {
  const long total = 4 * g->plane + kOrigin + 64;
  HIPCHK(hipMalloc(&g->mem[k], (size_t) total * g->esz));
  if (dbl(g)) {
    double* b = (double*) g->mem[k] + kOrigin;
    for (int v = 0; v < 4; v++) g->vd[k].p[v] = b + v * g->plane;
  } else {
    float* b = (float*) g->mem[k] + kOrigin;
    for (int v = 0; v < 4; v++) g->vf[k].p[v] = b + v * g->plane;
  }
  HIPCHK(hipMemsetAsync(g->mem[k], 0, (size_t) total * g->esz, g->st));
  return 0;
}

static int validate(const hydro_amd_params* p) {
  if (!p) return fail("null params");
  if (p->nx < 1 || p->ny < 1) return fail("nx, ny must be >= 1 (got %d, %d)", p->nx, p->ny);
  // x-sweep row segments are counted in 32-bit ints (hydro_sweeps.hpp SegWalk)
  if ((long) (p->nx + 4) * (p->ny + 4) > (1L << 40) ||
      (long) ((p->nx + kXSeg - 1) / kXSeg) * p->ny > (1L << 30))
    return fail("grid too large");
  if (!(p->dx > 0)) return fail("dx must be > 0");
  if (!(p->gamma > 1)) return fail("gamma must be > 1");
  if (p->precision != HYDRO_AMD_FP64 && p->precision != HYDRO_AMD_MIXED &&
      p->precision != HYDRO_AMD_FP64_FAST)
    return fail("unknown precision %d", p->precision);
  if (p->scheme < 1 || p->scheme > 3) return fail("unknown scheme %d", p->scheme);
  if (p->niter_riemann < 0) return fail("niter_riemann must be >= 0");
  return 0;
}

// The mirror's run control to the device, no step open.  fresh: the pinned
// copy was never used.
static int write_ctl(hydro_amd_grid* g, bool fresh = false) {
  if (!fresh) HIPCHK(hipStreamSynchronize(g->st));  // it may still feed a queued copy
  RunCtl c{};
  c.t = g->t;
  c.dt = g->dt;
  c.tend = g->p.tend;
  c.nstep = g->nstep;
  c.nstepmax = g->p.nstepmax;
  g->hctl[0] = g->hctl[1] = c;
  g->queued = false;
  HIPCHK(hipMemcpyAsync(g->ctl, g->hctl, 2 * sizeof(RunCtl), hipMemcpyHostToDevice, g->st));
  HIPCHK(hipStreamSynchronize(g->st));
  return 0;
}

extern "C" hydro_amd_grid* hydro_amd_grid_create(const hydro_amd_params* p) {
  if (validate(p)) return nullptr;
  hydro_amd_grid* g = new hydro_amd_grid();
  g->p = *p;
  g->prec = p->precision;
  g->esz = dbl(g) ? sizeof(double) : sizeof(float);
  g->tune = SweepTune{0, dbl(g) ? 1 : 4, 0, 0, -1};
  g->geom.nx = p->nx;
  g->geom.ny = p->ny;
  g->geom.pitch = ((long) p->nx + 4 + 31) / 32 * 32;
  g->plane = g->geom.pitch * (p->ny + 4);
  g->ph = phys_of(*p);
  g->t = 0;
  g->nstep = 0;
  g->dt = 0;
  if (hipStreamCreateWithFlags(&g->st, hipStreamNonBlocking) != hipSuccess ||
      alloc_buffer(g, 0) || alloc_buffer(g, 1) ||
      hipMalloc(&g->cour, 2 * kCourSlots * sizeof(uint64_t)) != hipSuccess ||
      hipMalloc(&g->ctl, 2 * sizeof(RunCtl)) != hipSuccess ||
      hipHostMalloc(&g->hctl, 2 * sizeof(RunCtl), hipHostMallocDefault) != hipSuccess) {
    if (g_err.empty()) fail("device allocation failed");
    hydro_amd_grid_destroy(g);
    return nullptr;
  }
  launch_clear_slots(g->cour, g->st);
  if (write_ctl(g, true)) {
    fail("grid setup failed");
    hydro_amd_grid_destroy(g);
    return nullptr;
  }
  return g;
}

extern "C" long long hydro_amd_grid_bytes(const hydro_amd_grid* g) {
  return g ? (long long) (2 * (4 * g->plane + kOrigin + 64) * g->esz +
                          2 * kCourSlots * sizeof(uint64_t) + 2 * sizeof(RunCtl) +
                          g->dlog_cap * 8)
           : 0;
}

static void bump(hydro_amd_grid* g) { g->state_ver++; }

static int run_finish(hydro_amd_grid* g, int* steps_done);

// Takes up the outcome of queued steps: which buffer the state is in, t, nstep.
static int settle(hydro_amd_grid* g) { return g->queued ? run_finish(g, nullptr) : 0; }

static int do_init(hydro_amd_grid* g, int bx, int by0, int by1, double e) {
  if (settle(g)) return -1;  // (queued steps may leave maxima in the CFL slots)
  if (dbl(g))
    launch_init<double>(g->geom, g->vd[0], g->vd[1], bx, by0, by1, e, g->st);
  else
    launch_init<float>(g->geom, g->vf[0], g->vf[1], bx, by0, by1, e, g->st);
  HIPCHK(hipGetLastError());
  g->cur = 0;
  bump(g);
  g->t = 0;
  g->nstep = 0;
  g->dt = 0;
  return write_ctl(g);
}

extern "C" int hydro_amd_grid_init(hydro_amd_grid* g, int testcase) {
  if (!g) return fail("null grid");
  const int nxt = g->p.nx + 4, nyt = g->p.ny + 4;
  const double eb = 1.0 / g->p.dx / g->p.dx;  // hydro_funcs.c:92
  switch (testcase) {
    case 0: return do_init(g, nxt / 2, nyt / 2, nyt / 2 + 1, eb);
    case 1: return do_init(g, 2, 2, 3, eb);
    case 2: return do_init(g, 2, 2, nyt, eb);
    default: return fail("testcase %d not implemented", testcase);
  }
}

extern "C" int hydro_amd_grid_init_blast(hydro_amd_grid* g, int bx, int by, double e) {
  if (!g) return fail("null grid");
  if (bx < 0 || by < 0 || bx >= g->p.nx || by >= g->p.ny)
    return fail("blast cell (%d, %d) outside %dx%d", bx, by, g->p.nx, g->p.ny);
  return do_init(g, bx + 2, by + 2, by + 3, e);
}

extern "C" int hydro_amd_grid_upload(hydro_amd_grid* g, const double* u) {
  if (!g || !u) return fail("null argument");
  if (settle(g)) return -1;
  const long nxt = g->p.nx + 4, rows = 4L * (g->p.ny + 4);
  void* dst = (char*) g->mem[0] + kOrigin * g->esz;
  if (stage_h2d(dst, (int) g->esz, g->geom.pitch, u, 8, nxt, rows, g->st)) return -1;
  // the second buffer carries the same ghosts (they are refreshed into both)
  const long total = 4 * g->plane + kOrigin + 64;
  HIPCHK(hipMemcpyAsync(g->mem[1], g->mem[0], (size_t) total * g->esz,
                        hipMemcpyDeviceToDevice, g->st));
  g->cur = 0;
  bump(g);
  return 0;
}

extern "C" int hydro_amd_grid_download(hydro_amd_grid* g, double* u) {
  if (!g || !u) return fail("null argument");
  if (settle(g)) return -1;
  const long nxt = g->p.nx + 4, rows = 4L * (g->p.ny + 4);
  const void* src = (const char*) g->mem[g->cur] + kOrigin * g->esz;
  return stage_d2h(u, 8, src, (int) g->esz, g->geom.pitch, nxt, rows, g->st) ? -1 : 0;
}

// Image size rule of HydroC99_2Domp/Src/Image.c:124-126 (single rank): the
// smallest shrink with nx/shrink and ny/shrink both <= shrink_size.
extern "C" int hydro_amd_grid_image(hydro_amd_grid* g, int shrink_size, unsigned char* rgb,
                                    long long cap, int* width, int* height) {
  if (!g || !width || !height) return fail("null argument");
  if (shrink_size < 1) return fail("shrink_size %d: must be at least 1", shrink_size);
  int s = 1;
  while (g->p.nx / s > shrink_size || g->p.ny / s > shrink_size) s++;
  const int w = g->p.nx / s, h = g->p.ny / s;
  *width = w;
  *height = h;
  if (!rgb) return 0;
  const long long need = 3LL * w * h;
  if (cap < need) return fail("image buffer of %lld bytes, %lld needed", cap, need);
  if (need == 0) return 0;
  if (settle(g)) return -1;
  void* d = nullptr;  // [8-byte maximum key][pixels]
  HIPCHK(hipMallocAsync(&d, (size_t) (8 + need), g->st));
  unsigned long long* key = (unsigned long long*) d;
  unsigned char* px = (unsigned char*) d + 8;
  if (dbl(g))
    launch_image<double>(g->geom, g->vd[g->cur].p[0], s, w, h, key, px, g->st);
  else
    launch_image<float>(g->geom, g->vf[g->cur].p[0], s, w, h, key, px, g->st);
  const hipError_t e1 = hipMemcpyAsync(rgb, px, (size_t) need, hipMemcpyDeviceToHost, g->st);
  const hipError_t e2 = hipFreeAsync(d, g->st);
  const hipError_t e3 = hipStreamSynchronize(g->st);
  if (e1 != hipSuccess || e2 != hipSuccess || e3 != hipSuccess)
    return fail("image: %s", hipGetErrorString(e1 != hipSuccess ? e1 : e2 != hipSuccess ? e2 : e3));
  return 0;
}

// ---- steps ---------------------------------------------------------------------------

static void enq_boundary(hydro_amd_grid* g, int idim, int src, const RunCtl* ctl) {
  timed(g, 2, [&] {
    if (dbl(g))
      launch_boundary<double>(idim, g->geom, g->ph, g->vd[src], g->vd[1 - src], ctl, g->st);
    else
      launch_boundary<float>(idim, g->geom, g->ph, g->vf[src], g->vf[1 - src], ctl, g->st);
  });
}

// The sweeps form their own ghosts, unless the grid is too narrow for that.
static bool folds_ghosts(const hydro_amd_grid* g) {
  return g->p.nx >= kGhostMin && g->p.ny >= kGhostMin;
}

// One sweep with its ghosts, reading buffer `src` and writing the other; the
// ghost values are left in buffer `state`, which holds the state between steps.
static void enq_sweep(hydro_amd_grid* g, int idim, int src, int state, double dt,
                      const RunCtl* ctl, RunCtl* nxt, bool cour) {
  uint64_t* c = cour ? g->cour : nullptr;
  const int fill = folds_ghosts(g) ? (src == state ? 1 : 2) : -1;
  if (fill < 0) enq_boundary(g, idim, src, ctl);
  timed(g, idim == 1 ? 0 : 1, [&] {
    if (g->prec == HYDRO_AMD_FP64_FAST)
      launch_sweep_fast(idim, g->geom, g->ph, g->vd[src], g->vd[1 - src], dt, ctl, nxt, c, g->tune,
                        fill, g->st);
    else if (g->prec == HYDRO_AMD_FP64)
      launch_sweep<double>(idim, g->geom, g->ph, g->vd[src], g->vd[1 - src], dt, ctl, nxt, c,
                           g->tune, fill, g->st);
    else
      launch_sweep<float>(idim, g->geom, g->ph, g->vf[src], g->vf[1 - src], dt, ctl, nxt, c,
                          g->tune, fill, g->st);
  });
}

static void enq_courant(hydro_amd_grid* g, const RunCtl* ctl) {
  timed(g, 3, [&] {
    if (dbl(g))  // (the FP64 fast form too: one launch per state, IEEE arithmetic)
      launch_courant<double>(g->geom, g->ph, g->vd[g->cur], g->cour, ctl, g->st);
    else
      launch_courant<float>(g->geom, g->ph, g->vf[g->cur], g->cour, ctl, g->st);
  });
}

// Rows a wave of the march kernel takes: the segments fill the GPU's `slots`
// resident waves once or a whole number of times, sqrt(wave rows) / 240 (a
// segment's fixed cost against the unevenness of its end, as y_rows).  The best
// of 1-12 times, fast form: 2048x1536 (54000 wave rows) 1, 3200x2400 1-2, 4099x3001
// 2-3, 6000x5000 3, 8192x8192 4-5, 16384x12000 (3.3e6) 7-10; mixed the same.
static int march_rows(long ncol, long ny, long slots) {
  const long times = std::max(1L, (long) (std::sqrt((double) (ncol * ny)) / 240 + 0.5));
  const long nseg = std::max(1L, times * slots / ncol);
  return (int) ((ny + nseg - 1) / nseg);
}

// How a whole step is launched on this grid (SweepTune::step).  Times below are of
// a step, of a blast (in brackets: of a flow that moves everywhere).
// Tiles save a launch and the y march's serial solves and pay with halo cells,
// so they are for grids whose waves do not fill the GPU; counted in their waves,
// the lines lie where they and the next were measured alike.  Tiles / two sweeps:
// 250x125 FP64 21.3 / 23.5 us (17.4 / 21.4), fast 13.7 / 17.3 (12.6 / 16.4), mixed
// 12.1 / 15.3; 500x500 (9000 waves) FP64 38.1 / 40.7 (48.2 / 47.6), fast 24.9 / 26.8
// (28.8 / 30.5); 600x600 (12000) FP64 43.1 / 48.1 (55.2 / 56.5); 777x600 (15600) FP64
// 48.6 / 51.8 (67.8 / 62.4), fast 31.2 / 34.3 (38.4 / 39.6); 850x700 (21000) fast 38.2 /
// 39.0 (46.9 / 45.0); mixed with 16 rows 500x500 18.3 / 21.5, 1021x767 (18400) 30.3 /
// 33.1, 1531x1200 (41600) 53.7 / 53.9.
// The march passes over memory once a step instead of twice, which is what bounds
// the large grids' sweeps in the fast form and half bounds them in the mixed
// form (the FP64 form's arithmetic bounds it: no march).  March / two sweeps, fast:
// 1021x767 (13800 wave rows) 43.7 / 42.5 (57.3 / 50.1), 1100x900 (17100) 49.6 / 51.4
// (65.5 / 61.0), 1150x950 (19000) 49.9 / 54.5 (64.7 / 62.9), 1400x1150 61.6 / 70.9
// (83.3 / 85.4), 2048x1536 103 / 106 (146 / 145), 3200x2400 205 / 234 (310 / 322),
// 4099x3001 317 / 364 (455 / 474), 8192x1024 228 / 257 (326 / 332), 8192x8192 1543 /
// 1815 (1988 / 2077); mixed: 3400x2400 (137000) 144 / 144 (183 / 183), 3600x2600
// (156000) 161 / 171 (206 / 210), 4099x3001 204 / 219, 8192x8192 933 / 993,
// 16384x12000 2650 / 2810.  Its waves update 60 columns, the sweeps' 63 and 64: in
// the mixed form, where that counts, not where the grid's width makes it much
// worse (500x15000 145 / 142, 192 / 176).
static int default_step(const hydro_amd_grid* g) {
  if (!folds_ghosts(g)) return 0;
  const long nx = g->p.nx, ny = g->p.ny, ncol = (nx + 59) / 60;
  auto waves = [&](long rows) { return ncol * ((ny + rows - 5) / (rows - 4)) * rows; };
  if (g->prec == HYDRO_AMD_FP64) return waves(8) <= 10000 ? 8 : 0;
  if (g->prec == HYDRO_AMD_FP64_FAST) {
    if (waves(8) <= 16000) return 8;
    return ncol * ny >= 16000 && nx < kMarchWidest ? kMarch + march_rows(ncol, ny, 4 * kSimds)
                                                   : 0;
  }
  if (waves(8) <= 5000) return 8;
  if (waves(16) <= 24000) return 16;
  const long lanes = (nx + 251) / 252 * 256 + (nx + 63) / 64 * 64;  // of the sweeps
  return ncol * ny >= 150000 && nx < kMarchWidest && 100 * 2 * 64 * ncol <= 108 * lanes
             ? kMarch + march_rows(ncol, ny, 5 * kSimds)
             : 0;
}

static int unprofiled_rows(const hydro_amd_grid* g) {
  return g->tune.step >= 0 ? g->tune.step : default_step(g);
}

static int step_rows(const hydro_amd_grid* g) {
  return g->prof ? 0 : unprofiled_rows(g);  // (profiles are of the sweeps)
}

extern "C" int hydro_amd_grid_whole_steps(const hydro_amd_grid* g) {
  return g && unprofiled_rows(g) > 0;
}

// hydro_godunov.c:98-237: both directions, ghosts refilled before each, on the
// state in buffer src; returns the buffer that the new state is in.  `cour`
// folds the CFL maxima of the result into the second sweep.
static int enq_godunov(hydro_amd_grid* g, int src, int idim_start, double dt, const RunCtl* ctl,
                       RunCtl* nxt, bool cour) {
  const int d1 = idim_start == 1 ? 1 : 2, d2 = 3 - d1;
  const int rows = d1 == 2 || !cour ? step_rows(g) : 0;  // (x first folds no maxima)
  if (rows) {
    uint64_t* c = cour ? g->cour : nullptr;
    if (g->prec == HYDRO_AMD_FP64_FAST)
      launch_step_fast(d1, g->geom, g->ph, g->vd[src], g->vd[1 - src], dt, ctl, nxt, c, rows,
                       g->st);
    else if (g->prec == HYDRO_AMD_FP64)
      launch_step<double>(d1, g->geom, g->ph, g->vd[src], g->vd[1 - src], dt, ctl, nxt, c, rows,
                          g->st);
    else
      launch_step<float>(d1, g->geom, g->ph, g->vf[src], g->vf[1 - src], dt, ctl, nxt, c, rows,
                         g->st);
    return 1 - src;
  }
  enq_sweep(g, d1, src, src, dt, ctl, nxt, false);
  enq_sweep(g, d2, 1 - src, src, dt, ctl, nullptr, cour);
  return src;
}

static void prepare_slots(hydro_amd_grid* g) {
  if (g->cour_dirty) launch_clear_slots(g->cour, g->st);
  g->cour_dirty = false;
  g->cour_ver = 0;
}

static int godunov_impl(hydro_amd_grid* g, int idim, double dt, bool want_cour) {
  if (idim != 1 && idim != 2) return fail("idim must be 1 or 2 (got %d)", idim);
  if (settle(g)) return -1;
  if (want_cour) prepare_slots(g);
  g->cur = enq_godunov(g, g->cur, idim, dt, nullptr, nullptr, want_cour);
  HIPCHK(hipGetLastError());
  bump(g);
  if (want_cour) {
    g->cour_ver = g->state_ver;
    g->cour_dirty = true;
  } else if (g->cour_dirty) {
    g->cour_ver = 0;
  }
  return 0;
}

extern "C" int hydro_amd_grid_godunov(hydro_amd_grid* g, int idim, double dt) {
  if (!g) return fail("null grid");
  // the reference alternates x-then-y (even steps) and y-then-x (odd steps);
  // dt is recomputed after odd steps, so those fold the CFL maxima in.
  return godunov_impl(g, idim, dt, idim == 2);
}

extern "C" int hydro_amd_grid_make_boundary(hydro_amd_grid* g, int idim) {
  if (!g) return fail("null grid");
  if (idim != 1 && idim != 2) return fail("idim must be 1 or 2 (got %d)", idim);
  if (settle(g)) return -1;
  enq_boundary(g, idim, g->cur, nullptr);
  HIPCHK(hipGetLastError());
  return 0;
}

static void ensure_cour(hydro_amd_grid* g) {
  if (g->cour_ver == g->state_ver) return;
  prepare_slots(g);
  enq_courant(g, nullptr);
  g->cour_ver = g->state_ver;
  g->cour_dirty = true;
}

extern "C" int hydro_amd_grid_compute_deltat(hydro_amd_grid* g, double* dt) {
  if (!g || !dt) return fail("null argument");
  if (settle(g)) return -1;
  ensure_cour(g);
  // (straight into pinned memory: a copy would be a launch more)
  launch_dt_finalize(g->cour, g->p.courant_factor, g->p.dx, g->p.smallc, &g->hctl->dt, g->st);
  HIPCHK(hipGetLastError());
  g->cour_dirty = false;
  g->cour_ver = 0;
  HIPCHK(hipStreamSynchronize(g->st));
  *dt = g->hctl->dt;
  return 0;
}

// ---- device time loop ------------------------------------------------------------------

// One step of main.c:244-298 with run control on the device; `n` is the step
// number the host expects (its parity fixes the sweep order and the control).
// From the state in buffer src; returns the buffer of the new state.
static int enq_step(hydro_amd_grid* g, int src, int n) {
  if (n % 2 == 0) {
    launch_ctl_begin(g->ctl, g->cour, g->p.courant_factor, g->p.dx, g->p.smallc, g->st);
    return enq_godunov(g, src, 1, 0.0, g->ctl, g->ctl + 1, false);
  }
  return enq_godunov(g, src, 2, 0.0, g->ctl + 1, nullptr, true);
}

// The outcome of the queued steps (ctl[0]).
static int read_ctl(hydro_amd_grid* g, RunCtl* c) {
  HIPCHK(hipMemcpyAsync(g->hctl, g->ctl, sizeof(RunCtl), hipMemcpyDeviceToHost, g->st));
  HIPCHK(hipStreamSynchronize(g->st));
  *c = *g->hctl;
  return 0;
}

static int get_graph(hydro_amd_grid* g, int src) {
  // steps (even, odd) captured once; valid while the grid's buffers live (two
  // steps leave the state in the buffer that they found it in)
  if (g->gexec[src]) return 0;
  hipGraph_t graph;
  HIPCHK(hipStreamBeginCapture(g->st, hipStreamCaptureModeThreadLocal));
  enq_step(g, enq_step(g, src, 0), 1);
  hipError_t e = hipStreamEndCapture(g->st, &graph);
  if (e != hipSuccess) return fail("graph capture: %s", hipGetErrorString(e));
  e = hipGraphInstantiate(&g->gexec[src], graph, nullptr, nullptr, 0);
  (void) hipGraphDestroy(graph);
  if (e != hipSuccess) {
    g->gexec[src] = nullptr;
    return fail("graph instantiate: %s", hipGetErrorString(e));
  }
  return 0;
}

static int run_finish(hydro_amd_grid* g, int* steps_done) {
  RunCtl c;
  if (read_ctl(g, &c)) return -1;
  g->queued = false;
  if (g->prof) prof_collect(g);
  const int done = c.nstep - g->nstep;
  if (done > 0) {
    if (g->flips && done % 2 == 1) g->cur = 1 - g->cur;
    g->state_ver += done;
    // after an odd step the slots hold the maxima of the current state; after
    // an even one they were consumed by that step's dt
    if (c.nstep % 2 == 0) {
      g->cour_ver = g->state_ver;
      g->cour_dirty = true;
    } else {
      g->cour_ver = 0;
      g->cour_dirty = false;
    }
  }
  g->t = c.t;
  g->dt = c.dt;
  g->nstep = c.nstep;
  if (steps_done) *steps_done = done;
  return 0;
}

// `start`, when given, is recorded on the stream right before the first step
// (the autotuner's clock, which the run control's set-up stays outside of).
static int run_enqueue(hydro_amd_grid* g, int max_steps, int log_cap,
                       hipEvent_t start = nullptr) {
  if (max_steps <= 0) return 0;
  if (settle(g)) return -1;  // the step parity below is the mirror's
  // dt of an even step comes from the CFL maxima of the current state; an odd
  // step folds its maxima into slots that hold no other state's
  if (g->nstep % 2 == 0) ensure_cour(g);
  else prepare_slots(g);
  // control, log setup + limits
  HIPCHK(hipStreamSynchronize(g->st));  // the pinned copy may still feed a queued copy
  RunCtl c{};
  c.t = g->t;
  c.dt = g->dt;
  c.nstep = g->nstep;
  c.tend = g->p.tend;
  c.nstepmax = g->p.nstepmax;
  c.log_base = g->nstep;
  c.log_cap = log_cap;
  c.log = log_cap > 0 ? g->dlog : nullptr;
  g->hctl[0] = c;
  // an odd step to begin with is open from the start
  c.active = g->nstep % 2 == 1 && (c.t < c.tend) && (c.nstep < c.nstepmax);
  g->hctl[1] = c;
  // nothing rewrites the pinned copy before the next synchronising call
  HIPCHK(hipMemcpyAsync(g->ctl, g->hctl, 2 * sizeof(RunCtl), hipMemcpyHostToDevice, g->st));
  g->queued = true;
  g->flips = step_rows(g) > 0;
  if (start) HIPCHK(hipEventRecord(start, g->st));
  int n = g->nstep, left = max_steps, src = g->cur;
  if (n % 2 == 1) {  // finish the odd step first so the graph starts even
    src = enq_step(g, src, n);
    n++;
    left--;
  }
  if (left >= 2 && !g->prof) {
    if (get_graph(g, src)) return -1;
    for (; left >= 2; left -= 2, n += 2) HIPCHK(hipGraphLaunch(g->gexec[src], g->st));
  }
  for (; left >= 2; left--, n++) src = enq_step(g, src, n);
  if (left == 1) {
    src = enq_step(g, src, n);
    n++;
  }
  launch_ctl_end(g->ctl, n % 2 == 0, g->st);  // (n: the next step)
  HIPCHK(hipGetLastError());
  return 0;
}

// Steps queued between host checks of the device loop: a run stopped by tend
// is noticed within one chunk, so no more than this many no-op steps are
// ever queued past its end.
static constexpr int kRunChunk = 256;

extern "C" int hydro_amd_grid_run(hydro_amd_grid* g, int max_steps, double* dt_log) {
  if (!g) return fail("null grid");
  if (max_steps < 0) return fail("max_steps < 0");
  long left = max_steps;
  if (left > (long) g->p.nstepmax - g->nstep) left = (long) g->p.nstepmax - g->nstep;
  if (left < 0) left = 0;
  int total = 0;
  while (left > 0) {
    const int chunk = (int) (left < kRunChunk ? left : kRunChunk);
    const int cap = dt_log ? chunk : 0;
    if (cap > g->dlog_cap) {
      if (g->dlog) (void) hipFree(g->dlog);
      g->dlog = nullptr;
      g->dlog_cap = 0;
      HIPCHK(hipMalloc(&g->dlog, (size_t) kRunChunk * sizeof(double)));
      g->dlog_cap = kRunChunk;
    }
    if (run_enqueue(g, chunk, cap)) return -1;
    int done = 0;
    if (run_finish(g, &done)) return -1;
    if (dt_log && done > 0)
      HIPCHK(hipMemcpy(dt_log + total, g->dlog, (size_t) done * sizeof(double),
                       hipMemcpyDeviceToHost));
    total += done;
    left -= chunk;
    if (done < chunk) break;  // the device loop ended (t >= tend)
  }
  return total;
}

extern "C" int hydro_amd_grid_run_async(hydro_amd_grid* g, int max_steps) {
  if (!g) return fail("null grid");
  if (max_steps < 0) return fail("max_steps < 0");
  long n = max_steps;
  if (n > (long) g->p.nstepmax - g->nstep) n = (long) g->p.nstepmax - g->nstep;
  if (run_enqueue(g, n > 0 ? (int) n : 0, 0)) return -1;
  return 0;
}

extern "C" int hydro_amd_grid_sync(hydro_amd_grid* g) {
  if (!g) return fail("null grid");
  HIPCHK(hipStreamSynchronize(g->st));
  return run_finish(g, nullptr);
}

extern "C" int hydro_amd_grid_state(hydro_amd_grid* g, double* t, int* nstep, double* dt) {
  if (!g) return fail("null grid");
  if (t) *t = g->t;
  if (nstep) *nstep = g->nstep;
  if (dt) *dt = g->dt;
  return 0;
}

extern "C" int hydro_amd_grid_set_state(hydro_amd_grid* g, double t, int nstep, double dt) {
  if (!g) return fail("null grid");
  if (nstep < 0) return fail("nstep < 0");
  if (settle(g)) return -1;
  g->t = t;
  g->nstep = nstep;
  g->dt = dt;
  return write_ctl(g);
}

extern "C" int hydro_amd_grid_set_limits(hydro_amd_grid* g, double tend, int nstepmax) {
  if (!g) return fail("null grid");
  if (settle(g)) return -1;
  g->p.tend = tend;
  g->p.nstepmax = nstepmax;
  return write_ctl(g);
}

extern "C" int hydro_amd_grid_set_profile(hydro_amd_grid* g, int on) {
  if (!g) return fail("null grid");
  HIPCHK(hipStreamSynchronize(g->st));
  prof_collect(g);
  g->prof = on != 0;
  for (int k = 0; k < 4; k++) {
    g->prof_ms[k] = 0;
    g->prof_n[k] = 0;
  }
  return 0;
}

extern "C" int hydro_amd_grid_profile(hydro_amd_grid* g, double* ms, long long* n) {
  if (!g) return fail("null grid");
  HIPCHK(hipStreamSynchronize(g->st));
  prof_collect(g);
  for (int k = 0; k < 4; k++) {
    if (ms) ms[k] = g->prof_ms[k];
    if (n) n[k] = g->prof_n[k];
  }
  return 0;
}

// ---- autotuner ------------------------------------------------------------------------

// Times one sweep launch shape: `reps` launches reading the state's buffer and
// writing the other's interior (the state is untouched; the other buffer is
// scratch between steps), HIP events on the grid's stream.  Returns ms per launch.
// Average time of one sweep launch in direction idim with launch shape t
// (reading the state, writing the scratch buffer); with cour non-null, the
// variant that also folds the CFL maxima of its output into cour.
static double time_sweep(hydro_amd_grid* g, int idim, const SweepTune& t, int reps,
                         uint64_t* cour = nullptr) {
  hipEvent_t a, b;
  if (hipEventCreate(&a) != hipSuccess) return 1e30;
  if (hipEventCreate(&b) != hipSuccess) {
    (void) hipEventDestroy(a);
    return 1e30;
  }
  const int fill = folds_ghosts(g) ? 0 : -1, src = g->cur, dst = 1 - g->cur;
  auto launch = [&] {
    if (g->prec == HYDRO_AMD_FP64_FAST)
      launch_sweep_fast(idim, g->geom, g->ph, g->vd[src], g->vd[dst], 1e-12, nullptr, nullptr, cour, t,
                        fill, g->st);
    else if (g->prec == HYDRO_AMD_FP64)
      launch_sweep<double>(idim, g->geom, g->ph, g->vd[src], g->vd[dst], 1e-12, nullptr, nullptr, cour, t,
                           fill, g->st);
    else
      launch_sweep<float>(idim, g->geom, g->ph, g->vf[src], g->vf[dst], 1e-12, nullptr, nullptr, cour, t,
                          fill, g->st);
  };
  launch();  // warm
  (void) hipEventRecord(a, g->st);
  for (int r = 0; r < reps; r++) launch();
  (void) hipEventRecord(b, g->st);
  float ms = 0;
  if (hipEventSynchronize(b) != hipSuccess || hipEventElapsedTime(&ms, a, b) != hipSuccess)
    ms = 1e30f;
  (void) hipEventDestroy(a);
  (void) hipEventDestroy(b);
  return ms / reps;
}

// Indices of the k smallest scores.
static std::vector<int> best_of(const std::vector<double>& ms, int k) {
  std::vector<int> idx(ms.size());
  for (size_t c = 0; c < ms.size(); c++) idx[c] = (int) c;
  std::sort(idx.begin(), idx.end(), [&](int a, int b) { return ms[a] < ms[b]; });
  if ((int) idx.size() > k) idx.resize(k);
  return idx;
}

// Whole steps with each candidate shape, from a saved copy of the state and
// the CFL slots that is put back before each trial and at the end, with t,
// nstep and dt, so the run continues exactly as if untuned: the isolated
// launches of the first pass miss how a shape fares between the other kernels
// of a step (tails, caches), which moved their pick by a few per cent.
// Returns the fastest candidate, or `fallback` when the copy cannot be
// allocated or a call fails.
static SweepTune tune_by_steps(hydro_amd_grid* g, const std::vector<SweepTune>& cand,
                               const SweepTune& fallback) {
  if (cand.size() < 2 || g->prof) return fallback;
  const size_t bytes = (size_t) (4 * g->plane + kOrigin + 64) * g->esz;
  const size_t slot_bytes = 2 * kCourSlots * sizeof(uint64_t);
  char* save = nullptr;
  if (hipMalloc(&save, bytes + slot_bytes) != hipSuccess) {
    (void) hipGetLastError();
    return fallback;
  }
  const double t0 = g->t, dt0 = g->dt;
  const int n0 = g->nstep, cur0 = g->cur;
  const bool slots_valid = g->cour_ver == g->state_ver;
  const bool dirty0 = g->cour_dirty;
  bool ok = hipMemcpyAsync(save, g->mem[cur0], bytes, hipMemcpyDeviceToDevice, g->st) ==
                hipSuccess &&
            hipMemcpyAsync(save + bytes, g->cour, slot_bytes, hipMemcpyDeviceToDevice, g->st) ==
                hipSuccess;
  auto restore = [&] {
    ok = ok &&
         hipMemcpyAsync(g->mem[cur0], save, bytes, hipMemcpyDeviceToDevice, g->st) == hipSuccess &&
         hipMemcpyAsync(g->cour, save + bytes, slot_bytes, hipMemcpyDeviceToDevice, g->st) ==
             hipSuccess;
    g->t = t0;
    g->nstep = n0;
    g->dt = dt0;
    g->cur = cur0;
    bump(g);
    g->cour_ver = slots_valid ? g->state_ver : 0;
    g->cour_dirty = dirty0;
    ok = ok && write_ctl(g) == 0;
  };
  constexpr int kSteps = 8;  // of each parity, half (the odd ones fold the CFL maxima)
  std::vector<double> ms(cand.size(), 0.0);
  hipEvent_t a = nullptr, b = nullptr;
  ok = ok && hipEventCreate(&a) == hipSuccess && hipEventCreate(&b) == hipSuccess;
  for (int pass = 0; pass < 2 && ok; pass++)
    for (size_t k = 0; k < cand.size() && ok; k++) {
      const size_t c = pass ? cand.size() - 1 - k : k;
      g->tune = cand[c];
      drop_graph(g);
      restore();  // a first run builds the shape's graph
      ok = ok && run_enqueue(g, 2, 0) == 0 && run_finish(g, nullptr) == 0;
      restore();
      if (n0 % 2 == 0) ensure_cour(g);  // (outside the clock)
      ok = ok && run_enqueue(g, kSteps, 0, a) == 0 && hipEventRecord(b, g->st) == hipSuccess &&
           run_finish(g, nullptr) == 0;
      float e = 0;
      ok = ok && hipEventElapsedTime(&e, a, b) == hipSuccess;
      ms[c] += e;
    }
  if (a) (void) hipEventDestroy(a);
  if (b) (void) hipEventDestroy(b);
  restore();
  (void) hipStreamSynchronize(g->st);
  (void) hipFree(save);
  drop_graph(g);
  if (!ok) return fallback;
  return cand[best_of(ms, 1)[0]];
}

namespace {
struct TuneKey {
  int nx, ny, prec;
  bool operator<(const TuneKey& o) const {
    return nx != o.nx ? nx < o.nx : ny != o.ny ? ny < o.ny : prec < o.prec;
  }
};
std::map<TuneKey, SweepTune> g_tuned;
std::mutex g_tuned_mu;
}  // namespace

extern "C" int hydro_amd_grid_autotune(hydro_amd_grid* g, int reps, int* best) {
  if (!g) return fail("null grid");
  if (reps < 1) reps = 1;
  const TuneKey key{g->p.nx, g->p.ny, g->prec};
  {
    std::lock_guard<std::mutex> lk(g_tuned_mu);
    auto it = g_tuned.find(key);
    if (it != g_tuned.end() && reps > 0) {
      g->tune = it->second;
      drop_graph(g);
      if (best) {
        best[0] = g->tune.yseg; best[1] = g->tune.ywaves;
        best[2] = g->tune.xwaves; best[3] = g->tune.xiter;
      }
      return 0;
    }
  }
  HIPCHK(hipStreamSynchronize(g->st));
  if (settle(g)) return -1;
  SweepTune cur = g->tune, bt = g->tune;
  const int whole = default_step(g);  // tried against the sweeps, kept where they can't be timed
  cur.step = bt.step = 0;
  // y sweep: rows per lane (the slab height each column march covers) x
  // waves per workgroup
  // Candidates are timed in two passes, in opposite orders, and scored by
  // the sum, so a clock that drifts during tuning favours none of them.
  std::vector<SweepTune> ys;
  const long ncb = (g->p.nx + 63) / 64;
  for (int yseg : {1, 2, 4, 8, 16, 32, 64, 128, 256, 512}) {
    if (yseg > 4 * g->p.ny && yseg != 16) continue;
    // short segments are for grids with few columns (y_rows, hydro_kernels.hip)
    if (yseg < 16 && ncb * ((g->p.ny + yseg - 1) / yseg) > 16384) continue;
    for (int yw : {1, 2, 4}) {
      SweepTune t = cur;
      t.yseg = yseg;
      t.ywaves = yw;
      ys.push_back(t);
    }
  }
  std::vector<double> yms(ys.size(), 0.0);
  for (int pass = 0; pass < 2; pass++)
    for (size_t k = 0; k < ys.size(); k++) {
      const size_t c = pass ? ys.size() - 1 - k : k;
      yms[c] += time_sweep(g, 2, ys[c], reps);
    }
  double by = 1e30;
  for (size_t c = 0; c < ys.size(); c++)
    if (yms[c] < by) { by = yms[c]; bt.yseg = ys[c].yseg; bt.ywaves = ys[c].ywaves; }
  // x sweep: waves per workgroup x segments walked per wave.  Two steps run
  // one plain x sweep and one that folds the CFL maxima (odd steps), so a
  // shape is scored by the sum; the maxima go to scratch slots, not the
  // grid's.
  uint64_t* scour = nullptr;
  HIPCHK(hipMalloc(&scour, 2 * kCourSlots * sizeof(uint64_t)));
  std::vector<SweepTune> xs;
  for (int xw : {1, 2, 4}) {
    for (int xi : {1, 2, 4, 8, 16, 32}) {
      SweepTune t = cur;
      t.xwaves = xw;
      t.xiter = xi;
      xs.push_back(t);
    }
  }
  std::vector<double> xms(xs.size(), 0.0);
  for (int pass = 0; pass < 2; pass++)
    for (size_t k = 0; k < xs.size(); k++) {
      const size_t c = pass ? xs.size() - 1 - k : k;
      xms[c] += time_sweep(g, 1, xs[c], reps) + time_sweep(g, 1, xs[c], reps, scour);
    }
  double bx = 1e30;
  for (size_t c = 0; c < xs.size(); c++)
    if (xms[c] < bx) { bx = xms[c]; bt.xwaves = xs[c].xwaves; bt.xiter = xs[c].xiter; }
  (void) hipStreamSynchronize(g->st);
  (void) hipFree(scour);
  HIPCHK(hipGetLastError());
  // the three best of each direction, combined, timed as whole steps
  std::vector<SweepTune> combos;
  for (int yi : best_of(yms, 3))
    for (int xi : best_of(xms, 3)) {
      SweepTune t = ys[yi];
      t.xwaves = xs[xi].xwaves;
      t.xiter = xs[xi].xiter;
      combos.push_back(t);
    }
  if (whole) {
    SweepTune t = combos[0];
    t.step = whole;
    combos.push_back(t);
  }
  bt.step = whole;
  bt = tune_by_steps(g, combos, bt);
  HIPCHK(hipGetLastError());
  g->tune = bt;
  drop_graph(g);
  {
    std::lock_guard<std::mutex> lk(g_tuned_mu);
    g_tuned[key] = bt;
  }
  if (best) {
    best[0] = bt.yseg; best[1] = bt.ywaves; best[2] = bt.xwaves; best[3] = bt.xiter;
  }
  return 0;
}

extern "C" int hydro_amd_grid_set_tune(hydro_amd_grid* g, int yseg, int ywaves, int xwaves,
                                       int xiter) {
  if (!g) return fail("null grid");
  if (yseg < 1 || yseg > 1 << 20) return fail("yseg out of range");
  if (ywaves < 1 || ywaves > 4) return fail("ywaves must be 1..4");
  if (xwaves < 1 || xwaves > 4) return fail("xwaves must be 1..4");
  if (xiter < 1 || xiter > 4096) return fail("xiter out of range");
  g->tune.yseg = yseg;
  g->tune.ywaves = ywaves;
  g->tune.xwaves = xwaves;
  g->tune.xiter = xiter;
  g->tune.step = 0;
  drop_graph(g);
  return 0;
}

// ---- measurement support -------------------------------------------------------------

extern "C" double hydro_amd_copy_probe(long long bytes, int reps) {
  if (bytes < 8 || reps < 1) return fail("bad copy probe size");
  const long n = (long) (bytes / 8);
  double *a = nullptr, *b = nullptr;
  hipEvent_t e0, e1;
  if (hipMalloc(&a, n * 8) != hipSuccess || hipMalloc(&b, n * 8) != hipSuccess) {
    if (a) (void) hipFree(a);
    return fail("copy probe allocation failed");
  }
  (void) hipMemset(a, 0, n * 8);
  (void) hipEventCreate(&e0);
  (void) hipEventCreate(&e1);
  launch_copy_probe(a, b, n, nullptr);  // warm
  (void) hipEventRecord(e0, nullptr);
  for (int r = 0; r < reps; r++) launch_copy_probe(a, b, n, nullptr);
  (void) hipEventRecord(e1, nullptr);
  (void) hipEventSynchronize(e1);
  float ms = 0;
  (void) hipEventElapsedTime(&ms, e0, e1);
  (void) hipEventDestroy(e0);
  (void) hipEventDestroy(e1);
  (void) hipFree(a);
  (void) hipFree(b);
  // bytes moved per launch: n*8 read + n*8 written
  return 2.0 * n * 8 * reps / (ms * 1e-3) / 1e9;
}

extern "C" double hydro_amd_stream_probe(long long cells, int reps) {
  // (at most 2^36 cells: far beyond any device memory, and 2^28 workgroups)
  if (cells < 1 || cells > (1LL << 36) || reps < 1) return fail("bad stream probe size");
  const long n = (long) cells;
  StreamProbe4 p{};
  double* bufs[8] = {};
  for (int k = 0; k < 8; k++) {
    if (hipMalloc(&bufs[k], n * 8) != hipSuccess) {
      for (int j = 0; j < k; j++) (void) hipFree(bufs[j]);
      return fail("stream probe allocation failed");
    }
    if (k < 4) (void) hipMemset(bufs[k], 0, n * 8);
  }
  for (int k = 0; k < 4; k++) {
    p.in[k] = bufs[k];
    p.out[k] = bufs[4 + k];
  }
  hipEvent_t e0, e1;
  (void) hipEventCreate(&e0);
  (void) hipEventCreate(&e1);
  launch_stream_probe(p, n, nullptr);  // warm
  launch_stream_probe(p, n, nullptr);
  (void) hipEventRecord(e0, nullptr);
  for (int r = 0; r < reps; r++) launch_stream_probe(p, n, nullptr);
  (void) hipEventRecord(e1, nullptr);
  (void) hipEventSynchronize(e1);
  float ms = 0;
  (void) hipEventElapsedTime(&ms, e0, e1);
  (void) hipEventDestroy(e0);
  (void) hipEventDestroy(e1);
  for (int k = 0; k < 8; k++) (void) hipFree(bufs[k]);
  // bytes moved per launch: 4 arrays of n doubles read + 4 written
  return 64.0 * n * reps / (ms * 1e-3) / 1e9;
}

// ---- reference call surface ------------------------------------------------------------

// Globals the reference's driver expects (main.c:69, perfcnt.c); weak so a
// driver that defines them itself keeps its own.
extern "C" {
__attribute__((weak)) double functim[TIM_END];
__attribute__((weak)) long flopsAri, flopsSqr, flopsMin, flopsTra;
__attribute__((weak)) double MflopsSUM;
__attribute__((weak)) long nbFLOPS;
}

namespace {
// The GPU grid behind a surface uold is created on first GPU use
// (allocate_work_space, compute_deltat, hydro_godunov, ...), from the host
// state hydro_init built; until then the host array is the state.
struct SurfaceCtx {
  hydro_amd_grid* g = nullptr;
  size_t n = 0;  // elements of uold
  hydro_amd_params p;
  double* host = nullptr;
};
std::map<const double*, SurfaceCtx> g_surface;
const double* g_last_uold = nullptr;

[[noreturn]] void die(const char* where) {
  fprintf(stderr, "libhydro_amd: %s failed: %s\n", where, g_err.c_str());
  fflush(stderr);
  abort();
}

void ensure_grid(SurfaceCtx& c, const char* where) {
  if (c.g) return;
  c.g = hydro_amd_grid_create(&c.p);
  if (!c.g || hydro_amd_grid_upload(c.g, c.host)) die(where);
}

SurfaceCtx& ctx_of(const hydrovar_t* Hv, const char* where) {
  auto it = g_surface.find(Hv ? Hv->uold : nullptr);
  if (it == g_surface.end()) {
    fail("uold %p was not created by hydro_init", Hv ? (void*) Hv->uold : nullptr);
    die(where);
  }
  ensure_grid(it->second, where);
  return it->second;
}

SurfaceCtx& last_ctx(const char* where) {
  auto it = g_surface.find(g_last_uold);
  if (it == g_surface.end()) {
    fail("no grid: call hydro_init first");
    die(where);
  }
  ensure_grid(it->second, where);
  return it->second;
}
}  // namespace

extern "C" void hydro_init(hydroparam_t* H, hydrovar_t* Hv) {
  // HydroC99_2DMpi/Src/hydro_funcs.c:51-146 (single rank)
  H->imin = H->jmin = 0;
  H->imax = H->nx + 4;
  H->jmax = H->ny + 4;
  H->nxt = H->imax - H->imin;
  H->nyt = H->jmax - H->jmin;
  H->nxyt = H->nxt > H->nyt ? H->nxt : H->nyt;
  const size_t nxt = H->nxt, nyt = H->nyt, n = (size_t) H->nvar * nxt * nyt;
  if (H->nvar != 4) {
    fail("nvar = %d: only the 4 conservative variables are supported", H->nvar);
    die("hydro_init");
  }
  double* u = (double*) calloc(n, sizeof(double));
  if (!u) {
    fail("host allocation of %zu doubles", n);
    die("hydro_init");
  }
  auto at = [&](size_t i, size_t j, int v) -> double& { return u[i + nxt * (j + nyt * v)]; };
  for (size_t j = 2; j < nyt - 2; j++)
    for (size_t i = 2; i < nxt - 2; i++) {
      at(i, j, 0) = 1.0;
      at(i, j, 1) = 0.0;
      at(i, j, 2) = 0.0;
      at(i, j, 3) = 1e-5;
    }
  const double eb = 1.0 / H->dx / H->dx;
  if (H->testCase == 0) {
    at(nxt / 2, nyt / 2, 3) = eb;
    printf("Centered test case : %d %d\n", (int) (nxt / 2), (int) (nyt / 2));
  } else if (H->testCase == 1) {
    at(2, 2, 3) = eb;
    printf("Lower corner test case : %d %d\n", 2, 2);
  } else if (H->testCase == 2) {
    for (size_t j = 2; j < nyt; j++) at(2, j, 3) = eb;
    printf("SOD tube test case\n");
  } else {
    printf("Test case not implemented -- aborting !\n");
    fflush(stdout);
    abort();
  }
  fflush(stdout);
  SurfaceCtx c;
  hydro_amd_params_from_surface(H, &c.p);
  if (validate(&c.p)) die("hydro_init");
  c.n = n;
  c.host = u;
  Hv->uold = u;
  g_surface[u] = c;
  g_last_uold = u;
}

extern "C" void hydro_finish(const hydroparam_t H, hydrovar_t* Hv) {
  (void) H;
  auto it = g_surface.find(Hv ? Hv->uold : nullptr);
  if (it != g_surface.end()) {
    hydro_amd_grid_destroy(it->second.g);
    g_surface.erase(it);
  }
  if (Hv && Hv->uold == g_last_uold) g_last_uold = nullptr;
  if (Hv) {
    free(Hv->uold);
    Hv->uold = nullptr;
  }
}

extern "C" void allocate_work_space(int ngrid, const hydroparam_t H, hydrowork_t* Hw,
                                    hydrovarwork_t* Hvw) {
  // The GPU grid already holds its ping-pong buffer; no host work arrays.
  (void) ngrid;
  (void) H;
  (void) last_ctx("allocate_work_space");
  if (Hw) memset(Hw, 0, sizeof(*Hw));
  if (Hvw) memset(Hvw, 0, sizeof(*Hvw));
}

extern "C" void deallocate_work_space(int ngrid, const hydroparam_t H, hydrowork_t* Hw,
                                      hydrovarwork_t* Hvw) {
  (void) ngrid;
  (void) H;
  if (Hw) memset(Hw, 0, sizeof(*Hw));
  if (Hvw) memset(Hvw, 0, sizeof(*Hvw));
}

extern "C" void compute_deltat_init_mem(const hydroparam_t H, hydrowork_t* Hw,
                                        hydrovarwork_t* Hvw) {
  (void) H;
  (void) last_ctx("compute_deltat_init_mem");
  if (Hw) memset(Hw, 0, sizeof(*Hw));
  if (Hvw) memset(Hvw, 0, sizeof(*Hvw));
}

extern "C" void compute_deltat_clean_mem(const hydroparam_t H, hydrowork_t* Hw,
                                         hydrovarwork_t* Hvw) {
  (void) H;
  if (Hw) memset(Hw, 0, sizeof(*Hw));
  if (Hvw) memset(Hvw, 0, sizeof(*Hvw));
}

extern "C" void compute_deltat(real_t* dt, const hydroparam_t H, hydrowork_t* Hw,
                               hydrovar_t* Hv, hydrovarwork_t* Hvw) {
  (void) H;
  (void) Hw;
  (void) Hvw;
  SurfaceCtx& c = ctx_of(Hv, "compute_deltat");
  if (hydro_amd_grid_compute_deltat(c.g, dt)) die("compute_deltat");
}

extern "C" void hydro_godunov(int idim, real_t dt, const hydroparam_t H, hydrovar_t* Hv,
                              hydrowork_t* Hw, hydrovarwork_t* Hvw) {
  (void) Hw;
  (void) Hvw;
  SurfaceCtx& c = ctx_of(Hv, "hydro_godunov");
  // main.c:254: dt is recomputed at the start of every even step, i.e. right
  // after an odd step; fold that step's CFL maxima into its last sweep.
  if (godunov_impl(c.g, idim, dt, (H.nstep % 2) == 1)) die("hydro_godunov");
}

extern "C" void make_boundary(int idim, const hydroparam_t H, hydrovar_t* Hv) {
  (void) H;
  SurfaceCtx& c = ctx_of(Hv, "make_boundary");
  if (hydro_amd_grid_make_boundary(c.g, idim)) die("make_boundary");
}

extern "C" int hydro_amd_sync_host(hydrovar_t* Hv) {
  auto it = g_surface.find(Hv ? Hv->uold : nullptr);
  if (it == g_surface.end()) return fail("uold was not created by hydro_init");
  if (!it->second.g) return 0;  // no GPU state yet: the host array is current
  return hydro_amd_grid_download(it->second.g, Hv->uold);
}

extern "C" hydro_amd_grid* hydro_amd_surface_grid(hydrovar_t* Hv) {
  auto it = g_surface.find(Hv ? Hv->uold : nullptr);
  if (it == g_surface.end()) return nullptr;
  ensure_grid(it->second, "hydro_amd_surface_grid");
  return it->second.g;
}

extern "C" int hydro_amd_sync_device(hydrovar_t* Hv) {
  auto it = g_surface.find(Hv ? Hv->uold : nullptr);
  if (it == g_surface.end()) return fail("uold was not created by hydro_init");
  if (!it->second.g) return 0;  // the grid will be built from the host array
  return hydro_amd_grid_upload(it->second.g, Hv->uold);
}
