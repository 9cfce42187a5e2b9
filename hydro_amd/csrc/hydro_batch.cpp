// Batch of independent grids (instances) advanced per launch -- the C ABI
// hydro_amd_batch_* of include/hydro_amd.h.  Host bookkeeping only; the
// kernels are in hydro_batch.hip.
//
// Instances are admitted against an HBM budget; their state buffers come from
// the stream-ordered allocator (hipMallocAsync / hipFreeAsync on the batch's
// stream), so admitting or retiring an instance never synchronises the
// device.  The per-step work is two phase task tables (P and Q) built from
// each instance's step parity, for each of two groups of the instances, which
// run beside each other on streams of their own; a small load is one group, whose
// two steps (P,Q then Q,P) are captured once as a HIP graph and replayed until the
// set of instances changes.
#include <hip/hip_runtime.h>

#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "../../include/hydro_amd.h"
#include "hydro_batch.hpp"

using namespace hydro;

extern "C" int hydro_amd_set_error(const char* fmt, ...);  // hydro_capi.cpp

#define BCHK(call)                                                                         \
  do {                                                                                     \
    hipError_t e_ = (call);                                                                \
    if (e_ != hipSuccess) return hydro_amd_set_error("%s: %s", #call, hipGetErrorString(e_)); \
  } while (0)

namespace {
constexpr long kOrigin = 30;  // same row origin as single grids (hydro_capi.cpp)
constexpr int kMaxInst = 8192;
constexpr int kGroups = 2;        // instances advanced side by side (split_load)
constexpr long kSplitSegs = 4000;  // least x segments of a load in two groups

struct Inst {
  bool live = false;
  hydro_amd_params p;
  GridGeom g;
  long plane = 0;
  void* mem[2] = {nullptr, nullptr};
  long long bytes = 0;
  bool need_cour = false;  // CFL maxima of the initial state still to compute
  // the state is in mem[base] after step n0; where steps are whole (march > 0,
  // their rows a wave), it changes buffers with each
  int base = 0, n0 = 0, march = 0;
};

// Instances that are advanced together, launch by launch, on one stream.
struct Group {
  // task lists, in this order: Px Py (phase P: x of even-step instances, y of
  // odd ones), Qx Qy (phase Q: the other sweep of each), PB QB (ghost fills)
  int n[6] = {0, 0, 0, 0, 0, 0};
  int off[6] = {0, 0, 0, 0, 0, 0};
  int n1[6] = {0, 0, 0, 0, 0, 0};  // leading tasks of slope_type == 1 instances
  int first = 0, nids = 0;         // its part of the live ids
};
}  // namespace

struct hydro_amd_batch {
  int prec;
  size_t esz;
  long long budget, used = 0;
  hipStream_t st = nullptr;
  std::vector<Inst> inst;
  RunCtl* ctl = nullptr;         // kMaxInst run controls
  uint64_t* cour = nullptr;      // kMaxInst * 2 * kInstSlots
  void* idev = nullptr;          // InstDev<S>[kMaxInst]
  BTask* tasks = nullptr;        // the groups' task lists
  int task_cap = 0;
  int* ids = nullptr;            // live ids (device)
  int* cids = nullptr;           // ids needing a CFL pass (device)
  Group grp[kGroups];
  int ngrp = 1;
  hipStream_t st2 = nullptr;     // group 1's (group 0: st); made when first needed
  hipEvent_t fork = nullptr, join = nullptr;
  BList* lists = nullptr;          // what the task tables are written from (device)
  int nids = 0;
  int maxid = -1;                // highest live id
  bool dirty = true;
  bool flip = false;             // next step runs Q before P
  hipGraphExec_t gexec[2] = {nullptr, nullptr};
  BatchTune tune = {1, 0, 0};
  int xiter = 1, yseg = 1, march = 0;  // the shape in use (rebuild)
  bool fresh = false;            // no step has been queued since hctl was read
  std::vector<int> live_ids;
  RunCtl* hctl = nullptr;        // pinned host copy of the run controls
  void* hidev = nullptr;         // pinned host copy of the instance array
};

// FP64 storage (the FP64 and FP64 fast forms) rather than FP32.
static bool dbl(const hydro_amd_batch* b) { return b->prec != HYDRO_AMD_MIXED; }

static void drop_graphs(hydro_amd_batch* b) {
  for (auto& g : b->gexec)
    if (g) {
      (void) hipGraphExecDestroy(g);
      g = nullptr;
    }
}

extern "C" void hydro_amd_batch_destroy(hydro_amd_batch* b) {
  if (!b) return;
  if (b->st) (void) hipStreamSynchronize(b->st);
  if (b->st2) (void) hipStreamSynchronize(b->st2);
  drop_graphs(b);
  for (auto& in : b->inst)
    for (auto& m : in.mem)
      if (m) (void) hipFree(m);
  for (void* p : {(void*) b->ctl, (void*) b->cour, b->idev, (void*) b->tasks, (void*) b->ids,
                  (void*) b->cids, (void*) b->lists})
    if (p) (void) hipFree(p);
  if (b->hctl) (void) hipHostFree(b->hctl);
  if (b->hidev) (void) hipHostFree(b->hidev);
  if (b->st) (void) hipStreamDestroy(b->st);
  if (b->st2) (void) hipStreamDestroy(b->st2);
  for (auto e : {b->fork, b->join})
    if (e) (void) hipEventDestroy(e);
  delete b;
}

extern "C" hydro_amd_batch* hydro_amd_batch_create(int precision, long long budget_bytes) {
  if (precision != HYDRO_AMD_FP64 && precision != HYDRO_AMD_MIXED &&
      precision != HYDRO_AMD_FP64_FAST) {
    hydro_amd_set_error("unknown precision %d", precision);
    return nullptr;
  }
  hydro_amd_batch* b = new hydro_amd_batch();
  b->prec = precision;
  b->esz = dbl(b) ? 8 : 4;
  b->budget = budget_bytes > 0 ? budget_bytes : (1LL << 62);
  b->inst.resize(kMaxInst);
  const size_t isz = dbl(b) ? sizeof(InstDev<double>) : sizeof(InstDev<float>);
  bool ok = hipStreamCreateWithFlags(&b->st, hipStreamNonBlocking) == hipSuccess &&
            hipMalloc(&b->ctl, sizeof(RunCtl) * kMaxInst) == hipSuccess &&
            hipMalloc(&b->cour, sizeof(uint64_t) * 2 * kInstSlots * kMaxInst) == hipSuccess &&
            hipMalloc(&b->idev, isz * kMaxInst) == hipSuccess &&
            hipMalloc(&b->ids, sizeof(int) * kMaxInst) == hipSuccess &&
            hipMalloc(&b->cids, sizeof(int) * kMaxInst) == hipSuccess &&
            hipMalloc(&b->lists, sizeof(BList) * 4 * kMaxInst) == hipSuccess &&
            hipHostMalloc((void**) &b->hctl, sizeof(RunCtl) * kMaxInst) == hipSuccess &&
            hipHostMalloc(&b->hidev, isz * kMaxInst) == hipSuccess;
  if (!ok) {
    hydro_amd_set_error("batch allocation failed");
    hydro_amd_batch_destroy(b);
    return nullptr;
  }
  launch_zero_u64(b->cour, 2L * kInstSlots * kMaxInst, b->st);
  // keep freed instance memory in the pool instead of returning it
  hipMemPool_t pool;
  int dev = 0;
  if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetDefaultMemPool(&pool, dev) == hipSuccess) {
    uint64_t thr = ~0ULL;
    (void) hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &thr);
  }
  if (hipStreamSynchronize(b->st) != hipSuccess) {
    hydro_amd_set_error("batch setup failed");
    hydro_amd_batch_destroy(b);
    return nullptr;
  }
  return b;
}

static long long inst_bytes(const hydro_amd_batch* b, const GridGeom& g, long plane) {
  (void) g;
  return 2LL * (4 * plane + kOrigin + 64) * (long long) b->esz;
}

extern "C" long long hydro_amd_batch_bytes_needed(const hydro_amd_batch* b, int nx, int ny) {
  if (!b || nx < 1 || ny < 1) return -1;
  GridGeom g;
  g.nx = nx;
  g.ny = ny;
  g.pitch = ((long) nx + 4 + 31) / 32 * 32;
  return inst_bytes(b, g, g.pitch * (ny + 4));
}

extern "C" long long hydro_amd_batch_bytes_used(const hydro_amd_batch* b) {
  return b ? b->used : -1;
}

template <typename S>
static GridView<S> view_of(const hydro_amd_batch* b, const Inst& in, int k) {
  GridView<S> v;
  S* base = (S*) in.mem[in.base ^ k] + kOrigin;  // k = 0: the state's after step n0
  for (int q = 0; q < 4; q++) v.p[q] = base + q * in.plane;
  (void) b;
  return v;
}

// A new initial state is (being) put into both buffers and the run control reset.
static void reset_run(hydro_amd_batch* b, int id) {
  Inst& in = b->inst[id];
  in.base = in.n0 = in.march = 0;
  in.need_cour = true;
  RunCtl& c = b->hctl[id];
  c = RunCtl();
  c.tend = in.p.tend;
  c.nstepmax = in.p.nstepmax;
  launch_zero_u64(b->cour + (size_t) id * 2 * kInstSlots, 2 * kInstSlots, b->st);
  launch_batch_set_ctl(b->ctl + id, 0.0, 0.0, in.p.tend, 0, in.p.nstepmax, 0, b->st);
  b->dirty = true;  // parity back to even
}

extern "C" int hydro_amd_batch_add(hydro_amd_batch* b, const hydro_amd_params* p) {
  if (!b || !p) return hydro_amd_set_error("null argument");
  if (p->nx < 1 || p->ny < 1 || !(p->dx > 0) || !(p->gamma > 1) || p->scheme < 1 ||
      p->scheme > 3 || p->niter_riemann < 0)
    return hydro_amd_set_error("invalid instance parameters");
  if ((long) ((p->nx + kXSeg - 1) / kXSeg) * p->ny > (1L << 30))
    return hydro_amd_set_error("instance too large");
  if (p->precision != b->prec) return hydro_amd_set_error("instance precision differs from batch");
  int id = -1;
  for (int k = 0; k < kMaxInst; k++)
    if (!b->inst[k].live) {
      id = k;
      break;
    }
  if (id < 0) return hydro_amd_set_error("batch full (%d instances)", kMaxInst);
  Inst& in = b->inst[id];
  in.p = *p;
  in.g.nx = p->nx;
  in.g.ny = p->ny;
  in.g.pitch = ((long) p->nx + 4 + 31) / 32 * 32;
  in.plane = in.g.pitch * (p->ny + 4);
  in.bytes = inst_bytes(b, in.g, in.plane);
  if (b->used + in.bytes > b->budget)
    return hydro_amd_set_error("over budget: %lld + %lld > %lld bytes", b->used, in.bytes,
                               b->budget);
  const size_t sz = (size_t) in.bytes / 2;
  for (int k = 0; k < 2; k++) {
    if (hipMallocAsync(&in.mem[k], sz, b->st) != hipSuccess) {
      if (k == 1) (void) hipFreeAsync(in.mem[0], b->st);
      in.mem[0] = in.mem[1] = nullptr;
      return hydro_amd_set_error("device allocation of %zu bytes failed", sz);
    }
    BCHK(hipMemsetAsync(in.mem[k], 0, sz, b->st));
  }
  in.live = true;
  b->used += in.bytes;
  reset_run(b, id);
  BCHK(hipGetLastError());
  return id;
}

static Inst* live(hydro_amd_batch* b, int id) {
  if (!b || id < 0 || id >= kMaxInst || !b->inst[id].live) {
    hydro_amd_set_error("no live instance %d", id);
    return nullptr;
  }
  return &b->inst[id];
}

extern "C" int hydro_amd_batch_remove(hydro_amd_batch* b, int id) {
  Inst* in = live(b, id);
  if (!in) return -1;
  for (auto& m : in->mem) {
    if (m) BCHK(hipFreeAsync(m, b->st));
    m = nullptr;
  }
  in->live = false;
  b->used -= in->bytes;
  b->dirty = true;
  return 0;
}

static int init_inst(hydro_amd_batch* b, int id, int bx, int by0, int by1, double e) {
  Inst* in = live(b, id);
  if (!in) return -1;
  reset_run(b, id);
  if (dbl(b))
    launch_init<double>(in->g, view_of<double>(b, *in, 0), view_of<double>(b, *in, 1), bx, by0,
                        by1, e, b->st);
  else
    launch_init<float>(in->g, view_of<float>(b, *in, 0), view_of<float>(b, *in, 1), bx, by0, by1,
                       e, b->st);
  BCHK(hipGetLastError());
  return 0;
}

extern "C" int hydro_amd_batch_init(hydro_amd_batch* b, int id, int testcase) {
  Inst* in = live(b, id);
  if (!in) return -1;
  const int nxt = in->p.nx + 4, nyt = in->p.ny + 4;
  const double eb = 1.0 / in->p.dx / in->p.dx;  // hydro_funcs.c:92
  switch (testcase) {
    case 0: return init_inst(b, id, nxt / 2, nyt / 2, nyt / 2 + 1, eb);
    case 1: return init_inst(b, id, 2, 2, 3, eb);
    case 2: return init_inst(b, id, 2, 2, nyt, eb);
    default: return hydro_amd_set_error("testcase %d not implemented", testcase);
  }
}

extern "C" int hydro_amd_batch_init_blast(hydro_amd_batch* b, int id, int bx, int by, double e) {
  Inst* in = live(b, id);
  if (!in) return -1;
  if (bx < 0 || by < 0 || bx >= in->p.nx || by >= in->p.ny)
    return hydro_amd_set_error("blast cell (%d, %d) outside %dx%d", bx, by, in->p.nx, in->p.ny);
  return init_inst(b, id, bx + 2, by + 2, by + 3, e);
}

// Reads the run controls of ids [0, maxid] into the pinned host copy.
static int read_ctl(hydro_amd_batch* b) {
  if (b->maxid < 0) return 0;
  BCHK(hipMemcpyAsync(b->hctl, b->ctl, sizeof(RunCtl) * (b->maxid + 1), hipMemcpyDeviceToHost,
                      b->st));
  BCHK(hipStreamSynchronize(b->st));
  b->fresh = true;
  return 0;
}

// The buffer that an instance's state is in, -1 on error.  Waits for the
// batch's stream if steps of the instance may have been queued since its run
// control was read.
static int state_buf(hydro_amd_batch* b, int id) {
  const Inst& in = b->inst[id];
  if (!in.march) return in.base;
  const RunCtl& c = b->hctl[id];
  const bool ended = c.fault || !(c.t < c.tend) || c.nstep >= c.nstepmax;
  if (!b->fresh && !ended && read_ctl(b)) return -1;
  return in.base ^ ((c.nstep - in.n0) & 1);
}

extern "C" int hydro_amd_batch_download(hydro_amd_batch* b, int id, double* u) {
  Inst* in = live(b, id);
  if (!in || !u) return in ? hydro_amd_set_error("null argument") : -1;
  const long nxt = in->p.nx + 4, rows = 4L * (in->p.ny + 4);
  const int k = state_buf(b, id);
  if (k < 0) return -1;
  const void* src = (const char*) in->mem[k] + kOrigin * b->esz;
  return stage_d2h(u, 8, src, (int) b->esz, in->g.pitch, nxt, rows, b->st) ? -1 : 0;
}

// Where an instance's state lives: `rows` rows of `width` elements of `esz`
// bytes, `pitch` elements apart, starting at *src (layout [4][ny+4][nx+4]).
int hydro_amd_batch_raw_view(hydro_amd_batch* b, int id, const void** src, long* pitch,
                             long* width, long* rows, int* esz) {
  Inst* in = live(b, id);
  if (!in) return -1;
  const int k = state_buf(b, id);
  if (k < 0) return -1;
  *src = (const char*) in->mem[k] + kOrigin * b->esz;
  *pitch = in->g.pitch;
  *width = in->p.nx + 4;
  *rows = 4L * (in->p.ny + 4);
  *esz = (int) b->esz;
  return 0;
}

// Copies an instance's state as stored (element size 8 or 4), layout
// [4][ny+4][nx+4]; for the serving loop (no conversion on its critical path).
// The copy is queued on `st` (the batch's stream if null), so it can run
// beside kernels on the batch's stream that do not touch this instance.
int hydro_amd_batch_download_raw(hydro_amd_batch* b, int id, void* dst, int* elem_size,
                                 hipStream_t st) {
  Inst* in = live(b, id);
  if (!in || !dst) return in ? hydro_amd_set_error("null argument") : -1;
  const long nxt = in->p.nx + 4, rows = 4L * (in->p.ny + 4);
  const size_t w = b->esz;
  const int k = state_buf(b, id);
  if (k < 0) return -1;
  const void* src = (const char*) in->mem[k] + kOrigin * w;
  if (stage_d2h(dst, (int) w, src, (int) w, in->g.pitch, nxt, rows, st ? st : b->st)) return -1;
  if (elem_size) *elem_size = (int) w;
  return 0;
}

static int rebuild(hydro_amd_batch* b);

// Whether each listed live instance's interior state is finite: one CFL pass
// over it (k_batch_courant) into its slots, whose maxima are NaN or inf
// exactly when some cell's density, momenta or energy is (a NaN orders above
// +inf in the slots' integer maximum).  Meant for instances whose run has
// ended -- it overwrites their CFL slots -- such as the serving loop's
// finished requests.  Waits for the batch's stream.
int hydro_amd_batch_finite(hydro_amd_batch* b, const int* ids, int n, int* finite) {
  if (!b || n < 0 || (n > 0 && (!ids || !finite))) return hydro_amd_set_error("bad argument");
  if (n == 0) return 0;
  if (n > kMaxInst) return hydro_amd_set_error("too many instances");
  BCHK(hipStreamSynchronize(b->st));
  if (b->dirty && rebuild(b)) return -1;
  for (int k = 0; k < n; k++) {
    if (!live(b, ids[k])) return -1;
    launch_zero_u64(b->cour + (size_t) ids[k] * 2 * kInstSlots, 2 * kInstSlots, b->st);
  }
  BCHK(hipMemcpyAsync(b->cids, ids, sizeof(int) * n, hipMemcpyHostToDevice, b->st));
  if (dbl(b))
    launch_batch_courant<double>((const InstDev<double>*) b->idev, b->cids, n, b->st);
  else
    launch_batch_courant<float>((const InstDev<float>*) b->idev, b->cids, n, b->st);
  std::vector<uint64_t> slots((size_t) n * 2 * kInstSlots);
  for (int k = 0; k < n; k++)
    BCHK(hipMemcpyAsync(slots.data() + (size_t) k * 2 * kInstSlots,
                        b->cour + (size_t) ids[k] * 2 * kInstSlots,
                        sizeof(uint64_t) * 2 * kInstSlots, hipMemcpyDeviceToHost, b->st));
  BCHK(hipStreamSynchronize(b->st));  // (also: `ids` and `slots` outlive the copies)
  for (int k = 0; k < n; k++) {
    int ok = 1;
    for (int q = 0; q < 2 * kInstSlots; q++) {
      double v;
      memcpy(&v, &slots[(size_t) k * 2 * kInstSlots + q], sizeof v);
      if (!std::isfinite(v)) ok = 0;
    }
    finite[k] = ok;
  }
  return 0;
}

extern "C" int hydro_amd_batch_upload(hydro_amd_batch* b, int id, const double* u) {
  Inst* in = live(b, id);
  if (!in || !u) return in ? hydro_amd_set_error("null argument") : -1;
  const long nxt = in->p.nx + 4, rows = 4L * (in->p.ny + 4);
  void* dst = (char*) in->mem[0] + kOrigin * b->esz;
  if (stage_h2d(dst, (int) b->esz, in->g.pitch, u, 8, nxt, rows, b->st)) return -1;
  BCHK(hipMemcpyAsync(in->mem[1], in->mem[0], (size_t) in->bytes / 2, hipMemcpyDeviceToDevice,
                      b->st));
  reset_run(b, id);
  return 0;
}

// ---- task tables -------------------------------------------------------------------

static long x_segments(const hydro_amd_params& p) {
  return (long) ((p.nx + kXSeg - 1) / kXSeg) * p.ny;
}

// The sweeps form the ghosts of all but very narrow instances.
static bool folds_ghosts(const Inst& in) {
  return in.p.nx >= kGhostMin && in.p.ny >= kGhostMin;
}

// Task shape by the load.  As in a single grid's y sweep (y_rows,
// hydro_kernels.hip), a task's fixed cost and the unevenness that long tasks
// leave at a launch's end balance at a length proportional to the square root
// of the work: sqrt(wave rows) / 28 rows, sqrt(segments) / 50 segments (with
// one chain of launches, before split_load, half the segments).  The best of
// all shapes tried, x segments / y rows: 4 grids of 64-100 a side 1 / 1; 12 of
// 64-256 1 / 2-3; 2 of 900-1024 3-4 / 4; 30 of 150-500 4 / 6-8; 60 of 64-1024
// 8-12 / 16-24; 300 of 64-1024 and 24 of 128-4096 8-32 / 32-64.  A step took
// with fixed shapes (2 or 4 waves of 8 or 32 segments, 32 or 64 rows) in one
// chain and takes with these: 12 small grids, mixed, 138 and 24 us; 30, fast,
// 156 and 94; 60, FP64, 701 and 565; 24 of up to 4096, mixed, 1.21 and 1.12 ms.
// Large loads of the fast and mixed forms take whole steps instead (step_march;
// for the line's reasons see step_rows, hydro_capi.cpp), in segments that fill the
// 4096 waves the GPU holds twice, of at most 64 rows.  A step, sweeps and whole, the
// best segment in brackets, of blasts in loads of so many wave rows: fast 46000 (30
// grids of 150-500) 91 and 93 us (8), 68000 (40 of 150-550) 129 and 124 (8), 167000
// (60 of 64-1024) 291 and 255 (20), 818000 (24 of 128-4096) 1365 and 1137 (64),
// 967000 (300 of 64-1024) 1625 and 1352 (64); with flows that move everywhere 46000
// 134 and 138, 68000 190 and 195, 167000 420 and 384.  Mixed 49000 67 and 65 (8),
// 219000 224 and 209 (20-32), 1.07e6 1068 and 956 (96), 1.21e6 1136 and 1021 (64);
// moving 167000 246 and 238, 818000 959 and 876.
static void shape_by_load(hydro_amd_batch* b) {
  long segs = 0, wrows = 0, mrows = 0;
  bool fold = true;
  for (int id : b->live_ids) {
    const hydro_amd_params& p = b->inst[id].p;
    segs += x_segments(p);
    wrows += (long) ((p.nx + 63) / 64) * p.ny;
    mrows += (long) ((p.nx + 59) / 60) * p.ny;
    fold = fold && folds_ghosts(b->inst[id]) && p.nx < kMarchWidest;
  }
  auto root = [](long n, double by, int most) {
    return std::max(1, std::min(most, (int) (std::sqrt((double) n) / by + 0.5)));
  };
  b->xiter = b->tune.xiter > 0 ? b->tune.xiter : root(segs, 50, 16);
  b->yseg = b->tune.yseg > 0 ? b->tune.yseg : root(wrows, 28, 40);
  const long line = b->prec == HYDRO_AMD_FP64_FAST ? 80000 : 150000;
  b->march = b->prec != HYDRO_AMD_FP64 && fold && b->tune.xiter <= 0 && mrows >= line
                 ? (int) std::min(64L, mrows / 8192)
                 : 0;
}

// Rows per wave in an instance's y tasks: the instance's rows split evenly
// over as few row groups (of waves x b->yseg rows) as cover them, so no
// group ends with a short segment that pays the full halo.
static int inst_yseg(const hydro_amd_batch* b, int ny) {
  const long W = b->tune.waves, per = W * b->yseg;
  const long nrg = (ny + per - 1) / per;
  return (int) ((ny + W * nrg - 1) / (W * nrg));
}

template <typename S>
static InstDev<S> inst_dev(hydro_amd_batch* b, int id) {
  const Inst& in = b->inst[id];
  InstDev<S> d;
  d.g = in.g;
  d.ph = make_phys<S>(in.p.gamma, in.p.smallr, in.p.smallc, in.p.slope_type, in.p.niter_riemann,
                      in.p.iorder, in.p.scheme);
  d.dx = in.p.dx;
  d.cf = in.p.courant_factor;
  d.smallc = in.p.smallc;
  d.buf[0] = view_of<S>(b, in, 0);
  d.buf[1] = view_of<S>(b, in, 1);
  d.ctl = b->ctl + id;
  d.cour = b->cour + (size_t) id * 2 * kInstSlots;
  d.bl = in.p.boundary_left;
  d.br = in.p.boundary_right;
  d.bd = in.p.boundary_down;
  d.bu = in.p.boundary_up;
  d.fold = folds_ghosts(in);
  d.nseg = (in.p.nx + kXSeg - 1) / kXSeg;
  d.yseg = inst_yseg(b, in.p.ny);
  d.march = in.march;
  d.n0 = in.n0;
  return d;
}

// An instance's x (kind 1) or y (kind 2) tasks.
static BList sweep_tasks(const hydro_amd_batch* b, int id, int kind) {
  const hydro_amd_params& p = b->inst[id].p;
  const long W = b->tune.waves;
  BList l{id, kind, 0, 0, 0, 0};
  if (kind == 1) {
    const long per = W * b->xiter, tot = x_segments(p);
    l.per = (int) per;
    l.count = (int) ((tot + per - 1) / per);
  } else {
    const long rows = W * inst_yseg(b, p.ny);
    l.ncb = (p.nx + 63) / 64;
    l.count = (int) (l.ncb * ((p.ny + rows - 1) / rows));
  }
  return l;
}

// An instance's whole steps.
static BList march_tasks(const hydro_amd_batch* b, int id) {
  const Inst& in = b->inst[id];
  BList l{id, 3, 0, 0, 0, 0};
  l.ncb = (in.p.nx + 59) / 60;
  l.count = (int) (l.ncb * ((in.p.ny + in.march - 1) / in.march));
  return l;
}

// Ghost fills of one narrow instance in direction idim, kBoundaryChunk
// (line, var) pairs per task so a large instance spreads over many workgroups.
static BList ghost_tasks(const hydro_amd_batch* b, int id, int idim) {
  const hydro_amd_params& p = b->inst[id].p;
  const long tot = 4L * (idim == 1 ? p.ny : p.nx);
  return BList{id, idim, 0, (int) ((tot + kBoundaryChunk - 1) / kBoundaryChunk), kBoundaryChunk, 0};
}

// Parts a load into two groups of about the same work, each with a
// stream of its own: an instance waits only for its own sweeps, so where one
// group's launch runs out of tasks the other's fills the GPU (alone, the y
// sweeps of 60 grids of 64-1024 a side kept 3.05 of 4 waves a SIMD busy and
// issued 75 % of the time; the x sweeps 4.35 of 5, 89 %), and longer tasks pay.  A
// step, one group and two, each at its best shape: 12 grids of 64-256, mixed, 30
// and 24 us; 30 of 150-500, fast, 115 and 94; 60 of 64-1024, FP64 640 and 558,
// fast 400 and 373, mixed 238 and 218; 24 of 128-4096, mixed, 1146 and 1117.
// Three groups: the same within 1 %.  Below kSplitSegs the ten launches of a
// step of two groups are what the step costs (17-19 us on the host): 4 grids of
// 64-100 a side, 625 segments, mixed, 13.2 us as one group's graph and 18.6; 12
// of 64-256, 5500 segments, 20.9 and 18.9, FP64 38.0 and 29.4.
static int split_load(hydro_amd_batch* b) {
  auto work = [&](int id) { return (long) b->inst[id].p.nx * b->inst[id].p.ny; };
  for (auto& gr : b->grp) gr = Group();
  b->grp[0].nids = (int) b->live_ids.size();
  long segs = 0;
  for (int id : b->live_ids) segs += x_segments(b->inst[id].p);
  b->ngrp = b->grp[0].nids > 1 && segs >= kSplitSegs ? 2 : 1;
  if (b->ngrp == 1) return 0;
  if (!b->st2) BCHK(hipStreamCreateWithFlags(&b->st2, hipStreamNonBlocking));
  if (!b->fork) BCHK(hipEventCreateWithFlags(&b->fork, hipEventDisableTiming));
  if (!b->join) BCHK(hipEventCreateWithFlags(&b->join, hipEventDisableTiming));
  // the largest first, each to the group with the least so far
  std::stable_sort(b->live_ids.begin(), b->live_ids.end(),
                   [&](int x, int y) { return work(x) > work(y); });
  std::vector<int> part[kGroups];
  long sum[kGroups] = {0, 0};
  for (int id : b->live_ids) {
    const int q = sum[1] < sum[0] ? 1 : 0;
    part[q].push_back(id);
    sum[q] += work(id);
  }
  b->live_ids = part[0];
  b->live_ids.insert(b->live_ids.end(), part[1].begin(), part[1].end());
  b->grp[0].nids = b->grp[1].first = (int) part[0].size();
  b->grp[1].nids = (int) part[1].size();
  return 0;
}

// Rebuilds the device instance array and the phase tables from the current
// live set and their step parities (the stream must be idle; the batch's device
// the current one).
static int rebuild_tables(hydro_amd_batch* b) {
  drop_graphs(b);
  b->live_ids.clear();
  b->maxid = -1;
  for (int k = 0; k < kMaxInst; k++)
    if (b->inst[k].live) {
      b->live_ids.push_back(k);
      b->maxid = k;
    }
  if (read_ctl(b)) return -1;
  shape_by_load(b);
  for (int id : b->live_ids) {
    Inst& in = b->inst[id];
    in.base = state_buf(b, id);
    in.n0 = b->hctl[id].nstep;
    // (even segments)
    const int nseg = b->march ? (in.p.ny + b->march - 1) / b->march : 1;
    in.march = b->march ? (in.p.ny + nseg - 1) / nseg : 0;
  }
  if (split_load(b)) return -1;
  std::vector<BList> all;
  long need = 0;
  for (int q = 0; q < b->ngrp; q++) {
    Group& gr = b->grp[q];
    // each sweep list: tasks of slope_type == 1 instances first (their own
    // kernel variant), then the others
    std::vector<BList> L[6][2];
    for (int m = gr.first; m < gr.first + gr.nids; m++) {
      const int id = b->live_ids[m];
      const bool even = (b->hctl[id].nstep % 2) == 0;
      const int gen = b->inst[id].p.slope_type == 1.0 ? 0 : 1;
      if (b->march) {
        L[0][gen].push_back(march_tasks(b, id));
        continue;
      }
      L[even ? 0 : 2][gen].push_back(sweep_tasks(b, id, 1));
      L[even ? 3 : 1][gen].push_back(sweep_tasks(b, id, 2));
      if (!folds_ghosts(b->inst[id])) {
        L[4][0].push_back(ghost_tasks(b, id, even ? 1 : 2));
        L[5][0].push_back(ghost_tasks(b, id, even ? 2 : 1));
      }
    }
    for (int k = 0; k < 6; k++) {
      gr.off[k] = (int) need;
      for (auto& part : L[k]) {
        for (BList& l : part) {
          l.first = (int) need;
          need += l.count;
          all.push_back(l);
        }
        if (&part == &L[k][0]) gr.n1[k] = (int) (need - gr.off[k]);
      }
      gr.n[k] = (int) (need - gr.off[k]);
    }
  }
  if (need > (1L << 30)) return hydro_amd_set_error("batch too large: %ld tasks", need);
  b->nids = (int) b->live_ids.size();
  if (need > b->task_cap) {
    if (b->tasks) BCHK(hipFree(b->tasks));
    b->tasks = nullptr;
    b->task_cap = 0;
    const long cap = std::max(need + need / 2, 4096L);
    BCHK(hipMalloc(&b->tasks, sizeof(BTask) * cap));
    b->task_cap = (int) cap;
  }
  // (the tables are written on the device: a large load has 1e5 tasks)
  if (!all.empty()) {
    BCHK(hipMemcpy(b->lists, all.data(), sizeof(BList) * all.size(), hipMemcpyHostToDevice));
    launch_batch_tasks(b->lists, (int) all.size(), b->tasks, b->st);
    BCHK(hipGetLastError());
  }
  if (b->nids)
    BCHK(hipMemcpy(b->ids, b->live_ids.data(), sizeof(int) * b->nids, hipMemcpyHostToDevice));
  if (b->maxid >= 0) {
    if (dbl(b)) {
      auto* v = (InstDev<double>*) b->hidev;
      for (int id : b->live_ids) v[id] = inst_dev<double>(b, id);
      BCHK(hipMemcpy(b->idev, v, sizeof(v[0]) * (b->maxid + 1), hipMemcpyHostToDevice));
    } else {
      auto* v = (InstDev<float>*) b->hidev;
      for (int id : b->live_ids) v[id] = inst_dev<float>(b, id);
      BCHK(hipMemcpy(b->idev, v, sizeof(v[0]) * (b->maxid + 1), hipMemcpyHostToDevice));
    }
  }
  b->flip = false;
  b->dirty = false;
  return 0;
}

// The same whichever device is current: what it makes on the way (task tables, the
// second group's stream and its events) is the batch's device's.
static int rebuild(hydro_amd_batch* b) {
  int current = 0, own = 0;
  BCHK(hipGetDevice(&current));
  BCHK(hipStreamGetDevice(b->st, &own));
  if (own == current) return rebuild_tables(b);
  BCHK(hipSetDevice(own));
  const int rc = rebuild_tables(b);
  (void) hipSetDevice(current);
  return rc;
}

static hipStream_t stream_of(const hydro_amd_batch* b, int q) { return q == 0 ? b->st : b->st2; }

// The sweeps of group q's task list k (kind 1: x, 2: y) in the batch's
// arithmetic form, reading buffer `phase`.
template <typename S>
static void sweep_list(hydro_amd_batch* b, int q, int kind, int k, int phase, bool ghosts) {
  const InstDev<S>* I = (const InstDev<S>*) b->idev;
  const Group& gr = b->grp[q];
  if constexpr (sizeof(S) == 8) {
    if (b->prec == HYDRO_AMD_FP64_FAST) {
      launch_batch_sweep_fast(kind, I, b->tasks + gr.off[k], gr.n[k], gr.n1[k], phase, ghosts,
                              b->tune.waves, b->xiter, stream_of(b, q));
      return;
    }
  }
  launch_batch_sweep<S>(kind, I, b->tasks + gr.off[k], gr.n[k], gr.n1[k], phase, ghosts,
                        b->tune.waves, b->xiter, stream_of(b, q));
}

// One phase of a group: the ghost fills of its narrow instances, then its x
// tasks and its y tasks.
template <typename S>
static void enq_phase(hydro_amd_batch* b, int q, int which, int phase) {
  const int x = which == 0 ? 0 : 2, y = x + 1, bd = which == 0 ? 4 : 5;
  launch_batch_boundary<S>((const InstDev<S>*) b->idev, b->tasks + b->grp[q].off[bd],
                           b->grp[q].n[bd], phase, stream_of(b, q));
  sweep_list<S>(b, q, 1, x, phase, true);
  sweep_list<S>(b, q, 2, y, phase, true);
}

template <typename S>
static void enq_ctl(hydro_amd_batch* b, int q, bool begin) {
  launch_batch_ctl<S>((const InstDev<S>*) b->idev, b->ids + b->grp[q].first, b->grp[q].nids,
                      begin, stream_of(b, q));
}

template <typename S>
static void enq_step_t(hydro_amd_batch* b, int q, bool flip) {
  enq_ctl<S>(b, q, true);
  if (b->march) {
    const Group& gr = b->grp[q];
    const BTask* t = b->tasks + gr.off[0];
    if constexpr (sizeof(S) == 8)
      launch_batch_march_fast((const InstDev<S>*) b->idev, t, gr.n[0], gr.n1[0], stream_of(b, q));
    else
      launch_batch_march((const InstDev<S>*) b->idev, t, gr.n[0], gr.n1[0], stream_of(b, q));
    return;
  }
  enq_phase<S>(b, q, flip ? 1 : 0, 0);
  enq_phase<S>(b, q, flip ? 0 : 1, 1);
}

// Closes the last step of a run (each step closes the one before it).
static void enq_close(hydro_amd_batch* b, int q) {
  if (dbl(b)) enq_ctl<double>(b, q, false);
  else enq_ctl<float>(b, q, false);
}

static void enq_step(hydro_amd_batch* b, int q, bool flip) {
  if (dbl(b)) enq_step_t<double>(b, q, flip);
  else enq_step_t<float>(b, q, flip);
}

// The second group's stream starts after what is queued on the batch's stream.
static int fork_groups(hydro_amd_batch* b) {
  if (b->ngrp == 1) return 0;
  BCHK(hipEventRecord(b->fork, b->st));
  BCHK(hipStreamWaitEvent(b->st2, b->fork, 0));
  return 0;
}

// What the batch's stream is given next starts after both groups' work.
static int join_groups(hydro_amd_batch* b) {
  if (b->ngrp == 1) return 0;
  if (hipEventRecord(b->join, b->st2) != hipSuccess ||
      hipStreamWaitEvent(b->st, b->join, 0) != hipSuccess)
    BCHK(hipStreamSynchronize(b->st2));
  return 0;
}

static int pending_courant(hydro_amd_batch* b) {
  std::vector<int> need;
  for (int id : b->live_ids)
    if (b->inst[id].need_cour) {
      need.push_back(id);
      b->inst[id].need_cour = false;
    }
  if (need.empty()) return 0;
  BCHK(hipMemcpyAsync(b->cids, need.data(), sizeof(int) * need.size(), hipMemcpyHostToDevice,
                      b->st));
  if (dbl(b))
    launch_batch_courant<double>((const InstDev<double>*) b->idev, b->cids, (int) need.size(),
                                 b->st);
  else
    launch_batch_courant<float>((const InstDev<float>*) b->idev, b->cids, (int) need.size(),
                                b->st);
  // `need` must outlive the async copy
  BCHK(hipStreamSynchronize(b->st));
  return 0;
}

static int get_graph(hydro_amd_batch* b, int f) {
  if (b->gexec[f]) return 0;
  hipGraph_t graph;
  BCHK(hipStreamBeginCapture(b->st, hipStreamCaptureModeThreadLocal));
  enq_step(b, 0, f != 0);
  enq_step(b, 0, f == 0);
  hipError_t e = hipStreamEndCapture(b->st, &graph);
  if (e != hipSuccess) return hydro_amd_set_error("graph capture: %s", hipGetErrorString(e));
  e = hipGraphInstantiate(&b->gexec[f], graph, nullptr, nullptr, 0);
  (void) hipGraphDestroy(graph);
  if (e != hipSuccess) {
    b->gexec[f] = nullptr;
    return hydro_amd_set_error("graph instantiate: %s", hipGetErrorString(e));
  }
  return 0;
}

extern "C" int hydro_amd_batch_run_async(hydro_amd_batch* b, int steps) {
  if (!b) return hydro_amd_set_error("null batch");
  if (steps < 0) return hydro_amd_set_error("steps < 0");
  if (b->dirty) {
    BCHK(hipStreamSynchronize(b->st));
    if (rebuild(b)) return -1;
  }
  if (b->nids == 0 || steps == 0) return 0;
  if (pending_courant(b)) return -1;
  b->fresh = false;
  if (b->ngrp > 1) {
    // launch by launch: each group's run is one chain on its stream, met again
    // only at the run's end (two steps of both groups as one graph: 12 grids of
    // 64-256, mixed, 43 us a step against 26; 60 of 64-1024, fast, 411 / 402; two
    // steps of each group as a graph on its own stream: half the host's time, 0.9 ms
    // for 100 steps of those 12 instead of 2.0, but they take 2.69 ms instead of 2.50)
    if (fork_groups(b)) return -1;
    for (int k = 0; k < steps; k++) {
      for (int q = 0; q < b->ngrp; q++) enq_step(b, q, b->flip);
      b->flip = !b->flip;
    }
    for (int q = 0; q < b->ngrp; q++) enq_close(b, q);
    if (join_groups(b)) return -1;
    BCHK(hipGetLastError());
    return 0;
  }
  int left = steps;
  if (left >= 2) {
    const int f = b->flip ? 1 : 0;
    if (get_graph(b, f)) return -1;
    for (; left >= 2; left -= 2) BCHK(hipGraphLaunch(b->gexec[f], b->st));
  }
  if (left == 1) {
    enq_step(b, 0, b->flip);
    b->flip = !b->flip;
  }
  enq_close(b, 0);
  BCHK(hipGetLastError());
  return 0;
}

extern "C" int hydro_amd_batch_sync(hydro_amd_batch* b) {
  if (!b) return hydro_amd_set_error("null batch");
  BCHK(hipStreamSynchronize(b->st));
  return 0;
}

extern "C" int hydro_amd_batch_run(hydro_amd_batch* b, int steps) {
  if (hydro_amd_batch_run_async(b, steps)) return -1;
  return hydro_amd_batch_sync(b);
}

extern "C" int hydro_amd_batch_query(hydro_amd_batch* b, int* ids, double* t, int* nstep,
                                     double* dt, int* active, int cap) {
  if (!b) return hydro_amd_set_error("null batch");
  BCHK(hipStreamSynchronize(b->st));
  int top = -1;
  for (int k = 0; k < kMaxInst; k++)
    if (b->inst[k].live) top = k;
  b->maxid = top > b->maxid ? top : b->maxid;
  if (read_ctl(b)) return -1;
  int n = 0;
  for (int k = 0; k <= top; k++) {
    if (!b->inst[k].live) continue;
    if (n < cap) {
      const RunCtl& c = b->hctl[k];
      // a step opens only if t < tend && nstep < nstepmax (main.c:244);
      // -1: stopped at a dt that was not positive and finite
      const int more = c.fault ? -1 : ((c.t < c.tend) && (c.nstep < c.nstepmax));
      if (ids) ids[n] = k;
      if (t) t[n] = c.t;
      if (nstep) nstep[n] = c.nstep;
      if (dt) dt[n] = c.dt;
      if (active) active[n] = more;
    }
    n++;
  }
  return n;
}

extern "C" int hydro_amd_batch_set_tune(hydro_amd_batch* b, int waves, int xiter, int yseg) {
  if (!b) return hydro_amd_set_error("null batch");
  if (waves < 1 || waves > 4 || xiter < 1 || xiter > 256 || yseg < 1 || yseg > 1 << 16)
    return hydro_amd_set_error("tune out of range");
  BCHK(hipStreamSynchronize(b->st));
  b->tune = BatchTune{waves, xiter, yseg};
  b->dirty = true;
  return 0;
}

// Times the phase sweeps of the current live set for one launch shape.  The
// run controls are saved, forced active for the timing (sweeps of phase 0
// read buffer 0 and write only buffer 1, the scratch), then restored: the
// state and the run are unchanged.
extern "C" int hydro_amd_batch_autotune(hydro_amd_batch* b, int reps, int* best) {
  if (!b) return hydro_amd_set_error("null batch");
  if (reps < 1) reps = 1;
  BCHK(hipStreamSynchronize(b->st));
  if (b->dirty && rebuild(b)) return -1;
  if (b->nids == 0) return hydro_amd_set_error("empty batch");
  if (b->march) {  // faster than the sweeps at their best shape (shape_by_load)
    if (best) {
      best[0] = b->tune.waves;
      best[1] = b->xiter;
      best[2] = b->yseg;
    }
    return 0;
  }
  const int nc = b->maxid + 1;
  std::vector<RunCtl> saved(nc);
  BCHK(hipMemcpy(saved.data(), b->ctl, sizeof(RunCtl) * nc, hipMemcpyDeviceToHost));
  std::vector<RunCtl> forced = saved;
  for (int id : b->live_ids) {
    forced[id].active = 1;
    forced[id].fault = 0;
    if (!(forced[id].dt > 0)) forced[id].dt = 1e-12;
  }
  const BatchTune keep = b->tune;
  BatchTune bt = keep;
  double bms = 1e30;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  hipError_t err = hipEventCreate(&e0);
  if (err == hipSuccess) err = hipEventCreate(&e1);
  // (from here to their restoration nothing returns: a control left active would
  // be closed as a step that ran)
  if (err == hipSuccess)
    err = hipMemcpy(b->ctl, forced.data(), sizeof(RunCtl) * nc, hipMemcpyHostToDevice);
  // around the shape that goes by the load
  b->tune = BatchTune{1, 0, 0};
  shape_by_load(b);
  const int rx = b->xiter, ry = b->yseg;
  for (int w : {1, 2, 4})
    for (int xi : {std::max(1, rx / 2), rx, 2 * rx})  // (none once err is set)
      for (int ys : {std::max(1, ry / 2), ry, 2 * ry}) {
        if (err != hipSuccess || hydro_amd_batch_set_tune(b, w, xi, ys) || rebuild(b)) break;
        for (int r = -1; r < reps; r++) {  // r = -1 warms up
          if (r == 0) (void) hipEventRecord(e0, b->st);
          // every x and y list at phase 0: reads buffer 0, writes buffer 1 only
          if (fork_groups(b)) break;
          for (int k = 0; k < 4; k++) {
            const int kind = (k % 2 == 0) ? 1 : 2;
            for (int q = 0; q < b->ngrp; q++)
              if (dbl(b)) sweep_list<double>(b, q, kind, k, 0, false);
              else sweep_list<float>(b, q, kind, k, 0, false);
          }
          if (join_groups(b)) break;
        }
        (void) hipEventRecord(e1, b->st);
        float ms = 1e30f;
        if (hipEventSynchronize(e1) == hipSuccess) (void) hipEventElapsedTime(&ms, e0, e1);
        if (ms < bms) {
          bms = ms;
          bt = b->tune;
        }
      }
  for (hipEvent_t e : {e0, e1})
    if (e) (void) hipEventDestroy(e);
  const hipError_t back =
      hipMemcpy(b->ctl, saved.data(), sizeof(RunCtl) * nc, hipMemcpyHostToDevice);
  if (err == hipSuccess) err = back;
  if (err != hipSuccess || bms == 1e30) {  // nothing could be timed
    b->tune = keep;
    b->dirty = true;
    BCHK(err);
  } else if (hydro_amd_batch_set_tune(b, bt.waves, bt.xiter, bt.yseg)) {
    return -1;
  }
  if (best) {
    best[0] = bt.waves;
    best[1] = bt.xiter > 0 ? bt.xiter : rx;
    best[2] = bt.yseg > 0 ? bt.yseg : ry;
  }
  return 0;
}
