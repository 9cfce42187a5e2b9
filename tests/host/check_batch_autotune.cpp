// A batch's autotuner whose HIP calls fail one after the other: the run controls
// on the device are as before afterwards, and the batch can be tuned again.
#include "hip_on_host.hpp"

#include <stdio.h>
#include <string.h>

#include <string>
#include <vector>

#include "../../hydro_amd/csrc/hydro_batch.hpp"
#include "../../include/hydro_amd.h"

using namespace hydro;

static std::vector<RunCtl*> ctls;  // of the instances, as they were added

namespace hydro {
void launch_batch_set_ctl(RunCtl* c, double t, double dt, double tend, int nstep, int nstepmax,
                          int active, hipStream_t) {
  *c = RunCtl();
  c->t = t;
  c->dt = dt;
  c->tend = tend;
  c->nstep = nstep;
  c->nstepmax = nstepmax;
  c->active = active;
  ctls.push_back(c);
}
// no kernel runs
void launch_zero_u64(uint64_t*, long, hipStream_t) {}
void launch_batch_tasks(const BList*, int, BTask*, hipStream_t) {}
void launch_batch_march(const InstDev<float>*, const BTask*, int, int, hipStream_t) {}
void launch_batch_march_fast(const InstDev<double>*, const BTask*, int, int, hipStream_t) {}
void launch_batch_sweep_fast(int, const InstDev<double>*, const BTask*, int, int, int, bool, int,
                             int, hipStream_t) {}
template <typename S>
void launch_batch_sweep(int, const InstDev<S>*, const BTask*, int, int, int, bool, int, int,
                        hipStream_t) {}
template <typename S>
void launch_batch_boundary(const InstDev<S>*, const BTask*, int, int, hipStream_t) {}
template <typename S>
void launch_batch_courant(const InstDev<S>*, const int*, int, hipStream_t) {}
template <typename S>
void launch_batch_ctl(const InstDev<S>*, const int*, int, bool, hipStream_t) {}
template <typename S>
void launch_init(const GridGeom&, GridView<S>, GridView<S>, int, int, int, double, hipStream_t) {}
#define INST(S)                                                                                  \
  template void launch_batch_sweep<S>(int, const InstDev<S>*, const BTask*, int, int, int, bool, \
                                      int, int, hipStream_t);                                    \
  template void launch_batch_boundary<S>(const InstDev<S>*, const BTask*, int, int, hipStream_t); \
  template void launch_batch_courant<S>(const InstDev<S>*, const int*, int, hipStream_t);        \
  template void launch_batch_ctl<S>(const InstDev<S>*, const int*, int, bool, hipStream_t);      \
  template void launch_init<S>(const GridGeom&, GridView<S>, GridView<S>, int, int, int, double, \
                               hipStream_t);
INST(double)
INST(float)
int stage_d2h(void*, int, const void*, int, long, long, long, hipStream_t) { return 0; }
int stage_h2d(void*, int, long, const void*, int, long, long, hipStream_t) { return 0; }
}  // namespace hydro

int main() {
  hydro_amd_batch* b = hydro_amd_batch_create(HYDRO_AMD_FP64, 0);
  if (!b) return 1;
  for (int n : {70, 130}) {
    hydro_amd_params p = {};
    p.nx = p.ny = n;
    p.dx = 1.0;
    p.gamma = 1.4;
    p.slope_type = 1.0;
    p.scheme = 1;
    p.tend = 1e30;
    p.nstepmax = 100;
    p.precision = HYDRO_AMD_FP64;
    if (hydro_amd_batch_add(b, &p) < 0) return 1;
  }
  auto intact = [&] {
    for (const RunCtl* c : ctls)
      if (c->active || c->nstep || c->t != 0.0 || c->dt != 0.0) return false;
    return true;
  };
  int failed = 0;
  for (int k = 1;; k++) {
    // (the last blocking copy of a call is the one that puts the controls back)
    int call = 0;
    std::string which;
    onhost::refuse = [&](const char* name) {
      if (++call != k) return false;
      which = name;
      return true;
    };
    const int rc = hydro_amd_batch_autotune(b, 1, nullptr);
    onhost::refuse = nullptr;
    if (which.empty()) {  // fewer than k calls: the tuner met no failure
      if (rc || !intact()) return 2;
      break;
    }
    if (!intact()) {
      // the restoration itself was refused: an error, nothing less
      if (which == "hipMemcpy" && rc) {
        for (RunCtl* c : ctls) {
          c->active = 0;
          c->dt = 0.0;
        }
        continue;
      }
      printf("call %d (%s) refused: the controls were left forced\n", k, which.c_str());
      return 3;
    }
    failed++;
  }
  hydro_amd_batch_destroy(b);
  printf("%d refusals\n", failed);
  return failed > 10 ? 0 : 4;
}
