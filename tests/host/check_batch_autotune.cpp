// A batch's autotuner whose HIP calls fail one after the other: the run controls
// on the device are as before afterwards, and the batch can be tuned again.
#include "batch_on_host.hpp"
#include "hip_on_host.hpp"

#include <stdio.h>
#include <string.h>

#include <string>
#include <vector>

#include "../../include/hydro_amd.h"

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
