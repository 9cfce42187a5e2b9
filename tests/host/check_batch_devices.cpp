// A batch on one device used while another is current: what it makes as its load
// grows (the second group's stream and events) belongs to its own device.
#include "batch_on_host.hpp"
#include "hip_on_host.hpp"

#include <stdio.h>

#include "../../include/hydro_amd.h"

static bool add(hydro_amd_batch* b, int n) {
  hydro_amd_params p = {};
  p.nx = p.ny = n;
  p.dx = 1.0;
  p.gamma = 1.4;
  p.slope_type = 1.0;
  p.scheme = 1;
  p.tend = 1e30;
  p.nstepmax = 100;
  p.precision = HYDRO_AMD_FP64;
  return hydro_amd_batch_add(b, &p) >= 0;
}

int main() {
  (void) hipSetDevice(0);
  hydro_amd_batch* b = hydro_amd_batch_create(HYDRO_AMD_FP64, 0);
  if (!b || !add(b, 70) || hydro_amd_batch_run_async(b, 1)) return 1;  // one group
  (void) hipSetDevice(1);
  if (!add(b, 900) || !add(b, 800)) return 1;  // two
  if (hydro_amd_batch_run_async(b, 1)) {
    printf("the batch's run failed with another device current\n");
    return 2;
  }
  int now = -1;
  (void) hipGetDevice(&now);
  hydro_amd_batch_destroy(b);
  return now == 1 ? 0 : 3;
}
