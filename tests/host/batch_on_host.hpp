// The kernels of a batch as hydro_batch.cpp calls them, for checks on the CPU: none
// runs, but the run controls that are set on the device are set.
#pragma once
#include <vector>

#include "../../hydro_amd/csrc/hydro_batch.hpp"

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
