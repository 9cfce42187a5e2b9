// The predictor of the range-gated FP64 kernels (trace_tail_scaled) against the
// reference's order of operations (trace_tail), bit for bit, on cells that pass the
// gate.  Compiled by g++: the device functions become plain ones, one lane a wave.
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdio.h>
#include <string.h>

#include <random>

#undef __device__
#undef __host__
#undef __forceinline__
#define __device__
#define __host__
#define __forceinline__ inline
// (the two functions need the first alone; the others are for the rest of the header)
#define __builtin_amdgcn_ballot_w64(p) ((unsigned long long) (p))
#define __builtin_amdgcn_rcp(x) (1.0 / (x))
#define __builtin_amdgcn_rsq(x) (1.0 / sqrt(x))
#define __builtin_amdgcn_rcpf(x) (1.0f / (x))
#define __builtin_amdgcn_rsqf(x) (1.0f / sqrtf(x))
#define __builtin_amdgcn_sqrtf(x) sqrtf(x)
#define __builtin_amdgcn_fmed3f(x, y, z) fmaxf(fminf(x, y), fminf(fmaxf(x, y), z))
#define __builtin_amdgcn_div_fixup(q, b, a) (q)
static inline int __double2hiint(double x) {
  long long b;
  memcpy(&b, &x, sizeof b);
  return (int) (b >> 32);
}
#include "../../hydro_amd/csrc/hydro_numerics.hpp"

using namespace hydro;

static std::mt19937_64 rng(7);
static double uniform(double a, double b) {
  return std::uniform_real_distribution<double>(a, b)(rng);
}
static bool one_in(int n) { return rng() % n == 0; }
// a zero of either sign, or up to 2^hi and down to 2^lo
static double signed_value(double lo, double hi) {
  if (one_in(4)) return one_in(2) ? 0.0 : -0.0;
  return (one_in(2) ? 1 : -1) * exp2(uniform(lo, hi));
}
// a neighbour's difference: of either zero, of the last bits, of any size
static double slope(double v, double lo, double hi) {
  if (one_in(3)) return one_in(2) ? 0.0 : -0.0;
  if (one_in(2)) return nextafter(v, one_in(2) ? INFINITY : -INFINITY) - v;
  return signed_value(lo, hi);
}

int main() {
  long differ = 0, zeros = 0;
  for (long n = 0; n < 4000000; n++) {
    Q4<double> q, dq;
    const double span = one_in(2) ? 3 : 40;  // a flow's values, or the whole range
    q.r = exp2(uniform(-span, span));
    q.p = exp2(uniform(-span, span));
    q.u = signed_value(-2 * span, 2 * span);
    q.v = signed_value(-2 * span, 2 * span);
    dq.r = slope(q.r, -span, span);
    dq.p = slope(q.p, -span, span);
    // (velocities are quotients: their differences are not finer than 2^-134)
    dq.u = q.u == 0.0 ? slope(1.0, -span, span) : slope(q.u, -2 * span, 2 * span);
    dq.v = q.v == 0.0 ? slope(1.0, -span, span) : slope(q.v, -2 * span, 2 * span);
    const double cc = sqrt(1.4 * q.p / q.r), csq = cc * cc;
    const TraceK<double> k = make_tracek<double>(exp2(uniform(-12, 3)), 1 + (int) (n % 3));
    Q4<double> a[2], b[2];
    const double dprcc = dq.p / (q.r * cc), a0r = dq.r - dq.p / csq;
    trace_tail<double>(q, dq, cc, csq, q.r / cc, cc / q.r, dprcc, a0r, k, a[0], a[1]);
    trace_tail_scaled<double>(q, dq, cc, csq, q.r / cc, cc / q.r, dprcc, a0r, k, b[0], b[1]);
    zeros += a[0].u == 0.0;
    if (memcmp(a, b, sizeof a) != 0) {
      if (differ++ < 3)
        printf("u %a p %a du %a dp %a: u- %a %a, u+ %a %a\n", q.u, q.p, dq.u, dq.p, a[0].u, b[0].u,
               a[1].u, b[1].u);
    }
  }
  printf("%ld cells differ, %ld with a zero velocity at the face\n", differ, zeros);
  return differ || zeros < 1000;
}
