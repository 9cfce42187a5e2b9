// The staged copies (stage_h2d, stage_d2h) against HIP calls that fail; the
// argument names the check.
#include "hip_on_host.hpp"

#include <stdio.h>
#include <string.h>

#include <string>
#include <vector>

#include "../../hydro_amd/csrc/hydro_kernels.hpp"

using namespace hydro;

// A state of `rows` x `width` doubles to a device of desz-byte elements and back.
static bool round_trip(hipStream_t st, long width, long rows, int desz) {
  const long pitch = (width + 31) / 32 * 32;
  std::vector<double> u((size_t) width * rows), back(u.size());
  for (size_t k = 0; k < u.size(); k++) u[k] = (double) (k % 8191) / 64.0;  // exact as float too
  std::vector<char> dev((size_t) pitch * rows * desz);
  if (stage_h2d(dev.data(), desz, pitch, u.data(), 8, width, rows, st)) return false;
  if (stage_d2h(back.data(), 8, dev.data(), desz, pitch, width, rows, st)) return false;
  return u == back;
}

// one slab, many slabs of many threads, rows wider than a slab
static const long kShapes[3][2] = {{7, 28}, {1001, 3000}, {300000, 12}};

static int no_pinned_memory() {
  hipStream_t st;
  if (hipStreamCreateWithFlags(&st, 0) != hipSuccess) return 1;
  for (const char* what : {"hipHostMalloc", "hipEventCreateWithFlags"}) {
    onhost::refuse = [&](const char* name) { return !strcmp(name, what); };
    for (auto& s : kShapes)
      for (int desz : {8, 4})
        if (!round_trip(st, s[0], s[1], desz)) {
          printf("%s refused: %ld x %ld of %d bytes\n", what, s[0], s[1], desz);
          return 2;
        }
  }
  onhost::refuse = nullptr;  // had again: used again
  for (auto& s : kShapes)
    if (!round_trip(st, s[0], s[1], 8)) return 3;
  return 0;
}

// Streams of two devices in turn, whichever device is current.
static int devices() {
  hipStream_t st[2];
  for (int d : {0, 1}) {
    (void) hipSetDevice(d);
    if (hipStreamCreateWithFlags(&st[d], 0) != hipSuccess) return 1;
  }
  for (int k = 0; k < 8; k++) {
    const int of = k & 1, current = (k >> 1) & 1;
    (void) hipSetDevice(current);
    for (auto& s : kShapes)
      if (!round_trip(st[of], s[0], s[1], 8)) {
        printf("device %d's stream with device %d current\n", of, current);
        return 2;
      }
    int now = -1;
    (void) hipGetDevice(&now);
    if (now != current) return 3;
  }
  return 0;
}

int main(int argc, char** argv) {
  const std::string which = argc > 1 ? argv[1] : "";
  if (which == "no_pinned_memory") return no_pinned_memory();
  if (which == "devices") return devices();
  return 99;
}
