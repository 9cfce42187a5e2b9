// The staged copies (stage_h2d, stage_d2h) against HIP calls that fail; the
// argument names the check.
#include "hip_on_host.hpp"

#include <stdio.h>
#include <string.h>

#include <chrono>
#include <future>
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

// A copy whose stream has work queued before it holds up no other thread's copy.
static int busy_stream(bool up) {
  hipStream_t busy, idle;
  if (hipStreamCreateWithFlags(&busy, 0) != hipSuccess ||
      hipStreamCreateWithFlags(&idle, 0) != hipSuccess)
    return 1;
  std::vector<double> host(64 * 64), dev(64 * 64);
  std::promise<void> reached;
  bool told = false;
  // (the copy has come as far as its stream's queued work)
  onhost::refuse = [&](const char* name) {
    if (!told && (!strcmp(name, "hipStreamSynchronize") || !strcmp(name, "hipEventSynchronize"))) {
      told = true;
      reached.set_value();
    }
    return false;
  };
  onhost::hold(busy, true);
  auto first = std::async(std::launch::async, [&] {
    return up ? stage_h2d(dev.data(), 8, 64, host.data(), 8, 64, 64, busy)
              : stage_d2h(host.data(), 8, dev.data(), 8, 64, 64, 64, busy);
  });
  reached.get_future().wait();
  auto second = std::async(std::launch::async, [&] { return round_trip(idle, 100, 80, 8); });
  const bool free = second.wait_for(std::chrono::seconds(10)) == std::future_status::ready;
  const bool waiting = first.wait_for(std::chrono::seconds(0)) != std::future_status::ready;
  onhost::hold(busy, false);
  if (!free || !waiting || !second.get() || first.get()) {
    printf("up %d: other thread free %d, the copy waits %d\n", up, free, waiting);
    return 2;
  }
  return 0;
}

int main(int argc, char** argv) {
  const std::string which = argc > 1 ? argv[1] : "";
  if (which == "no_pinned_memory") return no_pinned_memory();
  if (which == "devices") return devices();
  if (which == "busy_upload") return busy_stream(true);
  if (which == "busy_download") return busy_stream(false);
  return 99;
}
