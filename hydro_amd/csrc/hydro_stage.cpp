// Copies of pitched state between host and device through pinned staging
// buffers.
//
// A hipMemcpy2D to or from pageable host memory goes row by row (a 1021x767
// upload ran at 0.9 GB/s); between pinned memory and the device it runs at the
// link's rate (55-57 GB/s at every row length from 2 to 64 KB).  What is left
// is the host's own copy between the pinned buffers and the caller's array,
// with the FP32 <-> FP64 conversion on the way: one thread does 14 GB/s into
// fresh pages (5 GB/s where they are 4 KB ones), eight 30, so a large state is
// cut into slabs of rows that up to kLanes threads carry, each through two
// buffers of its own, the DMA of one beside the host copy of the other.
// 8192x8192 FP64 download: 153 ms with one thread, 54 with eight; 1021x767
// upload 28.4 ms through hipMemcpy2D, 0.8 so.  Where no pinned memory can be had,
// the rows go through hipMemcpy2D all the same.
#include <hip/hip_runtime.h>

#include <pthread.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <memory>
#include <mutex>
#include <new>
#include <thread>

#include "hydro_kernels.hpp"

extern "C" int hydro_amd_set_error(const char* fmt, ...);  // hydro_capi.cpp

namespace hydro {
namespace {
// Per buffer.  The link idles about 10 us between two DMA calls: 8192x8192
// FP64 in 72 ms with slabs of 1 MB, 54 with 2, 46 with 4; with 2 MB the memory
// that the process keeps pinned is 32 MB.  (To give memory back with the last
// grid or batch made programs that make one after the other pay 0.2-0.4 ms
// for each.)
constexpr size_t kSlabBytes = 2u << 20;
constexpr int kLanes = 8;  // threads, two buffers each
// Host bytes that are worth a thread (starting one takes about 17 us; 0.4 to
// 1.5 MB measured alike from 700x500 up).
constexpr size_t kThreadBytes = 3u << 19;

struct Lane {
  void* buf[2] = {nullptr, nullptr};
  hipEvent_t ev[2] = {nullptr, nullptr};
  int dev = -1;  // the events' device: a stream records only its own device's
};
struct Stage {
  std::mutex mu;  // one staged copy at a time per process
  Lane lane[kLanes];
};
Stage g_stage;

void drop_events(Lane& l) {
  for (hipEvent_t& e : l.ev) {
    if (e) (void) hipEventDestroy(e);
    e = nullptr;
  }
  l.dev = -1;
}

// The lane's buffers, and events of the current device `dev`.
bool lane_ready(Lane& l, int dev) {
  if (!l.buf[0]) {
    if (hipHostMalloc(&l.buf[0], 2 * kSlabBytes, hipHostMallocPortable) != hipSuccess) {
      l.buf[0] = nullptr;
      return false;
    }
    l.buf[1] = (char*) l.buf[0] + kSlabBytes;  // one allocation
  }
  if (l.dev == dev) return true;
  drop_events(l);
  if (hipEventCreateWithFlags(&l.ev[0], hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&l.ev[1], hipEventDisableTiming) != hipSuccess) {
    drop_events(l);
    return false;
  }
  l.dev = dev;
  return true;
}

// Up to n lanes for copies on device `dev`, the current one; how many there are
// (0: no pinned memory).
int lanes_for(int n, int dev) {
  int k = 0;
  while (k < n && lane_ready(g_stage.lane[k], dev)) k++;
  if (k < n) (void) hipGetLastError();
  return k;
}

// n elements of sesz bytes to desz bytes (4 or 8 each).
void convert(void* dst, int desz, const void* src, int sesz, size_t n) {
  if (desz == sesz) {
    memcpy(dst, src, n * (size_t) sesz);
  } else if (desz == 8) {
    const float* s = (const float*) src;
    double* d = (double*) dst;
    for (size_t k = 0; k < n; k++) d[k] = s[k];
  } else {
    const double* s = (const double*) src;
    float* d = (float*) dst;
    for (size_t k = 0; k < n; k++) d[k] = (float) s[k];
  }
}

// Runs work(k) for k = 0..n-1, k = 0 on the calling thread and the others on
// threads of their own, where they can be had.  Their stacks are small, so that
// the C library keeps them for the next call: eight of the usual 8 MB are
// more than it keeps, and were they unmapped each time, the next device
// allocations of the process took 0.3-0.7 ms longer.
template <typename F>
struct Share {
  const F* work;
  int k;
  static void* run(void* p) {
    const Share* s = (const Share*) p;
    (*s->work)(s->k);
    return nullptr;
  }
};
template <typename F>
void on_threads(int n, const F& work) {
  pthread_t th[kLanes];
  Share<F> share[kLanes];
  int started = 0;
  pthread_attr_t attr;
  if (n > 1 && pthread_attr_init(&attr) == 0) {
    (void) pthread_attr_setstacksize(&attr, 1u << 20);
    for (int k = 1; k < n; k++) {
      share[k] = Share<F>{&work, k};
      if (pthread_create(&th[k], &attr, Share<F>::run, &share[k]) != 0) break;
      started = k;
    }
    (void) pthread_attr_destroy(&attr);
  }
  work(0);
  for (int k = started + 1; k < n; k++) work(k);
  for (int k = 1; k <= started; k++) (void) pthread_join(th[k], nullptr);
}

int thread_count(size_t bytes) {
  static const int cpus = std::max(1, (int) std::thread::hardware_concurrency());
  const size_t want = std::max<size_t>(1, bytes / kThreadBytes);
  return (int) std::min<size_t>(want, (size_t) std::min(cpus, kLanes));
}

// One block of columns, at most a slab wide: `rows` rows of `width` elements;
// host rows hpitch elements apart, device rows dpitch.
struct Block {
  char* host;
  int hesz;
  long hpitch;
  char* dev;
  int desz;
  long dpitch, width, rows;
  hipStream_t st;
};

// `nr` host rows from row r0 on into (up) or out of a buffer of such rows.
void host_rows(const Block& b, bool up, void* buf, long r0, long nr) {
  const size_t row_bytes = (size_t) b.width * b.desz;
  char* h = b.host + (size_t) r0 * b.hpitch * b.hesz;
  if (b.hpitch == b.width) {
    const size_t m = (size_t) nr * b.width;
    if (up) convert(buf, b.desz, h, b.hesz, m);
    else convert(h, b.hesz, buf, b.desz, m);
    return;
  }
  for (long r = 0; r < nr; r++) {
    char* hr = h + (size_t) r * b.hpitch * b.hesz;
    char* br = (char*) buf + (size_t) r * row_bytes;
    if (up) convert(br, b.desz, hr, b.hesz, b.width);
    else convert(hr, b.hesz, br, b.desz, b.width);
  }
}

// Queues the copy of `nr` rows between the device and host memory at `buf`,
// whose rows are `pitch` bytes apart.
hipError_t copy_rows(const Block& b, bool up, void* buf, size_t pitch, long r0, long nr) {
  const size_t w = (size_t) b.width * b.desz, dp = (size_t) b.dpitch * b.desz;
  char* d = b.dev + (size_t) r0 * dp;
  return up ? hipMemcpy2DAsync(d, dp, buf, pitch, w, nr, hipMemcpyHostToDevice, b.st)
            : hipMemcpy2DAsync(buf, pitch, d, dp, w, nr, hipMemcpyDeviceToHost, b.st);
}

int copy_error(bool up) {
  return hydro_amd_set_error("%s copy failed", up ? "host-to-device" : "device-to-host");
}

// Without pinned memory: straight between the caller's array and the device, or
// slab by slab through pageable memory where the elements are converted.
int copy_pageable(const Block& b, bool up) {
  const size_t row_bytes = (size_t) b.width * b.desz;
  if (b.hesz == b.desz) {
    if (copy_rows(b, up, b.host, (size_t) b.hpitch * b.hesz, 0, b.rows) != hipSuccess ||
        hipStreamSynchronize(b.st) != hipSuccess)
      return copy_error(up);
    return 0;
  }
  const long per = std::max(1L, std::min((long) (kSlabBytes / row_bytes), b.rows));
  std::unique_ptr<char[]> buf(new (std::nothrow) char[(size_t) per * row_bytes]);
  if (!buf) return hydro_amd_set_error("staging allocation failed");
  for (long r0 = 0; r0 < b.rows; r0 += per) {
    const long nr = std::min(per, b.rows - r0);
    if (up) host_rows(b, up, buf.get(), r0, nr);
    if (copy_rows(b, up, buf.get(), row_bytes, r0, nr) != hipSuccess ||
        hipStreamSynchronize(b.st) != hipSuccess)
      return copy_error(up);
    if (!up) host_rows(b, up, buf.get(), r0, nr);
  }
  return 0;
}

// dev: the stream's device, the current one.
int copy_block(const Block& b, int dev, bool up) {
  const size_t row_bytes = (size_t) b.width * b.desz;
  int n = lanes_for(thread_count((size_t) b.width * b.rows * b.hesz), dev);
  if (n < 1) return copy_pageable(b, up);
  // slabs small enough that every thread has two or more
  const long per = std::max(1L, std::min((long) (kSlabBytes / row_bytes),
                                         (b.rows + 2L * n - 1) / (2L * n)));
  const long nslab = (b.rows + per - 1) / per;
  n = (int) std::min<long>(n, nslab);
  std::atomic<int> bad{0};
  // slab c to or from buffer q of lane k
  auto dma = [&](int k, int q, long c) {
    Lane& l = g_stage.lane[k];
    const long r0 = c * per, nr = std::min(per, b.rows - r0);
    if (copy_rows(b, up, l.buf[q], row_bytes, r0, nr) != hipSuccess ||
        hipEventRecord(l.ev[q], b.st) != hipSuccess)
      bad = 1;
  };
  auto work = [&](int k) {
    Lane& l = g_stage.lane[k];
    if (hipSetDevice(dev) != hipSuccess) {
      bad = 1;
      return;
    }
    int q = 0;
    for (long c = k; c < nslab && !bad; c += n, q ^= 1) {
      const long r0 = c * per, nr = std::min(per, b.rows - r0);
      if (up) {
        if (c >= k + 2L * n && hipEventSynchronize(l.ev[q]) != hipSuccess) bad = 1;
        host_rows(b, up, l.buf[q], r0, nr);
        if (!bad) dma(k, q, c);
      } else {
        if (c + n < nslab) dma(k, q ^ 1, c + n);  // its buffer was emptied a slab ago
        if (hipEventSynchronize(l.ev[q]) != hipSuccess) bad = 1;
        if (!bad) host_rows(b, up, l.buf[q], r0, nr);
      }
    }
  };
  // A download's first slabs are on their way before the threads start (queued by
  // the threads on a stream just waited for, they took 25-40 us longer: 500x500
  // FP64 372 us, 356 so).
  for (int k = 0; !up && k < n; k++) dma(k, 0, k);
  on_threads(n, work);
  // (the buffers are free again once the stream is past the copies)
  if ((up || bad) && hipStreamSynchronize(b.st) != hipSuccess) bad = 1;
  return bad ? copy_error(up) : 0;
}

int staged(char* host, int hesz, char* dev, int desz, long pitch, long width, long rows,
           hipStream_t st, bool up) {
  int current = 0, device = 0;  // (a stream may be another device's than the current one)
  if (hipGetDevice(&current) != hipSuccess || hipStreamGetDevice(st, &device) != hipSuccess ||
      (device != current && hipSetDevice(device) != hipSuccess))
    return copy_error(up);
  int rc = 0;
  // Earlier work on the stream is waited for before the lanes are taken, which
  // other threads' copies then do not wait for.
  if (hipStreamSynchronize(st) != hipSuccess) {
    rc = copy_error(up);
  } else {
    std::lock_guard<std::mutex> lk(g_stage.mu);
    const long most = (long) (kSlabBytes / desz);  // columns at a time
    for (long c = 0; c < width && rc == 0; c += most) {
      const Block b{host + (size_t) c * hesz, hesz, width, dev + (size_t) c * desz, desz, pitch,
                    std::min(most, width - c), rows, st};
      rc = copy_block(b, device, up);
    }
  }
  if (device != current) (void) hipSetDevice(current);
  return rc;
}
}  // namespace

// Copies `rows` rows of `width` elements (src_esz bytes each, source rows
// `src_pitch` elements apart on the device) to contiguous host rows of
// dst_esz-byte elements (dst_esz == src_esz, or 8 with src_esz == 4).
// Ordered after earlier work on `st`; returns when the data is in dst.
int stage_d2h(void* dst, int dst_esz, const void* src, int src_esz, long src_pitch, long width,
              long rows, hipStream_t st) {
  return staged((char*) dst, dst_esz, (char*) src, src_esz, src_pitch, width, rows, st, false);
}

// The way back: contiguous host rows of src_esz-byte elements to pitched rows
// on the device (dst_esz == src_esz, or 4 with src_esz == 8, rounded).
// Ordered after earlier work on `st`; returns when the data is on the device.
int stage_h2d(void* dst, int dst_esz, long dst_pitch, const void* src, int src_esz, long width,
              long rows, hipStream_t st) {
  return staged((char*) src, src_esz, (char*) dst, dst_esz, dst_pitch, width, rows, st, true);
}

// dst = src, n elements, on as many threads as that is worth (both in host memory).
void host_copy(void* dst, int dst_esz, const void* src, int src_esz, size_t n) {
  const int t = thread_count(n * (size_t) std::max(dst_esz, src_esz));
  const size_t per = (n + t - 1) / t;
  on_threads(t, [&](int k) {
    const size_t a = std::min(n, per * k), m = std::min(n, a + per) - a;
    convert((char*) dst + a * dst_esz, dst_esz, (const char*) src + a * src_esz, src_esz, m);
  });
}

}  // namespace hydro
