// A stand-in for the HIP runtime on the CPU, for checks of the library's host
// code alone (no kernel runs): device memory is host memory, every queued
// operation is done at once, and a check can refuse calls or hold a stream.
#pragma once
#include <hip/hip_runtime.h>

#include <functional>

namespace onhost {
// Asked before every call of the runtime (by its name); true: the call fails.
extern std::function<bool(const char*)> refuse;
// While held, waiting for the stream (or for an event recorded on it) blocks.
void hold(hipStream_t st, bool on);
}  // namespace onhost
