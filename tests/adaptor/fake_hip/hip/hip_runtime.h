// A HIP runtime of counters for host tests of code that allocates: nothing here
// touches a device.
#pragma once

#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <map>
#include <mutex>

#define __host__
#define __device__
#define __global__
#define __forceinline__ inline

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
inline const char *hipGetErrorString(hipError_t) { return "fake"; }
using hipStream_t = struct FakeStream *;
using hipEvent_t = struct FakeEvent *;
constexpr unsigned hipEventDisableTiming = 2;

namespace fake {
struct State {
  std::mutex mu;
  std::map<void *, std::size_t> device_memory, pinned_memory;
  std::map<void *, int> owner;  // device of each device allocation
  std::size_t capacity = SIZE_MAX;
  int device = 0, streams = 0, events = 0, syncs = 0, foreign_frees = 0;
  int events_left = 1 << 30;  // event creations that succeed
  hipError_t sync_result = hipSuccess;
  std::size_t used() {
    std::size_t s = 0;
    for (auto &m : device_memory) s += m.second;
    return s;
  }
};
inline State &state() {
  static State s;
  return s;
}
}  // namespace fake

inline hipError_t hipMalloc(void **p, std::size_t bytes) {
  auto &s = fake::state();
  std::lock_guard<std::mutex> g(s.mu);
  if (bytes > s.capacity || s.used() > s.capacity - bytes) return hipErrorOutOfMemory;
  *p = std::malloc(1);
  s.device_memory[*p] = bytes;
  s.owner[*p] = s.device;
  return hipSuccess;
}
inline hipError_t hipFree(void *p) {
  auto &s = fake::state();
  std::lock_guard<std::mutex> g(s.mu);
  s.foreign_frees += s.owner[p] != s.device;
  if (!s.device_memory.erase(p)) return hipErrorUnknown;
  s.owner.erase(p);
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipHostMalloc(void **p, std::size_t bytes) {
  auto &s = fake::state();
  std::lock_guard<std::mutex> g(s.mu);
  *p = std::malloc(1);
  s.pinned_memory[*p] = bytes;
  return hipSuccess;
}
inline hipError_t hipHostFree(void *p) {
  auto &s = fake::state();
  std::lock_guard<std::mutex> g(s.mu);
  if (!s.pinned_memory.erase(p)) return hipErrorUnknown;
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipStreamCreate(hipStream_t *st) {
  auto &s = fake::state();
  std::lock_guard<std::mutex> g(s.mu);
  ++s.streams;
  *st = reinterpret_cast<hipStream_t>(std::malloc(1));
  return hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t st) {
  auto &s = fake::state();
  std::lock_guard<std::mutex> g(s.mu);
  --s.streams;
  std::free(reinterpret_cast<void *>(st));
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) {
  auto &s = fake::state();
  std::lock_guard<std::mutex> g(s.mu);
  ++s.syncs;
  return s.sync_result;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  auto &s = fake::state();
  std::lock_guard<std::mutex> g(s.mu);
  if (s.events_left-- <= 0) return hipErrorUnknown;
  ++s.events;
  *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
  return hipSuccess;
}
inline hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
inline hipError_t hipEventDestroy(hipEvent_t e) {
  auto &s = fake::state();
  std::lock_guard<std::mutex> g(s.mu);
  --s.events;
  std::free(reinterpret_cast<void *>(e));
  return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int *d) {
  *d = fake::state().device;
  return hipSuccess;
}
inline hipError_t hipSetDevice(int d) {
  fake::state().device = d;
  return hipSuccess;
}
