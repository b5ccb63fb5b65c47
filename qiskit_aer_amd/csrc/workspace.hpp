// What a statevector handle allocates besides its plan: a stream, an event,
// pinned staging, device buffers and the state itself.  Creating and freeing
// them took most of a small simulator call (5 qubits, 1024 shots: 371 us, 155
// without), so a handle that ends leaves its set to a later one on the same
// device.
#pragma once

#include <cstddef>
#include <mutex>
#include <vector>

#include "common.hpp"

namespace aerhip {

struct Workspace {
  int device = -1;
  hipStream_t stream = nullptr;
  hipEvent_t event = nullptr;   // last upload from the staging buffer
  double *scalars = nullptr;    // pinned, 64 doubles
  struct Buffer {
    void *p = nullptr;
    size_t bytes = 0;
  };
  Buffer staging;               // pinned
  Buffer program, partial, scratch, probes, state;

  void release() {
    for (Buffer *b : {&program, &partial, &scratch, &probes, &state}) {
      if (b->p) (void)hipFree(b->p);
      *b = Buffer{};
    }
    if (staging.p) (void)hipHostFree(staging.p);
    staging = Buffer{};
    if (scalars) (void)hipHostFree(scalars);
    if (event) (void)hipEventDestroy(event);
    if (stream) (void)hipStreamDestroy(stream);
    scalars = nullptr;
    event = nullptr;
    stream = nullptr;
  }
};

// The sets of ended handles: at most four in a process, each with a state of at
// most 64 MiB (22 qubits in complex128) and buffers of at most 8 MiB; what is
// larger is freed with its handle, and all of it is freed when an allocation
// fails or the caller asks (aerhip_release_memory).  Any thread may take, give
// or release.
class WorkspacePool {
 public:
  static constexpr size_t kSets = 4, kStateBytes = 64u << 20, kBufferBytes = 8u << 20;

  static WorkspacePool &get() {
    static WorkspacePool *pool = new WorkspacePool;  // outlives every handle; not torn down after the runtime
    return *pool;
  }

  // A set for `device` whose state holds `bytes`; the current device is set.
  Workspace take(int device, size_t bytes) {
    Workspace w;
    {
      std::lock_guard<std::mutex> g(mu_);
      size_t at = sets_.size();
      for (size_t i = 0; i < sets_.size(); ++i)
        if (sets_[i].device == device && (at == sets_.size() || sets_[i].state.bytes == bytes)) at = i;
      if (at < sets_.size()) {
        w = sets_[at];
        sets_.erase(sets_.begin() + static_cast<std::ptrdiff_t>(at));
      }
    }
    try {
      w.device = device;
      if (!w.stream) AERHIP_CHECK(hipStreamCreate(&w.stream));
      if (!w.event) AERHIP_CHECK(hipEventCreateWithFlags(&w.event, hipEventDisableTiming));
      if (!w.scalars) AERHIP_CHECK(hipHostMalloc(reinterpret_cast<void **>(&w.scalars), 64 * sizeof(double)));
      if (w.state.bytes != bytes) grow(w.state, bytes);
    } catch (...) {
      w.release();
      throw;
    }
    return w;
  }

  // Takes back a set no work is pending on.
  void give(Workspace w) {
    auto drop = [](Workspace::Buffer &b) {
      if (b.p) (void)hipFree(b.p);
      b = Workspace::Buffer{};
    };
    if (w.state.bytes > kStateBytes) drop(w.state);
    for (Workspace::Buffer *b : {&w.program, &w.partial, &w.scratch, &w.probes})
      if (b->bytes > kBufferBytes) drop(*b);
    if (w.staging.bytes > kBufferBytes) {
      (void)hipHostFree(w.staging.p);
      w.staging = Workspace::Buffer{};
    }
    {
      std::lock_guard<std::mutex> g(mu_);
      sets_.push_back(w);
      if (sets_.size() <= kSets) return;
      w = sets_.front();
      sets_.erase(sets_.begin());
    }
    int device = 0;
    (void)hipGetDevice(&device);
    (void)hipSetDevice(w.device);
    w.release();
    (void)hipSetDevice(device);
  }

  void drain() {
    std::vector<Workspace> all;
    {
      std::lock_guard<std::mutex> g(mu_);
      all.swap(sets_);
    }
    int device = 0;
    (void)hipGetDevice(&device);
    for (Workspace &w : all) {
      (void)hipSetDevice(w.device);
      w.release();
    }
    (void)hipSetDevice(device);
  }

  // Device memory; a first failure frees the pool's sets and tries once more.
  static void *allocate(size_t bytes) {
    void *p = nullptr;
    hipError_t e = hipMalloc(&p, bytes);
    if (e == hipErrorOutOfMemory) {
      (void)hipGetLastError();
      get().drain();
      e = hipMalloc(&p, bytes);
    }
    AERHIP_CHECK(e);
    return p;
  }

  // Replaces a buffer (nothing on the device uses it) by one of `bytes`.
  static void grow(Workspace::Buffer &b, size_t bytes) {
    void *old = b.p;
    b = Workspace::Buffer{};
    if (old) AERHIP_CHECK(hipFree(old));
    b.p = allocate(bytes);
    b.bytes = bytes;
  }

 private:
  std::mutex mu_;
  std::vector<Workspace> sets_;
};

// A set for the life of a scope or an object, also one whose constructor throws
// later.  Back to the pool it goes when its stream is done; after an error there
// it is freed.
class WorkspaceLease {
 public:
  WorkspaceLease(int device, size_t bytes) : w_(WorkspacePool::get().take(device, bytes)) {}
  ~WorkspaceLease() {
    (void)hipSetDevice(w_.device);
    if (hipStreamSynchronize(w_.stream) == hipSuccess)
      WorkspacePool::get().give(w_);
    else
      w_.release();
  }
  WorkspaceLease(const WorkspaceLease &) = delete;
  WorkspaceLease &operator=(const WorkspaceLease &) = delete;
  Workspace *operator->() { return &w_; }

 private:
  Workspace w_;
};

// Two events that time what lies between them.
struct EventPair {
  hipEvent_t begin = nullptr, end = nullptr;
  EventPair() = default;
  ~EventPair() {
    if (begin) (void)hipEventDestroy(begin);
    if (end) (void)hipEventDestroy(end);
  }
  EventPair(const EventPair &) = delete;
  EventPair &operator=(const EventPair &) = delete;
  void create() {
    AERHIP_CHECK(hipEventCreate(&begin));
    AERHIP_CHECK(hipEventCreate(&end));
  }
};

}  // namespace aerhip
