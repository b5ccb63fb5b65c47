// The pool of ended handles' buffers (csrc/workspace.hpp) on a fake runtime.
// Usage: workspace_pool CASE; prints the case and ends with 0 if it holds.
#include <cstdio>
#include <cstring>
#include <optional>

#include "workspace.hpp"

using aerhip::Workspace;
using aerhip::WorkspacePool;

namespace {

int failures = 0;
void expect(bool ok, const char *what) {
  if (!ok) {
    std::printf("failed: %s\n", what);
    ++failures;
  }
}
#define EXPECT(x) expect((x), #x)

Workspace take(int device, std::size_t bytes) {
  (void)hipSetDevice(device);
  return WorkspacePool::get().take(device, bytes);
}

// At most four sets stay, none with a large buffer; the rest is freed.
void bounded() {
  auto &s = fake::state();
  Workspace w[7];
  for (int i = 0; i < 7; ++i) {
    w[i] = take(0, 1000 + i);
    WorkspacePool::grow(w[i].scratch, i % 2 ? WorkspacePool::kBufferBytes + 1 : 100);
  }
  WorkspacePool::grow(w[6].state, WorkspacePool::kStateBytes + 1);
  for (auto &x : w) WorkspacePool::get().give(x);
  EXPECT(s.streams == 4);
  EXPECT(s.events == 4);
  EXPECT(s.used() <= 4 * (1010 + 100));
  WorkspacePool::get().drain();
  EXPECT(s.used() == 0 && s.streams == 0 && s.events == 0 && s.pinned_memory.empty());
}

// A failed allocation frees the sets and is tried once more; a second failure
// is reported and leaks nothing.
void out_of_memory() {
  auto &s = fake::state();
  s.capacity = 10000;
  for (int i = 0; i < 2; ++i) {
    Workspace a = take(0, 3000), b = take(0, 3001);
    WorkspacePool::get().give(a);
    WorkspacePool::get().give(b);
  }
  EXPECT(s.used() == 6001);
  Workspace c = take(0, 9000);  // grows one of them in place of both
  EXPECT(c.state.bytes == 9000 && s.used() == 9000);
  bool threw = false;
  try {
    take(0, 2000);
  } catch (const std::exception &) {
    threw = true;
  }
  EXPECT(threw);
  EXPECT(s.used() == 9000 && s.streams == 1 && s.events == 1);
  WorkspacePool::get().give(c);
  EXPECT(s.used() == 9000);
}

// Sets are taken on their own device, and giving one back leaves the caller's
// current device as it was.
void devices() {
  auto &s = fake::state();
  Workspace w[6];
  for (int i = 0; i < 6; ++i) w[i] = take(i < 3 ? 0 : 1, 100);
  for (auto &x : w) {
    (void)hipSetDevice(x.device);
    WorkspacePool::get().give(x);
    EXPECT(s.device == x.device);
  }
  Workspace a = take(0, 100), b = take(1, 100);
  EXPECT(s.owner[a.state.p] == 0 && s.owner[b.state.p] == 1);
  (void)hipSetDevice(1);
  WorkspacePool::get().drain();
  EXPECT(s.device == 1);
  EXPECT(s.foreign_frees == 0);
}

// An object that takes a set and then fails to make its events leaves the set
// to the pool; one whose stream reports an error frees it.
void leases() {
  using aerhip::EventPair;
  using aerhip::WorkspaceLease;
  auto &s = fake::state();
  struct Object {
    std::optional<WorkspaceLease> ws;
    EventPair ev;
    explicit Object(std::size_t bytes) {
      ws.emplace(0, bytes);
      ev.create();
    }
  };
  for (int left : {1, 2}) {  // the set's own event, then none or one of the two
    s.events_left = left + (s.streams ? -1 : 0);
    bool threw = false;
    try {
      Object o(500);
    } catch (const std::exception &) {
      threw = true;
    }
    EXPECT(threw);
    EXPECT(s.streams == 1 && s.events == 1 && s.used() == 500 && s.syncs > 0);
  }
  s.events_left = 100;
  { Object o(500); }
  EXPECT(s.streams == 1 && s.events == 1 && s.used() == 500);
  {
    Object o(500);
    s.sync_result = hipErrorUnknown;
  }
  EXPECT(s.streams == 0 && s.events == 0 && s.used() == 0 && s.pinned_memory.empty());
}

}  // namespace

int main(int argc, char **argv) {
  const char *name = argc > 1 ? argv[1] : "";
  std::printf("case: %s\n", name);
  if (!std::strcmp(name, "bounded")) bounded();
  else if (!std::strcmp(name, "out_of_memory")) out_of_memory();
  else if (!std::strcmp(name, "devices")) devices();
  else if (!std::strcmp(name, "leases")) leases();
  else return 2;
  return failures ? 1 : 0;
}
