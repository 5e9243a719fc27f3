// Host check of the enqueue locks (EnqueueLocks in csrc/workspace_pool.h): calls
// from several threads on a few fake streams, each asking for a buffer (growing
// it now and then) and enqueueing three launches that use it, with other calls
// of a thread's own inside, as a call's row tail makes them.  On every stream
// the launches of one call have to follow one another, and no launch may be
// given a buffer that was freed before it was enqueued.  Built and run by
// tests/test_workspace_threads.py; prints "ok" and exits 0.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <set>
#include <thread>

#include "workspace_pool.h"

namespace {

std::mutex g_mu;  // as workspace.cpp's: the pool itself
std::set<void*> g_live;
std::atomic<int> g_failures{0};

struct Ops {
  void* alloc(size_t) {
    void* p = std::malloc(16);
    g_live.insert(p);
    return p;
  }
  bool free(void* p) {
    g_live.erase(p);
    return true;  // (kept allocated, so that no address comes back)
  }
  bool sync(int) { return true; }
  void clear_error() {}
  tsplat::StreamState state(int) { return tsplat::StreamState::kIdle; }
  uint64_t now_ns() { return 0; }
};

struct Launch {
  int call, step;
};
constexpr int kStreams = 3, kThreads = 8, kCalls = 400, kLaunches = 3;
std::vector<Launch> g_queue[kStreams];

tsplat::WorkspacePool<int, Ops> g_pool{Ops{}};
tsplat::EnqueueLocks g_locks;

void fail(const char* what) {
  if (g_failures++ < 5) std::printf("FAIL: %s\n", what);
}

void call(int id, int stream, int depth) {
  const auto enqueue = g_locks.hold(reinterpret_cast<const void*>((uintptr_t)stream * 4096));
  void* ptr;
  {
    std::lock_guard<std::mutex> lock(g_mu);
    ptr = g_pool.acquire(0, stream, depth, (size_t)1 << (16 + id % 7), false);
  }
  for (int step = 0; step < kLaunches; ++step) {
    std::this_thread::yield();
    if (step == 1 && depth == 0 && id % 3 == 0) call(id + 1000000, stream, 1);
    std::lock_guard<std::mutex> lock(g_mu);
    if (g_live.count(ptr) == 0) fail("a launch's buffer was freed before it");
    g_queue[stream].push_back(Launch{id, step});
  }
}

}  // namespace

int main() {
  std::vector<std::thread> threads;
  for (int t = 0; t < kThreads; ++t)
    threads.emplace_back([t] {
      for (int i = 0; i < kCalls; ++i) {
        call(t * kCalls + i, (t + i) % kStreams, 0);
        if (i % 50 == 49) {
          const auto all = g_locks.hold_all();
          std::lock_guard<std::mutex> lock(g_mu);
          g_pool.release(0, 0);
        }
      }
    });
  for (auto& t : threads) t.join();
  size_t launches = 0;
  for (auto& q : g_queue) {
    launches += q.size();
    int open = -1, inner = -1;
    for (const Launch& l : q) {
      int& call = l.call >= 1000000 ? inner : open;
      if (l.step == 0 && (call != -1 || (l.call < 1000000 && inner != -1))) fail("a call began inside another");
      if (l.step != 0 && call != l.call) fail("a call's launches were separated");
      if (l.call >= 1000000 && open != l.call - 1000000) fail("an inner call outside its own");
      call = l.step == kLaunches - 1 ? -1 : l.call;
    }
  }
  if (launches < (size_t)kThreads * kCalls * kLaunches) fail("launches are missing");
  if (g_failures == 0) std::printf("ok\n");
  return g_failures == 0 ? 0 : 1;
}
