// Keeps the two launches of a call that splits K together.
//
// Such a call writes partial tiles to a workspace in one launch and sums them in the next.  Calls on one
// stream run in order, so they may share a workspace; but with several host threads calling on one
// stream, another thread's first launch could be enqueued between the two and its partial tiles land
// before they are summed.  A LaunchPair held over both launches admits one thread per workspace;
// calls with another workspace are not waited for.  No memory is allocated, and nothing is kept of a
// call after it.
#pragma once

#include <condition_variable>
#include <mutex>
#include <new>

namespace mmm {

class LaunchPair {
 public:
  // workspace: where the partial tiles go; null (unsplit): nothing to keep.
  explicit LaunchPair(const void* workspace) : workspace_(workspace) {
    if (!workspace_) return;
    Held& h = held();
    std::unique_lock<std::mutex> lock(h.m);
    int slot;
    while ((slot = h.slot_for(workspace_)) < 0) {
      ++h.waiting;
      h.freed.wait(lock);
      --h.waiting;
    }
    h.workspaces[slot] = workspace_;
    if (slot >= h.used) h.used = slot + 1;
  }
  ~LaunchPair() {
    if (!workspace_) return;
    Held& h = held();
    bool wake;
    {
      std::lock_guard<std::mutex> lock(h.m);
      for (int i = 0; i < h.used; ++i)
        if (h.workspaces[i] == workspace_) h.workspaces[i] = nullptr;
      while (h.used > 0 && !h.workspaces[h.used - 1]) --h.used;
      wake = h.waiting > 0;
    }
    if (wake) h.freed.notify_all();
  }
  LaunchPair(const LaunchPair&) = delete;
  LaunchPair& operator=(const LaunchPair&) = delete;

 private:
  static constexpr int kMost = 64;  // threads inside a pair at one moment; one more waits for any of them
  struct Held {
    std::mutex m;
    std::condition_variable freed;
    int used = 0, waiting = 0;  // slots [used, kMost) are free
    const void* workspaces[kMost] = {};
    // a free slot if the workspace is in none, else -1
    int slot_for(const void* workspace) const {
      int free = used < kMost ? used : -1;
      for (int i = used - 1; i >= 0; --i) {
        if (workspaces[i] == workspace) return -1;
        if (!workspaces[i]) free = i;
      }
      return free;
    }
  };
  static Held& held() {
    // never destroyed: a thread may still launch while the process ends
    alignas(Held) static unsigned char mem[sizeof(Held)];
    static Held* h = new (mem) Held;
    return *h;
  }
  const void* workspace_;
};

}  // namespace mmm
