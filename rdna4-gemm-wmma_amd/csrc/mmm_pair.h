// Keeps the two launches of a call that splits K together on their stream.
//
// Such a call writes partial tiles to the caller's workspace in one launch and sums them in the next.
// Calls on one stream run in order, so they may share a workspace; but with several host threads
// calling on one stream, another thread's first launch could be enqueued between the two and its
// partial tiles land before they are summed.  A StreamPair held over both launches admits one thread
// per stream; threads on other streams are not waited for.  No memory is allocated, and nothing is
// kept of a call after it.
#pragma once

#include <condition_variable>
#include <mutex>
#include <new>

namespace mmm {

class StreamPair {
 public:
  // stream: an address that stands for it (pair_stream in mmm_kernels.h); null: nothing to keep.
  explicit StreamPair(const void* stream) : stream_(stream) {
    if (!stream_) return;
    Held& h = held();
    std::unique_lock<std::mutex> lock(h.m);
    int slot;
    while ((slot = h.slot_for(stream_)) < 0) h.freed.wait(lock);
    h.streams[slot] = stream_;
  }
  ~StreamPair() {
    if (!stream_) return;
    Held& h = held();
    {
      std::lock_guard<std::mutex> lock(h.m);
      for (const void*& s : h.streams)
        if (s == stream_) s = nullptr;
    }
    h.freed.notify_all();
  }
  StreamPair(const StreamPair&) = delete;
  StreamPair& operator=(const StreamPair&) = delete;

 private:
  static constexpr int kMost = 64;  // threads inside a pair at one moment; one more waits for any of them
  struct Held {
    std::mutex m;
    std::condition_variable freed;
    const void* streams[kMost] = {};
    // a free slot if the stream is in none, else -1
    int slot_for(const void* stream) const {
      int free = -1;
      for (int i = kMost - 1; i >= 0; --i) {
        if (streams[i] == stream) return -1;
        if (!streams[i]) free = i;
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
  const void* stream_;
};

}  // namespace mmm
