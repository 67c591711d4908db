// qs_copyout.hpp -- device-to-host copy of a large output to pageable memory, behind the work
// on a stream, by a few threads: each takes chunks of 1 MB, brings them through two pinned
// buffers of its own (the next chunk's transfer under way while one is copied out), and the
// call returns when all are copied.  The runtime's own pageable copy moves 128 MB in 11 ms
// (12 GB/s: one thread copies, and takes the page faults of a fresh array), these about
// 2.5 ms (a 4096^2 exit wave with its run 22.4 -> 13.7 ms).
//
// RT: the runtime's calls (the tests stand in for them).
#pragma once
#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <thread>

namespace qs {

template <class RT>
class CopyOut {
 public:
  using Error = typename RT::Error;
  using Stream = typename RT::Stream;
  static constexpr size_t kChunk = size_t(1) << 20;
  static constexpr int kWorkers = 5;

  ~CopyOut() { release(); }
  void release() {
    for (typename RT::Event& e : ev_)
      if (e) RT::event_destroy(e), e = {};
    if (pinned_) RT::host_free(pinned_), pinned_ = nullptr;
  }

  // Outputs below 16 MB, and those that the buffers and events cannot be had for, take the
  // runtime's own copy.
  Error copy(int device, void* dst, const void* src, size_t bytes, Stream st) {
    if (bytes < 16 * kChunk || !ready()) return RT::copy(dst, src, bytes, st);
    const size_t n = (bytes + kChunk - 1) / kChunk;
    std::atomic<size_t> next{0};
    std::atomic<int> failed{(int)RT::ok};
    auto work = [&](int w) {
      size_t at[2] = {n, n};                                // chunk on its way in each buffer
      Error e = w > 0 ? RT::set_device(device) : RT::ok;    // (a new thread's current device)
      for (int b = 0; e == RT::ok; b ^= 1) {
        char* const buf = static_cast<char*>(pinned_) + (2 * w + b) * kChunk;
        const size_t i = next.fetch_add(1);
        if (i < n) {  // (this buffer's last chunk was copied out below)
          e = RT::copy(buf, static_cast<const char*>(src) + i * kChunk, std::min(kChunk, bytes - i * kChunk), st);
          if (e == RT::ok) e = RT::event_record(ev_[2 * w + b], st);
          at[b] = i;
        }
        const size_t j = at[b ^ 1];
        if (e == RT::ok && j < n) {
          e = RT::event_wait(ev_[2 * w + (b ^ 1)]);
          if (e == RT::ok)
            memcpy(static_cast<char*>(dst) + j * kChunk, buf + (b ? -(ptrdiff_t)kChunk : (ptrdiff_t)kChunk),
                   std::min(kChunk, bytes - j * kChunk));
          at[b ^ 1] = n;
        }
        if (i >= n && at[0] >= n && at[1] >= n) break;
      }
      if (e != RT::ok) failed = (int)e;
    };
    std::thread helpers[kWorkers - 1];
    for (int w = 1; w < kWorkers; w++) {
      try {
        helpers[w - 1] = std::thread(work, w);
      } catch (...) {  // no more threads: the others and the caller take its chunks
        break;
      }
    }
    work(0);
    for (std::thread& t : helpers)
      if (t.joinable()) t.join();
    // after an error, transfers may still be on their way to the buffers
    if (failed.load() != (int)RT::ok) (void)RT::stream_wait(st);
    return (Error)failed.load();
  }

 private:
  // The pinned buffers and the events of their transfers: all of them or none.
  bool ready() {
    if (pinned_) return true;
    bool all = RT::host_alloc(&pinned_, 2 * kWorkers * kChunk) == RT::ok;
    if (!all) pinned_ = nullptr;
    for (int i = 0; all && i < 2 * kWorkers; i++)
      if (RT::event_create(&ev_[i]) != RT::ok) {
        ev_[i] = {};
        all = false;
      }
    if (!all) {
      release();
      RT::clear_error();
    }
    return all;
  }

  void* pinned_ = nullptr;
  typename RT::Event ev_[2 * kWorkers] = {};
};

}  // namespace qs
