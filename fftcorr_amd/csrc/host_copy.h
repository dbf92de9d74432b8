// Copies of large host arrays (catalogues) to the device through pinned
// staging memory, filled by a few threads.
//
// hipMemcpyAsync from pageable memory stages on the calling thread alone:
// 18 GB/s for a 24 or 72 MB catalogue, about a third of what the link takes.
// Here kThreads threads (the caller is one of them) each copy chunks into
// two pinned slots of their own and queue the transfers, so the link works
// while the next chunks are filled.  The transfers go to two streams in turn:
// on one, 15 us pass between two of them (24 MB 0.83 ms with 1 MB chunks on one
// stream, 0.69 with 2 MB chunks, 0.61 on two streams; 72 MB 2.37, 1.85 and 1.53
// ms).  The threads, streams, slots (16 MB in all) and events belong to one
// context and end with it.
#pragma once

#include <hip/hip_runtime.h>

#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace fc {

class HostCopier {
 public:
  // Shorter copies take the runtime's own path: waking the threads costs more
  // than they save.
  static constexpr size_t kMinBytes = size_t(4) << 20;

  explicit HostCopier(int device) : device_(device) {
    for (Slot& s : slots_) {
      if (hipHostMalloc(&s.mem, kChunk, hipHostMallocDefault) != hipSuccess) s.mem = nullptr;
      if (s.mem && hipEventCreateWithFlags(&s.done, hipEventDisableTiming) != hipSuccess)
        s.done = nullptr;
      usable_ = usable_ && s.mem && s.done;
    }
    for (Lane& l : lanes_) {
      if (hipStreamCreateWithFlags(&l.stream, hipStreamNonBlocking) != hipSuccess)
        l.stream = nullptr;
      if (hipEventCreateWithFlags(&l.done, hipEventDisableTiming) != hipSuccess)
        l.done = nullptr;
      usable_ = usable_ && l.stream && l.done;
    }
    if (hipEventCreateWithFlags(&fork_, hipEventDisableTiming) != hipSuccess) fork_ = nullptr;
    usable_ = usable_ && fork_;
    (void)hipGetLastError();
  }

  ~HostCopier() {
    {
      std::lock_guard<std::mutex> lk(mu_);
      stop_ = true;
    }
    wake_.notify_all();
    for (std::thread& t : threads_) t.join();
    for (Slot& s : slots_) {
      if (s.done) {
        if (s.busy) (void)hipEventSynchronize(s.done);
        (void)hipEventDestroy(s.done);
      }
      if (s.mem) (void)hipHostFree(s.mem);
    }
    for (Lane& l : lanes_) {
      if (l.stream) (void)hipStreamDestroy(l.stream);
      if (l.done) (void)hipEventDestroy(l.done);
    }
    if (fork_) (void)hipEventDestroy(fork_);
  }

  // Page-locked bytes it holds.
  size_t pinned_bytes() const {
    size_t b = 0;
    for (const Slot& s : slots_) b += s.mem ? kChunk : 0;
    return b;
  }

  HostCopier(const HostCopier&) = delete;
  HostCopier& operator=(const HostCopier&) = delete;

  // Copies dst[0, bytes) = src[0, bytes) after the work queued on stream s and
  // before what s is given next.  src may change or go when this returns, or
  // (shorter copies out of page-locked memory) when s has been waited for.
  // The caller's current device is the copier's.
  hipError_t copy(void* dst, const void* src, size_t bytes, hipStream_t s) {
    if (bytes < kMinBytes || !usable_)
      return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s);
    std::lock_guard<std::mutex> one(call_);
    hipError_t e = hipEventRecord(fork_, s);
    for (Lane& l : lanes_)
      if (e == hipSuccess) e = hipStreamWaitEvent(l.stream, fork_, 0);
    if (e != hipSuccess) return e;
    {
      std::lock_guard<std::mutex> lk(mu_);
      // On a failure to start threads the caller copies alone.
      try {
        while ((int)threads_.size() < kThreads - 1) {
          const int id = (int)threads_.size() + 1;
          threads_.emplace_back([this, id] { serve(id); });
        }
      } catch (const std::exception&) {
      }
      dst_ = static_cast<char*>(dst);
      src_ = static_cast<const char*>(src);
      bytes_ = bytes;
      next_ = 0;
      error_ = hipSuccess;
      running_ = (int)threads_.size();
      ++job_;
    }
    wake_.notify_all();
    fill(0);
    {
      std::unique_lock<std::mutex> lk(mu_);
      idle_.wait(lk, [this] { return running_ == 0; });
      e = error_;
    }
    for (Lane& l : lanes_) {
      hipError_t j = hipEventRecord(l.done, l.stream);
      if (j == hipSuccess) j = hipStreamWaitEvent(s, l.done, 0);
      if (j != hipSuccess) (void)hipStreamSynchronize(l.stream);
      if (e == hipSuccess) e = j;
    }
    return e;
  }

 private:
  static constexpr int kThreads = 4, kSlotsPer = 2, kLanes = 2;
  static constexpr size_t kChunk = size_t(2) << 20;
  struct Slot {
    void* mem = nullptr;
    hipEvent_t done = nullptr;
    bool busy = false;  // its last transfer may be on the way
  };

  struct Lane {
    hipStream_t stream = nullptr;
    hipEvent_t done = nullptr;
  };

  void serve(int id) {
    const hipError_t set = hipSetDevice(device_);
    uint64_t seen = 0;
    for (;;) {
      {
        std::unique_lock<std::mutex> lk(mu_);
        wake_.wait(lk, [&] { return stop_ || job_ != seen; });
        if (stop_) return;
        seen = job_;
      }
      if (set == hipSuccess) fill(id);  // else the others take its chunks
      bool last;
      {
        std::lock_guard<std::mutex> lk(mu_);
        last = --running_ == 0;
      }
      if (last) idle_.notify_all();
    }
  }

  void fill(int id) {
    for (int turn = 0;; turn = (turn + 1) % kSlotsPer) {
      size_t at;
      {
        std::lock_guard<std::mutex> lk(mu_);
        if (next_ >= bytes_ || error_ != hipSuccess) return;
        at = next_;
        next_ += kChunk;
      }
      Slot& slot = slots_[id * kSlotsPer + turn];
      hipStream_t s = lanes_[at / kChunk % kLanes].stream;
      const size_t len = bytes_ - at < kChunk ? bytes_ - at : kChunk;
      hipError_t e = slot.busy ? hipEventSynchronize(slot.done) : hipSuccess;
      if (e == hipSuccess) {
        slot.busy = false;
        std::memcpy(slot.mem, src_ + at, len);
        e = hipMemcpyAsync(dst_ + at, slot.mem, len, hipMemcpyHostToDevice, s);
      }
      if (e == hipSuccess) {
        e = hipEventRecord(slot.done, s);
        slot.busy = e == hipSuccess;
        if (!slot.busy) (void)hipStreamSynchronize(s);
      }
      if (e != hipSuccess) {
        std::lock_guard<std::mutex> lk(mu_);
        if (error_ == hipSuccess) error_ = e;
        return;
      }
    }
  }

  const int device_;
  bool usable_ = true;
  Slot slots_[kThreads * kSlotsPer];
  Lane lanes_[kLanes];
  hipEvent_t fork_ = nullptr;
  std::mutex call_;  // one copy at a time
  std::mutex mu_;    // everything below
  std::condition_variable wake_, idle_;
  std::vector<std::thread> threads_;
  bool stop_ = false;
  uint64_t job_ = 0;
  int running_ = 0;
  char* dst_ = nullptr;
  const char* src_ = nullptr;
  size_t bytes_ = 0, next_ = 0;
  hipError_t error_ = hipSuccess;
};

}  // namespace fc
