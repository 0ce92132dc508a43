// host_copy.hpp -- copies between pageable host memory and the device.
//
// The runtime moves pageable memory through its own pinned buffer with one
// thread: 30 GB/s up, 17 GB/s down and 10 GB/s into pages that have not been
// touched yet, against 57 GB/s of the link.  Here a few threads copy between
// the caller's memory and four pinned slots while the link moves the slots
// before and after.  The flow solver's cycle with 1.5M droplets (1.1 GB across
// the link) 68 -> 40 ms, restart records of 250k droplets in and out 12.8 -> 6.6.
#pragma once
#include <hip/hip_runtime.h>
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace ntlp {

// memcpy shared out among a fixed set of threads and the caller.  One caller
// at a time.
class CopyThreads {
 public:
  // workers besides the caller; fewer where threads cannot be made
  explicit CopyThreads(int workers) {
    try {
      for (int k = 0; k < workers; ++k) threads_.emplace_back([this, k] { work(k); });
    } catch (...) {  // as many as there are
    }
    parts_ = (int)threads_.size() + 1;
  }
  ~CopyThreads() {
    {
      std::lock_guard<std::mutex> lk(mu_);
      stop_ = true;
    }
    turn_.fetch_add(1);
    cv_.notify_all();
    for (auto& t : threads_) t.join();
  }
  CopyThreads(const CopyThreads&) = delete;
  CopyThreads& operator=(const CopyThreads&) = delete;

  void copy(void* dst, const void* src, size_t bytes) {
    if (threads_.empty() || bytes < kSolo) {
      memcpy(dst, src, bytes);
      return;
    }
    dst_ = static_cast<char*>(dst);
    src_ = static_cast<const char*>(src);
    bytes_ = bytes;
    left_.store((int)threads_.size(), std::memory_order_relaxed);
    {
      std::lock_guard<std::mutex> lk(mu_);
      turn_.fetch_add(1, std::memory_order_release);
    }
    cv_.notify_all();
    part((int)threads_.size());
    while (left_.load(std::memory_order_acquire) != 0) std::this_thread::yield();
  }

 private:
  static constexpr size_t kSolo = 256 << 10;  // below, waking the threads costs more than it saves
  static constexpr int kSpins = 200;          // looks for the next chunk of the same transfer before sleeping

  void part(int k) {
    const size_t per = (bytes_ / parts_ + 4095) & ~(size_t)4095;  // whole pages: no two threads fault the same one
    const size_t a = std::min(bytes_, per * k), b = k == parts_ - 1 ? bytes_ : std::min(bytes_, per * (k + 1));
    if (b > a) memcpy(dst_ + a, src_ + a, b - a);
  }
  void work(int k) {
    uint64_t seen = 0;
    for (;;) {
      int spins = 0;
      while (turn_.load(std::memory_order_acquire) == seen && spins < kSpins) {
        ++spins;
        std::this_thread::yield();
      }
      if (turn_.load(std::memory_order_acquire) == seen) {
        std::unique_lock<std::mutex> lk(mu_);
        cv_.wait(lk, [&] { return stop_ || turn_.load(std::memory_order_acquire) != seen; });
      }
      if (stop_.load(std::memory_order_acquire)) return;
      ++seen;  // the caller waits for every worker before the next turn
      part(k);
      left_.fetch_sub(1, std::memory_order_release);
    }
  }

  std::vector<std::thread> threads_;
  int parts_ = 1;
  std::mutex mu_;
  std::condition_variable cv_;
  std::atomic<uint64_t> turn_{0};
  std::atomic<int> left_{0};
  std::atomic<bool> stop_{false};
  char* dst_ = nullptr;
  const char* src_ = nullptr;
  size_t bytes_ = 0;
};

// The slots and threads of one context; made by its first large transfer.
class HostLink {
 public:
  static constexpr int kSlots = 4;
  static constexpr size_t kSlotBytes = 4 << 20;
  static constexpr size_t kDirect = 1 << 20;  // smaller copies go through the runtime: 50-70 us either way
  static constexpr int kWorkers = 7;          // 8 threads with the caller reach the link's 57 GB/s

  // hipErrorOutOfMemory when the slots cannot be had
  hipError_t open() {
    for (int k = 0; k < kSlots; ++k) {
      hipError_t e = hipHostMalloc(&slot_[k], kSlotBytes, hipHostMallocDefault);
      if (e == hipSuccess) e = hipEventCreateWithFlags(&ev_[k], hipEventDisableTiming);
      if (e != hipSuccess) return e;
    }
    cpu_set_t set;
    CPU_ZERO(&set);
    const int cpus = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
    threads_.reset(new (std::nothrow) CopyThreads(std::min(kWorkers, std::max(0, cpus / 2 - 1))));
    return threads_ ? hipSuccess : hipErrorOutOfMemory;
  }
  // returns the pinned memory (not done by the destructor, which may run after
  // the runtime's own)
  void close() {
    for (int k = 0; k < kSlots; ++k) {
      if (ev_[k]) (void)hipEventSynchronize(ev_[k]);
      if (ev_[k]) (void)hipEventDestroy(ev_[k]);
      if (slot_[k]) (void)hipHostFree(slot_[k]);
      ev_[k] = nullptr;
      slot_[k] = nullptr;
    }
    threads_.reset();
  }

  // In stream order with `stream`; src may be reused on return.
  hipError_t up(void* dst, const void* src, size_t bytes, hipStream_t stream) {
    const size_t step = chunk(bytes);
    for (size_t o = 0; o < bytes; o += step) {
      const size_t n = std::min(step, bytes - o);
      const int k = next();
      hipError_t e = hipEventSynchronize(ev_[k]);  // the slot's last transfer
      if (e != hipSuccess) return e;
      threads_->copy(slot_[k], (const char*)src + o, n);
      e = hipMemcpyAsync((char*)dst + o, slot_[k], n, hipMemcpyHostToDevice, stream);
      if (e == hipSuccess) e = hipEventRecord(ev_[k], stream);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  // In stream order with `stream`; dst is complete on return.
  hipError_t down(void* dst, const void* src, size_t bytes, hipStream_t stream) {
    const size_t step = chunk(bytes), count = (bytes + step - 1) / step;
    int at[kSlots];  // slot of chunk i at [i % kSlots]
    for (size_t i = 0; i < count + kSlots - 1; ++i) {
      if (i < count) {
        const size_t o = i * step, n = std::min(step, bytes - o);
        const int k = at[i % kSlots] = next();
        hipError_t e = hipEventSynchronize(ev_[k]);
        if (e == hipSuccess) e = hipMemcpyAsync(slot_[k], (const char*)src + o, n, hipMemcpyDeviceToHost, stream);
        if (e == hipSuccess) e = hipEventRecord(ev_[k], stream);
        if (e != hipSuccess) return e;
      }
      if (i + 1 >= kSlots) {  // the oldest chunk under way
        const size_t j = i + 1 - kSlots, o = j * step, n = std::min(step, bytes - o);
        const int k = at[j % kSlots];
        const hipError_t e = hipEventSynchronize(ev_[k]);
        if (e != hipSuccess) return e;
        threads_->copy((char*)dst + o, slot_[k], n);
      }
    }
    return hipSuccess;
  }

 private:
  // pieces of a transfer: four or more, of 512 KB to a slot
  static size_t chunk(size_t bytes) {
    const size_t c = ((bytes / 4 + 4095) & ~(size_t)4095);
    return std::min(kSlotBytes, std::max<size_t>(c, 512 << 10));
  }
  int next() { return turn_++ % kSlots; }

  void* slot_[kSlots] = {};
  hipEvent_t ev_[kSlots] = {};
  unsigned turn_ = 0;
  std::unique_ptr<CopyThreads> threads_;
};

}  // namespace ntlp
