// Bulk traffic between pageable host memory (or a file) and device memory.
//
// A copy from pageable memory runs at 29 GB/s here and one thread fills or empties fresh pages at 3 to 6 GB/s, while
// the copy engine moves 57 GB/s out of pinned memory.  So the data pass through a few pinned blocks: each of several
// threads takes every k-th block of the transfer and fills one of its two blocks while the other one is on its way.
// The blocks belong to an engine and are given back with it at the latest.
#pragma once
#include <hip/hip_runtime.h>
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <exception>
#include <mutex>
#include <stdexcept>
#include <string>
#include <system_error>
#include <thread>
#include <vector>

namespace cuhnsw_amd {

#define HIP_CHECK(expr)                                                                              \
  do {                                                                                               \
    hipError_t err_ = (expr);                                                                        \
    if (err_ != hipSuccess) {                                                                        \
      (void)hipGetLastError(); /* reported here, not by the next launch of a later call */           \
      throw std::runtime_error(std::string("HIP error: ") + hipGetErrorString(err_) + " at " #expr); \
    }                                                                                                \
  } while (0)

// What engines keep between calls so that the next one finds it allocated is bounded for the process as a whole: an
// engine that would go beyond keeps nothing and allocates anew each time.
class KeptMemory {
 public:
  explicit constexpr KeptMemory(size_t limit) : limit_(limit) {}
  bool take(size_t n) {
    if (total_.fetch_add(n) + n <= limit_) return true;
    total_ -= n;
    return false;
  }
  void give_back(size_t n) { total_ -= n; }

 private:
  const size_t limit_;
  std::atomic<size_t> total_{0};
};
inline KeptMemory kept_device_memory((size_t)4 << 30);  // (of 288 GB, on whichever GPUs)
inline KeptMemory kept_pinned_memory((size_t)256 << 20);

// threads worth using for `bytes` of host-side bulk work in steps of `block`
inline int host_threads(size_t bytes, size_t block) {
  cpu_set_t set;
  CPU_ZERO(&set);
  const int cpus = sched_getaffinity(0, sizeof(set), &set) == 0 ? std::max(1, std::min(CPU_COUNT(&set), 8)) : 1;
  return (int)std::max<size_t>(1, std::min<size_t>((size_t)cpus, (bytes + block - 1) / block));
}

// body(t) for t = 0 .. n-1 on n threads, `meanwhile` on this one; the first exception is thrown again here once
// every thread is done.
template <typename Body, typename Meanwhile>
void run_on_threads(int n, Body&& body, Meanwhile&& meanwhile) {
  std::mutex m;
  std::exception_ptr first;
  auto guarded = [&](auto&& f) {
    try {
      f();
    } catch (...) {
      std::lock_guard<std::mutex> lock(m);
      if (!first) first = std::current_exception();
    }
  };
  std::vector<std::thread> threads;
  threads.reserve((size_t)n);
  int started = 0;
  for (; started < n; ++started) {
    const int t = started;
    try {
      threads.emplace_back([&guarded, &body, t] { guarded([&] { body(t); }); });
    } catch (const std::system_error&) {
      break;  // no more threads to be had: this one does the rest
    }
  }
  guarded(meanwhile);
  for (int t = started; t < n; ++t) guarded([&] { body(t); });
  for (std::thread& t : threads) t.join();
  if (first) std::rethrow_exception(first);
}

class HostStaging {
 public:
  static constexpr size_t kBlock = (size_t)2 << 20;  // 2 MB (36 us on the bus), 16 of them: 32 MB of pinned memory
  static constexpr int kBlocks = 16;                 // two per thread

  HostStaging() {}
  HostStaging(const HostStaging&) = delete;
  HostStaging& operator=(const HostStaging&) = delete;
  ~HostStaging() { release(); }

  // blocks of at least `bytes`; on_device: their counterparts in device memory as well (data that a kernel spreads out)
  void reserve(size_t bytes, bool on_device) {
    bytes = (std::max(bytes, kBlock) + 255) & ~(size_t)255;
    if (bytes > block_) {
      release();
      HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&host_), bytes * kBlocks, hipHostMallocDefault));
      block_ = bytes;
      for (hipEvent_t& e : event_) HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    }
    if (on_device && !device_) HIP_CHECK(hipMalloc(reinterpret_cast<void**>(&device_), block_ * kBlocks));
  }
  size_t block() const { return block_; }
  // The call that needed the blocks is over: they stay for the next one, within the process's bounds.  (keep = false:
  // they do not.)
  void end(bool keep) {
    if (!host_) return;
    const size_t pinned = block_ * kBlocks, device = device_ ? pinned : 0;
    if (keep && pinned == counted_pinned_ && device == counted_device_) return;
    uncount();
    if (keep && kept_pinned_memory.take(pinned)) {
      counted_pinned_ = pinned;
      if (device == 0 || kept_device_memory.take(device)) {
        counted_device_ = device;
        return;
      }
    }
    release();
  }

  // Host to device, `block` bytes at a time: fill(to, at, n) puts bytes [at, at + n) of the transfer into pinned memory;
  // they are copied to target(at, n), or to the block's counterpart in device memory where that is null; after(there,
  // at, n) may launch work on them.  `meanwhile` runs on the calling thread, which with caller_too is one of the threads
  // as well.  Everything is on `stream` on return.
  template <typename Fill, typename Target, typename After, typename Meanwhile>
  void send(hipStream_t stream, size_t total, size_t block, Fill&& fill, Target&& target, After&& after, Meanwhile&& meanwhile,
            int most_threads = kBlocks / 2, bool caller_too = false) {
    int device = 0;
    HIP_CHECK(hipGetDevice(&device));
    const int threads = std::min(host_threads(total, block), most_threads);
    run(threads, total, stream, [&](int t) {
      HIP_CHECK(hipSetDevice(device));
      int use = 0;
      for (size_t at = (size_t)t * block; at < total; at += (size_t)threads * block, ++use) {
        const int slot = 2 * t + (use & 1);
        const size_t n = std::min(block, total - at);
        if (use >= 2) HIP_CHECK(hipEventSynchronize(event_[slot]));  // (the copy out of it two rounds ago)
        unsigned char* from = host_ + (size_t)slot * block_;
        fill(from, at, n);
        unsigned char* to = target(at, n);
        if (!to) to = device_ + (size_t)slot * block_;
        HIP_CHECK(hipMemcpyAsync(to, from, n, hipMemcpyHostToDevice, stream));
        after(to, at, n);
        HIP_CHECK(hipEventRecord(event_[slot], stream));
      }
    }, meanwhile, caller_too);
  }
  template <typename Fill, typename Target, typename After>
  void send(hipStream_t stream, size_t total, size_t block, Fill&& fill, Target&& target, After&& after) {
    send(stream, total, block, fill, target, after, [] {});
  }

  // Device to host: drain(from, at, n) takes bytes [at, at + n) of the transfer out of pinned memory, on several threads
  // at once if `side_by_side`, else in ascending order on one.  `meanwhile` runs on the calling thread.
  template <typename Drain, typename Meanwhile>
  void fetch(hipStream_t stream, const unsigned char* source, size_t total, bool side_by_side, Drain&& drain, Meanwhile&& meanwhile) {
    int device = 0;
    HIP_CHECK(hipGetDevice(&device));
    const size_t block = block_;
    const int threads = side_by_side ? std::min(host_threads(total, block), kBlocks / 2) : 1;
    const size_t stride = (size_t)threads * block;
    run(threads, total, stream, [&](int t) {
      HIP_CHECK(hipSetDevice(device));
      auto ask = [&](size_t at, int use) {
        const int slot = 2 * t + (use & 1);
        HIP_CHECK(hipMemcpyAsync(host_ + (size_t)slot * block_, source + at, std::min(block, total - at), hipMemcpyDeviceToHost, stream));
        HIP_CHECK(hipEventRecord(event_[slot], stream));
      };
      int use = 0;
      const size_t begin = (size_t)t * block;
      if (begin < total) ask(begin, 0);
      for (size_t at = begin; at < total; at += stride, ++use) {
        if (at + stride < total) ask(at + stride, use + 1);
        const int slot = 2 * t + (use & 1);
        HIP_CHECK(hipEventSynchronize(event_[slot]));
        drain(host_ + (size_t)slot * block_, at, std::min(block, total - at));
      }
    }, meanwhile);
  }

 private:
  // (one thread's worth of work is done by the calling thread; after a failure nothing may still be on its way
  // through the blocks)
  template <typename Body, typename Meanwhile>
  void run(int threads, size_t total, hipStream_t stream, Body&& body, Meanwhile&& meanwhile, bool caller_too = false) {
    try {
      if (threads <= 1) {
        if (total > 0) body(0);
        meanwhile();
      } else if (caller_too) {
        run_on_threads(threads - 1, [&](int t) { body(t + 1); }, [&] {
          body(0);
          meanwhile();
        });
      } else {
        run_on_threads(threads, body, meanwhile);
      }
    } catch (...) {
      (void)hipStreamSynchronize(stream);
      throw;
    }
  }
  void uncount() {
    kept_pinned_memory.give_back(counted_pinned_);
    kept_device_memory.give_back(counted_device_);
    counted_pinned_ = counted_device_ = 0;
  }
  void release() {
    uncount();
    for (hipEvent_t& e : event_) {
      if (e) (void)hipEventDestroy(e);
      e = nullptr;
    }
    if (host_) (void)hipHostFree(host_);
    if (device_) (void)hipFree(device_);
    host_ = device_ = nullptr;
    block_ = 0;
  }

  unsigned char* host_ = nullptr;
  unsigned char* device_ = nullptr;
  size_t block_ = 0;
  size_t counted_pinned_ = 0, counted_device_ = 0;
  hipEvent_t event_[kBlocks] = {};
};

}  // namespace cuhnsw_amd
