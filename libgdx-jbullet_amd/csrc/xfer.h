// xfer.h — copies between a caller's pageable host memory and the device.
//
// A copy goes through two pinned slots of the context: while one slot is on its way over the bus, the context's copying
// threads and the calling thread fill or empty the other.  One thread moves about 10 GB/s and pays the page faults of
// a fresh destination alone; the bus does about 55.
// The body records of 4,096 worlds of towers (132 MB) into fresh memory: 12.6 ms before, 2.7 ms now; into memory that is
// mapped 48 GB/s.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <condition_variable>
#include <functional>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace jbg {

// a few threads of one context that share large memory copies with the calling thread; they sleep between copies and
// end with the context
class CopyPool {
 public:
  ~CopyPool();
  void copy(void* dst, const void* src, size_t bytes);

 private:
  struct Job;
  void start();
  void loop();
  std::vector<std::thread> threads_;
  bool started_ = false, stop_ = false;
  std::mutex mu_;
  std::condition_variable cv_;
  std::shared_ptr<Job> job_;
  std::atomic<unsigned long long> jobs_{0};
};

class HostCopy {
 public:
  ~HostCopy();
  // queues dev[0, bytes) = host[0, bytes) on the stream; the host memory has to live until the stream gets there
  void send(hipStream_t s, void* dev, const void* host, size_t bytes);
  // host[0, bytes) = dev[0, bytes) after everything queued before; returns when the host memory holds it
  void fetch(hipStream_t s, void* host, const void* dev, size_t bytes);
  // as fetch, the bytes made by fill(slot, offset, bytes), which queues on the stream what writes [offset, offset +
  // bytes) of the result to the pinned (device-visible) slot; pieces are multiples of `unit`
  void fetchWith(hipStream_t s, void* host, size_t bytes, size_t unit,
                 const std::function<void(void*, size_t, size_t)>& fill);

 private:
  char* slot(int k, size_t bytes);
  char* slots_[2] = {nullptr, nullptr};
  size_t size_[2] = {0, 0};
  hipEvent_t ready_[2] = {};
  bool used_[2] = {false, false};
  CopyPool pool_;
};

}  // namespace jbg
