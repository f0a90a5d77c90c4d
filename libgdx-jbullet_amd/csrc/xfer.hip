// xfer.hip — see xfer.h.
#include "xfer.h"

#include <algorithm>
#include <atomic>
#include <cstring>

#include "internal.h"

namespace jbg {

namespace {
constexpr size_t kSlotBytes = 4u << 20;    // per slot at most
constexpr size_t kPieceBytes = 512u << 10;  // and at least, where there is more than one piece
constexpr size_t kPartBytes = 128u << 10;  // a thread's share at a time
constexpr size_t kPoolBytes = 512u << 10;  // smaller copies stay on the calling thread (waking one takes tens of us)
constexpr int kPoolSpins = 2000;           // polls for the next piece before a thread sleeps (some tens of us)
// Sends between these go through the runtime's own staging: the gradient of 4,096..65,536 samples (0.3..5 MB up) takes
// 98..289 us that way and 109..317 through the slots, 1,024 samples 86 and 76, 2^18 samples (20 MB) 838 and 788, 2^20
// 3645 and 2695.
constexpr size_t kSlotSend = 64u << 10;
constexpr size_t kPiecesSend = 8u << 20;
// fetches likewise: the 3 MB of keys of 10^6 boxes take as long either way, and the first costs the slots and threads
constexpr size_t kPiecesFetch = 4u << 20;
// four pieces or more, so that the bus and the threads work side by side
size_t pieceFor(size_t bytes) { return std::min(kSlotBytes, std::max(kPieceBytes, (bytes / 4 + 4095) / 4096 * 4096)); }
constexpr int kPoolThreads = 6;
}  // namespace

struct CopyPool::Job {
  char* dst;
  const char* src;
  size_t bytes;
  std::atomic<size_t> next{0}, done{0};
  void work() {
    for (;;) {
      const size_t at = next.fetch_add(kPartBytes);
      if (at >= bytes) return;
      const size_t n = std::min(kPartBytes, bytes - at);
      std::memcpy(dst + at, src + at, n);
      done.fetch_add(n);
    }
  }
};

void CopyPool::start() {
  if (started_) return;
  started_ = true;
  const int most = std::max(0, (int)std::thread::hardware_concurrency() / 2 - 1);
  try {
    for (int k = 0; k < std::min(kPoolThreads, most); k++) threads_.emplace_back([this] { loop(); });
  } catch (const std::exception&) {  // as many as there are
  }
}
CopyPool::~CopyPool() {
  {
    std::lock_guard<std::mutex> lock(mu_);
    stop_ = true;
  }
  cv_.notify_all();
  for (std::thread& t : threads_) t.join();
}
void CopyPool::loop() {
  unsigned long long seen = 0;
  for (;;) {
    std::shared_ptr<Job> job;
    for (int k = 0; k < kPoolSpins && jobs_.load(std::memory_order_relaxed) == seen; k++) __builtin_ia32_pause();
    {
      std::unique_lock<std::mutex> lock(mu_);
      cv_.wait(lock, [&] { return stop_ || jobs_ != seen; });
      if (stop_) return;
      seen = jobs_;
      job = job_;
    }
    if (job) job->work();
  }
}
void CopyPool::copy(void* dst, const void* src, size_t bytes) {
  if (bytes < kPoolBytes) {
    std::memcpy(dst, src, bytes);
    return;
  }
  start();
  auto job = std::make_shared<Job>();
  job->dst = (char*)dst;
  job->src = (const char*)src;
  job->bytes = bytes;
  {
    std::lock_guard<std::mutex> lock(mu_);
    job_ = job;
    jobs_++;
  }
  cv_.notify_all();
  job->work();
  while (job->done.load() != bytes) std::this_thread::yield();  // a thread still has its last part in hand
  std::lock_guard<std::mutex> lock(mu_);
  job_.reset();
}

HostCopy::~HostCopy() {
  for (int k = 0; k < 2; k++) {
    if (used_[k]) (void)hipEventSynchronize(ready_[k]);
    if (ready_[k]) (void)hipEventDestroy(ready_[k]);
    if (slots_[k]) (void)hipHostFree(slots_[k]);
  }
}
// slot k with room for `bytes`, its last transfer finished
char* HostCopy::slot(int k, size_t bytes) {
  if (!ready_[k]) JB_CHECK(hipEventCreateWithFlags(&ready_[k], hipEventDisableTiming));
  if (used_[k]) {
    JB_CHECK(hipEventSynchronize(ready_[k]));
    used_[k] = false;
  }
  if (bytes > size_[k]) {
    if (slots_[k]) (void)hipHostFree(slots_[k]);
    slots_[k] = nullptr;
    size_[k] = 0;
    size_t want = 64u << 10;
    while (want < bytes) want *= 2;
    JB_CHECK(hipHostMalloc((void**)&slots_[k], want, hipHostMallocDefault));
    size_[k] = want;
  }
  return slots_[k];
}
void HostCopy::send(hipStream_t s, void* dev, const void* host, size_t bytes) {
  if (bytes > kSlotSend && bytes < kPiecesSend) {
    JB_CHECK(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s));
    return;
  }
  int k = 0;
  const size_t piece = pieceFor(bytes);
  for (size_t at = 0; at < bytes; at += piece, k ^= 1) {
    const size_t n = std::min(piece, bytes - at);
    char* p = slot(k, n);
    pool_.copy(p, (const char*)host + at, n);
    JB_CHECK(hipMemcpyAsync((char*)dev + at, p, n, hipMemcpyHostToDevice, s));
    JB_CHECK(hipEventRecord(ready_[k], s));
    used_[k] = true;
  }
}
void HostCopy::fetchWith(hipStream_t s, void* host, size_t bytes, size_t unit,
                         const std::function<void(void*, size_t, size_t)>& fill) {
  const size_t piece = std::max(unit, pieceFor(bytes) / unit * unit);
  const size_t pieces = (bytes + piece - 1) / piece;
  auto start = [&](size_t i) {
    const int k = (int)(i & 1);
    const size_t at = i * piece, n = std::min(piece, bytes - at);
    fill(slot(k, n), at, n);
    JB_CHECK(hipEventRecord(ready_[k], s));
    used_[k] = true;
  };
  for (size_t i = 0; i < std::min<size_t>(pieces, 2); i++) start(i);
  for (size_t i = 0; i < pieces; i++) {
    const int k = (int)(i & 1);
    const size_t at = i * piece;
    char* p = slot(k, 1);  // waits for the piece
    pool_.copy((char*)host + at, p, std::min(piece, bytes - at));
    if (i + 2 < pieces) start(i + 2);
  }
}
void HostCopy::fetch(hipStream_t s, void* host, const void* dev, size_t bytes) {
  if (bytes > kSlotSend && bytes < kPiecesFetch) {
    JB_CHECK(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s));
    JB_CHECK(hipStreamSynchronize(s));
    return;
  }
  fetchWith(s, host, bytes, 1, [&](void* p, size_t at, size_t n) {
    JB_CHECK(hipMemcpyAsync(p, (const char*)dev + at, n, hipMemcpyDeviceToHost, s));
  });
}

}  // namespace jbg
