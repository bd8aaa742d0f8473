#include "readback.h"

#include <algorithm>
#include <cstring>

namespace cavs {

namespace {
// below this a plain copy is as fast: the pool's threads have to be woken up first
constexpr size_t kPlain = size_t(1) << 20;
// Up to here through a pinned buffer of the reader's own: the runtime stages such a copy itself, at the
// price of one more wait (one Tree-LSTM sentence, graph_out back: 127 us; 114 with this and the feeds on the
// idle stream).
constexpr size_t kSmall = size_t(256) << 10;
// Threads besides the caller's: a core copies and faults in about 10 GB/s, the link does 55.
constexpr int kThreads = 5;
}  // namespace

std::shared_ptr<ReadbackPool> ReadbackPool::shared() {
  static std::mutex m;
  static std::weak_ptr<ReadbackPool> pool;
  std::lock_guard<std::mutex> lock(m);
  std::shared_ptr<ReadbackPool> p = pool.lock();
  if (!p) {
    p.reset(new ReadbackPool);
    pool = p;
  }
  return p;
}

ReadbackPool::ReadbackPool() {
  ring_.reserve(kSlot * kSlots);
  const int spare = std::max(1, (int)std::thread::hardware_concurrency() - 1);
  for (int i = 0; i < std::min(kThreads, spare); i++) threads_.emplace_back([this] { thread_main(); });
}

ReadbackPool::~ReadbackPool() {
  {
    std::lock_guard<std::mutex> lock(m_);
    stop_ = true;
  }
  wake_.notify_all();
  for (std::thread &t : threads_) t.join();
}

// Takes chunks in order until there are none left.  The caller's own turn ends a chunk early when
// the next one is not on its way yet: queueing it is the caller's work.
void ReadbackPool::work(Job &j, bool caller) {
  for (;;) {
    long i = j.next.load(std::memory_order_relaxed);
    if (i >= j.chunks) return;
    if (i >= j.queued.load(std::memory_order_acquire)) {
      if (caller || j.failed.load(std::memory_order_relaxed)) return;
      std::this_thread::yield();
      continue;
    }
    if (!j.next.compare_exchange_weak(i, i + 1)) continue;
    const int slot = (int)(i % kSlots);
    if (cavs_event_sync((*j.events)[slot]) != CAVS_OK) j.failed = true;
    const size_t at = (size_t)i * kSlot;
    std::memcpy(j.host + at, ring_.get() + slot * kSlot, std::min(kSlot, j.bytes - at));
    j.slot_done[slot].store(i / kSlots + 1, std::memory_order_release);
    j.done.fetch_add(1, std::memory_order_release);
  }
}

void ReadbackPool::thread_main() {
  std::unique_lock<std::mutex> lock(m_);
  for (;;) {
    wake_.wait(lock, [this] { return stop_ || (job_ && job_->next.load() < job_->chunks); });
    if (stop_) return;
    Job *j = job_;
    inside_++;
    lock.unlock();
    work(*j, false);
    lock.lock();
    if (--inside_ == 0) idle_.notify_all();
  }
}

void ReadbackPool::read(char *host, const char *dev, size_t bytes, void *stream, const std::vector<void *> &events) {
  std::lock_guard<std::mutex> only(one_read_);
  Job j;
  j.host = host;
  j.bytes = bytes;
  j.chunks = (long)((bytes + kSlot - 1) / kSlot);
  j.events = &events;
  for (auto &s : j.slot_done) s = 0;
  {
    std::lock_guard<std::mutex> lock(m_);
    job_ = &j;
  }
  wake_.notify_all();
  int rc = CAVS_OK;
  for (long i = 0; i < j.chunks && rc == CAVS_OK; i++) {
    const int slot = (int)(i % kSlots);
    while (j.slot_done[slot].load(std::memory_order_acquire) < i / kSlots && !j.failed.load(std::memory_order_relaxed)) work(j, true);
    const size_t at = (size_t)i * kSlot;
    rc = cavs_memcpy_d2h(ring_.get() + slot * kSlot, dev + at, std::min(kSlot, bytes - at), stream);
    if (rc == CAVS_OK) rc = cavs_event_record(events[slot], stream);
    if (rc == CAVS_OK) j.queued.store(i + 1, std::memory_order_release);
  }
  if (rc != CAVS_OK) j.failed = true;
  work(j, true);
  while (j.done.load(std::memory_order_acquire) < (rc == CAVS_OK ? j.chunks : j.next.load())) std::this_thread::yield();
  {
    std::unique_lock<std::mutex> lock(m_);
    job_ = nullptr;
    idle_.wait(lock, [this] { return inside_ == 0; });
  }
  if (rc != CAVS_OK) check(rc);
  if (j.failed) fail(CAVS_EHIP, "reading device memory back failed");
}

Readback::~Readback() {
  for (void *e : events_) cavs_event_destroy(e);
}

void Readback::read(void *host, const void *dev, size_t bytes, void *stream) {
  if (bytes <= kSmall) {
    small_.reserve(bytes < 4096 ? 4096 : 2 * bytes < kSmall ? 2 * bytes : kSmall);
    check(cavs_memcpy_d2h(small_.get(), dev, bytes, stream));
    check(cavs_stream_sync(stream));
    std::memcpy(host, small_.get(), bytes);
    return;
  }
  if (bytes < kPlain) {
    check(cavs_memcpy_d2h(host, dev, bytes, stream));
    check(cavs_stream_sync(stream));
    return;
  }
  if (!pool_) pool_ = ReadbackPool::shared();
  while (events_.size() < (size_t)ReadbackPool::kSlots) {
    void *e = nullptr;
    check(cavs_event_create(&e));
    events_.push_back(e);
  }
  pool_->read(static_cast<char *>(host), static_cast<const char *>(dev), bytes, stream, events_);
}

}  // namespace cavs
