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
constexpr int kThreads = 11;
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

// Takes pieces in order until there are none left.  The caller's own turn ends early when the next piece
// is not on its way yet: queueing it is the caller's work.
void ReadbackPool::work(Job &j, bool caller) {
  constexpr long per = kSlot / kPiece;
  for (;;) {
    long i = j.next.load(std::memory_order_relaxed);
    if (i >= j.pieces) return;
    const long chunk = i / per;
    if (chunk >= j.queued.load(std::memory_order_acquire)) {
      if (caller || j.failed.load(std::memory_order_relaxed)) return;
      std::this_thread::yield();
      continue;
    }
    if (!j.next.compare_exchange_weak(i, i + 1)) continue;
    const int slot = (int)(chunk % kSlots);
    if (j.arrived.load(std::memory_order_acquire) <= chunk) {
      if (cavs_event_sync((*j.events)[slot]) != CAVS_OK) j.failed = true;
      long seen = j.arrived.load(std::memory_order_relaxed);
      // (chunks of one stream arrive in order, but the other stream's last one may still be under way)
      if (seen == chunk) j.arrived.compare_exchange_strong(seen, chunk + 1, std::memory_order_release);
    }
    const size_t at = (size_t)i * kPiece;
    std::memcpy(j.host + at, ring_.get() + slot * kSlot + at % kSlot, std::min(kPiece, j.bytes - at));
    j.slot_pieces[slot].fetch_add(1, std::memory_order_release);
    j.done.fetch_add(1, std::memory_order_release);
  }
}

void ReadbackPool::thread_main() {
  std::unique_lock<std::mutex> lock(m_);
  for (;;) {
    wake_.wait(lock, [this] { return stop_ || (job_ && job_->next.load() < job_->pieces); });
    if (stop_) return;
    Job *j = job_;
    inside_++;
    lock.unlock();
    work(*j, false);
    lock.lock();
    if (--inside_ == 0) idle_.notify_all();
  }
}

void ReadbackPool::read(char *host, const char *dev, size_t bytes, void *const streams[2], const std::vector<void *> &events) {
  std::lock_guard<std::mutex> only(one_read_);
  Job j;
  j.host = host;
  j.bytes = bytes;
  j.pieces = (long)((bytes + kPiece - 1) / kPiece);
  j.events = &events;
  for (auto &s : j.slot_pieces) s = 0;
  {
    std::lock_guard<std::mutex> lock(m_);
    job_ = &j;
  }
  wake_.notify_all();
  int rc = CAVS_OK;
  const long chunks = (long)((bytes + kSlot - 1) / kSlot);
  for (long i = 0; i < chunks && rc == CAVS_OK; i++) {
    const int slot = (int)(i % kSlots);
    // (only the last chunk of a read is shorter than its slot)
    while (j.slot_pieces[slot].load(std::memory_order_acquire) < i / kSlots * (long)(kSlot / kPiece) && !j.failed.load(std::memory_order_relaxed))
      work(j, true);
    const size_t at = (size_t)i * kSlot;
    rc = cavs_memcpy_d2h(ring_.get() + slot * kSlot, dev + at, std::min(kSlot, bytes - at), streams[i & 1]);
    if (rc == CAVS_OK) rc = cavs_event_record(events[slot], streams[i & 1]);
    if (rc == CAVS_OK) j.queued.store(i + 1, std::memory_order_release);
  }
  if (rc != CAVS_OK) j.failed = true;
  work(j, true);
  while (j.done.load(std::memory_order_acquire) < (rc == CAVS_OK ? j.pieces : j.next.load())) std::this_thread::yield();
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
  if (begin_) cavs_event_destroy(begin_);
  if (side_) cavs_stream_destroy(side_);
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
  void *streams[2] = {stream, stream};
  if (bytes > ReadbackPool::kSlot) {
    if (!side_) check(cavs_stream_create(&side_));
    if (!begin_) check(cavs_event_create(&begin_));
    check(cavs_event_record(begin_, stream));
    check(cavs_stream_wait_event(side_, begin_));
    streams[1] = side_;
  }
  pool_->read(static_cast<char *>(host), static_cast<const char *>(dev), bytes, streams, events_);
}

}  // namespace cavs
