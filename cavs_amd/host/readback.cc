#include "readback.h"

#include <algorithm>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <string>
#include <system_error>
#include <thread>

namespace cavs {

namespace {
// below this a plain copy is as fast: the pool's threads have to be woken up first
constexpr size_t kPlain = size_t(1) << 20;
// Up to here through a pinned buffer of the reader's own: the runtime stages such a copy itself, at the
// price of one more wait (one Tree-LSTM sentence, graph_out back: 127 us; 114 with this and the feeds on the
// idle stream).
constexpr size_t kSmall = size_t(256) << 10;
// Threads besides the caller's: a core copies and faults in about 10 GB/s, the link does 55 (89 MB with eleven
// 2.20 ms, with five 2.23).
constexpr int kThreads = 5;
// A plain copy takes 0.03 (11 MB) to 0.07 ms a megabyte longer: from here on a process has paid what the ring costs.
constexpr size_t kWorth = size_t(128) << 20;
// How long the ring stays without anybody attached to it.
constexpr auto kKeep = std::chrono::seconds(2);
}  // namespace

ReadbackPool &ReadbackPool::instance() {
  static ReadbackPool *pool = [] {
    auto *p = new ReadbackPool;  // (its threads may outlive every static object)
    std::atexit([] {
      ReadbackPool &q = instance();
      std::lock_guard<std::mutex> lock(q.m_);
      q.exiting_ = true;
    });
    return p;
  }();
  return *pool;
}

bool ReadbackPool::attach(size_t bytes) {
  std::lock_guard<std::mutex> lock(m_);
  if (exiting_) return false;
  if (ring_.capacity() == 0) {
    if (plain_ + bytes <= kWorth) {
      plain_ += bytes;
      return false;
    }
    try {
      ring_.reserve(kSlot * kSlots);
    } catch (const Error &) {  // no pinned memory for a ring: a plain copy will do
      return false;
    }
  }
  users_++;
  return true;
}

void ReadbackPool::detach() {
  std::lock_guard<std::mutex> lock(m_);
  if (--users_ > 0) return;
  if (threads_ == 0 && !exiting_) ring_.release();  // (else the threads see to it)
  more_.notify_all();
}

// Call with m_ held.  Threads for so many pieces, as far as they can be had.
void ReadbackPool::staff(long pieces) {
  const int spare = std::max(1, (int)std::thread::hardware_concurrency() - 1);
  try {
    while (threads_ < std::min<long>({kThreads, spare, pieces - 1})) {
      std::thread([this] { thread_main(); }).detach();
      threads_++;
    }
  } catch (const std::system_error &) {
  }
}

// Takes one piece on; call with j.can_take().  Pieces are taken in order, and one thread at a time waits for the
// link, for the first chunk that is not known to have arrived.
void ReadbackPool::carry(std::unique_lock<std::mutex> &lock, Job &j) {
  const long i = j.next++, chunk = i / (long)(kSlot / kPiece);
  const int slot = (int)(chunk % kSlots);
  while (j.arrived <= chunk && !j.failed) {
    if (j.waits) {
      progress_.wait(lock);
      continue;
    }
    j.waits = true;
    void *event = (*j.events)[j.arrived % kSlots];
    lock.unlock();
    const int rc = cavs_event_sync(event);
    lock.lock();
    j.waits = false;
    j.arrived++;
    if (rc != CAVS_OK) j.failed = true;
    progress_.notify_all();
  }
  if (!j.failed) {
    const size_t at = (size_t)i * kPiece;
    lock.unlock();
    std::memcpy(j.host + at, ring_.get() + slot * kSlot + at % kSlot, std::min(kPiece, j.bytes - at));
    lock.lock();
  }
  j.slot_pieces[slot]++;
  j.done++;
  progress_.notify_all();
}

void ReadbackPool::thread_main() {
  std::unique_lock<std::mutex> lock(m_);
  for (;;) {
    // (the system's clock: gcc 11's thread sanitizer does not know the wait by the steady one)
    const bool more = more_.wait_until(lock, std::chrono::system_clock::now() + kKeep, [this] { return job_ && job_->can_take(); });
    if (!more && users_ > 0) continue;
    if (!more) break;
    Job &j = *job_;
    inside_++;
    while (j.can_take()) carry(lock, j);
    inside_--;
    progress_.notify_all();
  }
  if (--threads_ == 0 && !exiting_) ring_.release();
}

void ReadbackPool::read(char *host, const char *dev, size_t bytes, void *const streams[2], const std::vector<void *> &events) {
  std::lock_guard<std::mutex> only(one_read_);
  Job j;
  j.host = host;
  j.bytes = bytes;
  j.pieces = (long)((bytes + kPiece - 1) / kPiece);
  j.events = &events;
  int rc = CAVS_OK;
  const long chunks = (long)((bytes + kSlot - 1) / kSlot);
  std::unique_lock<std::mutex> lock(m_);
  staff(j.pieces);
  job_ = &j;
  // (the caller carries pieces on as well, but queueing the next chunk comes first)
  auto work_until = [&](auto over) {
    while (!over()) {
      if (j.can_take()) carry(lock, j);
      else progress_.wait(lock);
    }
  };
  for (long i = 0; i < chunks && rc == CAVS_OK; i++) {
    const int slot = (int)(i % kSlots);
    // (only the last chunk of a read is shorter than its slot)
    work_until([&] { return j.failed || j.slot_pieces[slot] >= i / kSlots * (long)(kSlot / kPiece); });
    if (j.failed) break;
    lock.unlock();
    const size_t at = (size_t)i * kSlot;
    rc = cavs_memcpy_d2h(ring_.get() + slot * kSlot, dev + at, std::min(kSlot, bytes - at), streams[i & 1]);
    if (rc == CAVS_OK) rc = cavs_event_record(events[slot], streams[i & 1]);
    lock.lock();
    if (rc == CAVS_OK) j.queued = i + 1;
    else j.failed = true;
    more_.notify_all();
  }
  work_until([&] { return j.failed || j.done == j.pieces; });
  job_ = nullptr;
  progress_.wait(lock, [this] { return inside_ == 0; });
  lock.unlock();
  if (!j.failed) return;
  const std::string why = rc != CAVS_OK ? cavs_last_error() : "";
  for (int k = 0; k < 2; k++) (void)cavs_stream_sync(streams[k]);  // (nothing of it still on its way into the ring)
  fail(rc != CAVS_OK ? rc : CAVS_EHIP, "reading device memory back failed" + (why.empty() ? why : ": " + why));
}

Readback::~Readback() {
  for (void *e : events_) cavs_event_destroy(e);
  if (begin_) cavs_event_destroy(begin_);
  if (side_) cavs_stream_destroy(side_);
  if (attached_) ReadbackPool::instance().detach();
}

void Readback::read(void *host, const void *dev, size_t bytes, void *stream, void *second) {
  if (bytes <= kSmall) {
    small_.reserve(bytes < 4096 ? 4096 : 2 * bytes < kSmall ? 2 * bytes : kSmall);
    check(cavs_memcpy_d2h(small_.get(), dev, bytes, stream));
    check(cavs_stream_sync(stream));
    std::memcpy(host, small_.get(), bytes);
    return;
  }
  ReadbackPool &pool = ReadbackPool::instance();
  if (bytes >= kPlain && !attached_) attached_ = pool.attach(bytes);
  if (bytes < kPlain || !attached_) {
    check(cavs_memcpy_d2h(host, dev, bytes, stream));
    check(cavs_stream_sync(stream));
    return;
  }
  while (events_.size() < (size_t)ReadbackPool::kSlots) {
    void *e = nullptr;
    check(cavs_event_create(&e));
    events_.push_back(e);
  }
  void *streams[2] = {stream, stream};
  if (bytes > ReadbackPool::kSlot) {
    if (!second && !side_) check(cavs_stream_create(&side_));
    if (!begin_) check(cavs_event_create(&begin_));
    streams[1] = second ? second : side_;
    check(cavs_event_record(begin_, stream));
    check(cavs_stream_wait_event(streams[1], begin_));
  }
  pool.read(static_cast<char *>(host), static_cast<const char *>(dev), bytes, streams, events_);
}

}  // namespace cavs
