// Device memory to ordinary host memory, for whoever reads parameters, gradients or results back.
// A plain copy to pageable memory goes through the runtime's own bounce buffer on the calling thread,
// which also takes the page faults of a freshly allocated destination: 12 GB/s on one MI355X host, where
// the link does 55.  Here the link fills a small ring of pinned slots and a few threads carry them on,
// so that copying and first touch of the destination run beside the transfer and beside each other.
// One ring and one set of threads per process, made by the first large read and gone with the last
// object that holds them.
#ifndef CAVS_HOST_READBACK_H_
#define CAVS_HOST_READBACK_H_

#include <condition_variable>
#include <cstddef>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "device.h"

namespace cavs {

class ReadbackPool {
 public:
  static std::shared_ptr<ReadbackPool> shared();
  ~ReadbackPool();
  // `events`: one per slot, of the device the stream belongs to
  void read(char *host, const char *dev, size_t bytes, void *const streams[2], const std::vector<void *> &events);
  // Four megabytes per slot, carried on in pieces of one: a copy and its event cost about 15 us besides the
  // slot's 73 on the link, which the other stream's copy covers; short pieces so that the last ones end
  // together.  89 MB in 2.2 ms; 2.95 on one stream with slots of a megabyte.
  static constexpr size_t kSlot = size_t(4) << 20, kPiece = size_t(1) << 20;
  static constexpr int kSlots = 8;

 private:
  ReadbackPool();
  // One read.  Everything in here is guarded by m_; a piece takes some hundred microseconds.
  struct Job {
    char *host = nullptr;
    size_t bytes = 0;
    long pieces = 0;
    const std::vector<void *> *events = nullptr;
    long queued = 0, arrived = 0;         // chunks on their way, chunks known to be in their slots
    long next = 0, done = 0;              // pieces taken, carried on
    long slot_pieces[kSlots] = {};        // pieces of this slot carried on so far
    bool waits = false;                   // somebody waits for chunk `arrived` already
    bool failed = false;
    bool can_take() const { return !failed && next < pieces && next / (long)(kSlot / kPiece) < queued; }
  };
  void carry(std::unique_lock<std::mutex> &lock, Job &j);
  void thread_main();

  std::mutex one_read_;  // the ring serves one read at a time
  std::mutex m_;
  std::condition_variable more_, progress_;  // there may be pieces to take; pieces were carried on, a chunk has arrived
  Job *job_ = nullptr;
  int inside_ = 0;       // threads that hold job_
  bool stop_ = false;
  PinnedArray<char> ring_;
  std::vector<std::thread> threads_;  // as many as could be had: none is enough
};

// What one engine or executor reads through.
class Readback {
 public:
  ~Readback();
  // `bytes` of `dev` are at `host` when this returns; waits for what `stream` holds before it.
  void read(void *host, const void *dev, size_t bytes, void *stream);

 private:
  std::shared_ptr<ReadbackPool> pool_;
  std::vector<void *> events_;
  void *side_ = nullptr, *begin_ = nullptr;  // every other chunk of a large read
  PinnedArray<char> small_;
};

}  // namespace cavs
#endif
