// Device memory to ordinary host memory, for whoever reads parameters, gradients or results back.
// A plain copy to pageable memory goes through the runtime's own bounce buffer on the calling thread,
// which also takes the page faults of a freshly allocated destination: 12 GB/s on one MI355X host, where
// the link does 55.  Here the link fills a small ring of pinned slots and a few threads carry them on,
// so that copying and first touch of the destination run beside the transfer and beside each other.
// One ring and one set of threads per process.  Making them costs some 10 ms (the runtime's first copy to pinned
// memory alone 6), so they are made once a process has read as much by plain copies as would have paid for them,
// and sessions that follow each other find them there; some time after the last of these the memory goes back
// and the threads end.
#ifndef CAVS_HOST_READBACK_H_
#define CAVS_HOST_READBACK_H_

#include <condition_variable>
#include <cstddef>
#include <mutex>
#include <vector>

#include "device.h"

namespace cavs {

class ReadbackPool {
 public:
  static ReadbackPool &instance();  // (lives until the process ends)
  // Who reads through the pool attaches to it first: false where a plain copy is the better choice so far, `bytes`
  // being what the caller is about to read.
  bool attach(size_t bytes);
  void detach();
  // `events`: one per slot, of the device the stream belongs to
  void read(char *host, const char *dev, size_t bytes, void *const streams[2], const std::vector<void *> &events);
  // Four megabytes per slot, carried on in pieces of one: a copy and its event cost about 15 us besides the
  // slot's 73 on the link, which the other stream's copy covers; short pieces so that the last ones end
  // together.  89 MB in 2.2 ms; 2.95 on one stream with slots of a megabyte.
  static constexpr size_t kSlot = size_t(4) << 20, kPiece = size_t(1) << 20;
  static constexpr int kSlots = 8;

 private:
  ReadbackPool() = default;
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
  void staff(long pieces);

  std::mutex one_read_;  // the ring serves one read at a time
  std::mutex m_;
  std::condition_variable more_, progress_;  // there may be pieces to take; pieces were carried on, a chunk has arrived
  Job *job_ = nullptr;
  int inside_ = 0;       // threads that hold job_
  int threads_ = 0;      // as many as could be had: none is enough
  int users_ = 0;        // who has attached
  size_t plain_ = 0;     // bytes of large reads that went by plain copies
  bool exiting_ = false; // the process is on its way out: no more calls into the runtime
  PinnedArray<char> ring_;
};

// What one engine or executor reads through.
class Readback {
 public:
  ~Readback();
  // `bytes` of `dev` are at `host` when this returns; waits for what `stream` holds before it.  `second`: another
  // stream of the caller's with nothing on it (null: large reads make one; a stream more costs up to 3 ms).
  void read(void *host, const void *dev, size_t bytes, void *stream, void *second);

 private:
  bool attached_ = false;
  std::vector<void *> events_;
  void *side_ = nullptr, *begin_ = nullptr;  // every other chunk of a large read
  PinnedArray<char> small_;
};

}  // namespace cavs
#endif
