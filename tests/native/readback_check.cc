// Reads through cavs_amd/host/readback.cc over a stand-in for the device: streams are queues that a thread each
// works off, in order, some time after the call; a copy or a wait can be told to fail.  Exits with 0 and a line per
// scenario if every read gave the bytes it was asked for or the error it should.
#include <dlfcn.h>
#include <pthread.h>

#include <atomic>
#include <cerrno>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

#include "readback.h"

namespace {
bool g_no_threads = false;  // the reader's side gets no thread, as at a limit
thread_local bool t_device = false;
}  // namespace
#ifndef CHECK_UNDER_TSAN
extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg) {
  typedef int (*Fn)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
  static Fn real = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "pthread_create"));
  return g_no_threads && !t_device ? EAGAIN : real(t, a, f, arg);
}
#endif

namespace {
struct Stream {
  std::mutex m;
  std::condition_variable cv;
  std::deque<std::function<void()>> q;
  bool busy = false, stop = false;
  std::thread t;
  void run() {
    std::unique_lock<std::mutex> lock(m);
    for (;;) {
      cv.wait(lock, [this] { return stop || !q.empty(); });
      if (q.empty()) return;
      auto f = std::move(q.front());
      q.pop_front();
      busy = true;
      lock.unlock();
      f();
      lock.lock();
      busy = false;
      cv.notify_all();
    }
  }
  Stream() {
    t_device = true;
    t = std::thread([this] { run(); });
    t_device = false;
  }
  void push(std::function<void()> f) {
    std::lock_guard<std::mutex> lock(m);
    q.push_back(std::move(f));
    cv.notify_all();
  }
  void drain() {
    std::unique_lock<std::mutex> lock(m);
    cv.wait(lock, [this] { return q.empty() && !busy; });
  }
  ~Stream() {
    {
      std::lock_guard<std::mutex> lock(m);
      stop = true;
    }
    cv.notify_all();
    t.join();
  }
};
struct Event {
  std::mutex m;
  std::condition_variable cv;
  long recorded = 0, over = 0;
};
std::mutex g_m;
long g_fail_copy = -1, g_fail_sync = -1, g_fail_alloc = 0;  // countdown to the call that fails (-1: none)
std::atomic<long> g_pinned{0};  // allocations of pinned memory that stand
bool counts_down(long &n) {
  std::lock_guard<std::mutex> lock(g_m);
  return n >= 0 && n-- == 0;
}
void set(long copy, long sync) {
  std::lock_guard<std::mutex> lock(g_m);
  g_fail_copy = copy;
  g_fail_sync = sync;
}
}  // namespace

extern "C" {
const char *cavs_last_error(void) { return "told to fail"; }
int cavs_host_alloc(void **p, size_t n) {
  if (g_fail_alloc) return CAVS_ENOMEM;
  *p = std::malloc(n);
  g_pinned++;
  return CAVS_OK;
}
int cavs_host_free(void *p) {
  if (p) g_pinned--;
  std::free(p);
  return CAVS_OK;
}
int cavs_malloc(void **, size_t) { return CAVS_ENOMEM; }
int cavs_free(void *) { return CAVS_OK; }
int cavs_stream_create(void **s) {
  *s = new Stream;
  return CAVS_OK;
}
int cavs_stream_destroy(void *s) {
  delete static_cast<Stream *>(s);
  return CAVS_OK;
}
int cavs_stream_sync(void *s) {
  static_cast<Stream *>(s)->drain();
  return CAVS_OK;
}
int cavs_event_create(void **e) {
  *e = new Event;
  return CAVS_OK;
}
int cavs_event_destroy(void *e) {
  delete static_cast<Event *>(e);
  return CAVS_OK;
}
int cavs_event_record(void *ev, void *s) {
  Event *e = static_cast<Event *>(ev);
  long mine;
  {
    std::lock_guard<std::mutex> lock(e->m);
    mine = ++e->recorded;
  }
  static_cast<Stream *>(s)->push([e, mine] {
    std::lock_guard<std::mutex> lock(e->m);
    e->over = mine;
    e->cv.notify_all();
  });
  return CAVS_OK;
}
int cavs_event_sync(void *ev) {
  Event *e = static_cast<Event *>(ev);
  std::unique_lock<std::mutex> lock(e->m);
  const long upto = e->recorded;
  e->cv.wait(lock, [&] { return e->over >= upto; });
  return counts_down(g_fail_sync) ? CAVS_EHIP : CAVS_OK;
}
int cavs_stream_wait_event(void *, void *e) { return cavs_event_sync(e); }
int cavs_memcpy_d2h(void *dst, const void *src, size_t n, void *s) {
  if (counts_down(g_fail_copy)) return CAVS_EHIP;
  static_cast<Stream *>(s)->push([=] {
    std::this_thread::sleep_for(std::chrono::microseconds(n / 100000));
    std::memcpy(dst, src, n);
  });
  return CAVS_OK;
}
}

namespace {
std::vector<char> pattern(size_t n, unsigned seed) {
  std::vector<char> v(n);
  for (size_t i = 0; i < n; i += 61) v[i] = (char)((i * 2654435761u + seed) >> 13);
  if (n) v[n - 1] = (char)(seed + 5);
  return v;
}
void expect(bool ok, const char *what) {
  std::printf("%s: %s\n", what, ok ? "ok" : "WRONG");
  std::fflush(stdout);
  if (!ok) std::exit(1);
}
bool reads(cavs::Readback &r, size_t n, unsigned seed) {
  Stream s;
  const std::vector<char> dev = pattern(n, seed);
  std::vector<char> host(n, 1);
  Stream second;
  r.read(host.data(), dev.data(), n, &s, seed & 1 ? &second : nullptr);
  return host == dev;
}
bool fails(cavs::Readback &r, size_t n) {
  try {
    return !reads(r, n, 3) && false;
  } catch (const cavs::Error &) {
    return true;
  }
}
}  // namespace

int main(int argc, char **argv) {
  const bool threadless = argc > 1 && !std::strcmp(argv[1], "threadless"), ringless = argc > 1 && !std::strcmp(argv[1], "ringless");
  const size_t M = size_t(1) << 20;
  g_fail_alloc = ringless;
  g_no_threads = threadless;
  {
  cavs::Readback a, b;
  expect(reads(a, 100 * M + 8, 2) && g_pinned == 0, "plain copies first");
  expect(reads(a, 30 * M, 2) && g_pinned == (ringless ? 0 : 1), "the ring when it would have paid");
  if (!ringless) {
    expect(reads(a, 1, 1) && reads(a, 100, 1) && reads(a, 256 << 10, 2), "small");
  }
  expect(reads(a, (256 << 10) + 4, 4) && reads(a, M, 5) && reads(a, 4 * M, 6) && reads(a, 4 * M + 4, 7), "up to a slot and beyond");
  expect(reads(a, 33 * M + 12, 8) && reads(a, 32 * M, 9) && reads(a, 101 * M - 4, 10), "more than the ring holds");
  bool ok[2] = {true, true};
  t_device = true;
  std::thread other([&] {
    for (int i = 0; i < 6; i++) ok[1] = ok[1] && reads(b, (5 + 13 * i) * M + 4 * i, 20 + i);
  });
  t_device = false;
  for (int i = 0; i < 6; i++) ok[0] = ok[0] && reads(a, (40 - 6 * i) * M + 4, 40 + i);
  other.join();
  expect(ok[0] && ok[1], "two readers at a time");
  if (ringless) return 0;
  for (long k : argc > 1 ? std::vector<long>{1, 9} : std::vector<long>{0, 1, 5, 9, 20}) {
    set(k, -1);
    expect(fails(a, 90 * M), "a copy that fails");
    set(-1, k);
    expect(fails(a, 90 * M), "a wait that fails");
    set(-1, -1);
    expect(reads(a, 37 * M, 60), "and a read after it");
  }
  for (int i = 0; i < 3; i++) {
    cavs::Readback c;
    expect(reads(c, 9 * M, 70 + i), "a reader of its own");
  }
  }
  for (int i = 0; i < 300 && g_pinned > 0; i++) std::this_thread::sleep_for(std::chrono::milliseconds(20));
  expect(g_pinned == 0, "the ring goes back when nobody reads any more");
  cavs::Readback d;
  expect(reads(d, 40 * M, 80) && g_pinned == 1, "and comes again");
  return 0;
}
