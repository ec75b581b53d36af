/*
 * fe_host_copy.h -- copies of host memory by several threads (the transfers' way between the
 * caller's arrays and the pinned slots).
 */
#ifndef FE_HOST_COPY_H
#define FE_HOST_COPY_H

#include <sched.h>
#include <stdint.h>
#include <string.h>
#include <unistd.h>
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>

namespace {

/* Copies of host memory by the caller and up to three helper threads, in chunks that whoever is
 * free takes next: a helper that has not woken yet (it can take longer than the copy) holds
 * nobody up.  The helpers sleep except between begin() and end(), when they poll for work.  One
 * copy at a time; a second caller copies by itself. */
class HostCopy {
 public:
  static constexpr int MAXH = 3;
  static constexpr size_t CHUNK = 256 << 10;      /* 10 us of one thread */
  /* helpers poll until end(); starts them on the first call */
  void begin() {
    /* asked before the mutex, which another thread may have held at the fork */
    const pid_t me = getpid(), owner = pid_;
    if (owner != 0 && owner != me) return;
    std::lock_guard<std::mutex> l(m_);
    if (pid_ == 0) {
      pid_ = me;
      cpu_set_t set;
      const int n = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : 1;
      nh_ = std::min(MAXH, n - 1);
      try {
        for (int i = 0; i < nh_; ++i) th_[i] = std::thread([this] { help(); });
      } catch (...) {                             /* no thread to be had: the ones there are do */
        int k = 0;
        while (k < nh_ && th_[k].joinable()) ++k;
        nh_ = k;
      }
    }
    if (pid_ != me) return;
    ++users_;
    cv_.notify_all();
  }
  void end() {
    if (pid_ != getpid()) return;
    std::lock_guard<std::mutex> l(m_);
    if (users_ > 0) --users_;
  }
  /* Ends the helpers; from then on a copy is the caller's alone.  A forked child has none to end. */
  void stop() {
    if (pid_ != getpid()) return;
    {
      std::lock_guard<std::mutex> l(m_);
      quit_ = true;
      pid_ = -1;
    }
    cv_.notify_all();
    for (auto &t : th_) if (t.joinable()) t.join();
  }
  void copy(void *dst, const void *src, size_t n) {
    if (n <= CHUNK || nh_ <= 0 || pid_ != getpid() || users_ <= 0 || !one_.try_lock()) {
      memcpy(dst, src, n);
      return;
    }
    const unsigned nc = (unsigned)((n + CHUNK - 1) / CHUNK);
    /* The ticket holds the copy's number and the next chunk: taking one is a compare-exchange, which
     * fails if either has moved on since the copy's addresses were read.  It shows no chunk while
     * the addresses change. */
    const uint64_t g = ((ticket_.load() >> 32) + 1) << 32;
    ticket_.store(g | 0xffffffffu);
    dst_.store((char *)dst);
    src_.store((const char *)src);
    n_.store(n);
    done_.store(0);
    ticket_.store(g);
    while (take()) {}
    while (done_.load() < nc) __builtin_ia32_pause();
    one_.unlock();
  }

 private:
  /* copies the next chunk of the current copy; false if there is none to take */
  bool take() {
    uint64_t t = ticket_.load();
    char *d = dst_.load();
    const char *s = src_.load();
    const size_t n = n_.load(), o = (t & 0xffffffffu) * CHUNK;
    if (o >= n) return false;
    if (!ticket_.compare_exchange_strong(t, t + 1)) return true;
    memcpy(d + o, s + o, std::min(CHUNK, n - o));
    done_.fetch_add(1);
    return true;
  }
  void help() {
    for (;;) {
      if (quit_) return;
      if (users_ > 0) {
        if (!take()) __builtin_ia32_pause();
        continue;
      }
      std::unique_lock<std::mutex> l(m_);
      cv_.wait(l, [&] { return quit_ || users_ > 0; });
      if (quit_) return;
    }
  }
  std::thread th_[MAXH];
  int nh_ = 0;
  std::atomic<pid_t> pid_{0};                     /* the process that has the helpers; -1 once they are ended */
  std::mutex m_, one_;
  std::condition_variable cv_;
  std::atomic<int> users_{0};
  std::atomic<bool> quit_{false};
  std::atomic<uint64_t> ticket_{0};
  std::atomic<unsigned> done_{0};
  std::atomic<char *> dst_{nullptr};
  std::atomic<const char *> src_{nullptr};
  std::atomic<size_t> n_{0};
};

/* Never destroyed: in a forked child the parent's sleeping helpers still count as waiters of the
 * condition variable, and its destructor would wait for them for ever.  The helpers end with the
 * library of the process that started them. */
HostCopy &g_copy = *new HostCopy;
struct HostCopyEnd {
  ~HostCopyEnd() { g_copy.stop(); }
} g_copy_end;

}  // namespace

#endif
