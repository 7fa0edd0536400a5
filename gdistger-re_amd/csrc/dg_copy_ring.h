// dg_copy_ring.h - a copy through a ring of pinned chunks: a transfer engine
// fills the chunks in order, host threads copy them on to the caller's buffer.
// Knows nothing of the device (hostcopy.hip does), so it runs on the CPU alone.
#ifndef DG_COPY_RING_H
#define DG_COPY_RING_H

#include <stdint.h>
#include <string.h>
#include <sys/mman.h>

#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>

// Whether memory that makes copies faster is to be made for the next one: once
// the copies that went without it come to `after` bytes.  What it costs to make
// is about what those lost, so a program with few copies does not pay for it,
// and none pays more than twice what it would have to.
class MadeAfter {
 public:
  bool due(size_t bytes, size_t after) {
    if (without_ >= after) return true;
    without_ += bytes;
    return false;
  }
  void reset() { without_ = 0; }

 private:
  size_t without_ = 0;
};

// What became of a copy.
enum class CopyEnd {
  kDone,
  kRefused,  // go() said no: the buffer is as it was
  kFailed,   // a transfer failed: the buffer holds the chunks that came before it
};

class CopyRing {
 public:
  static constexpr size_t kChunk = 1u << 20;
  static constexpr size_t kChunks = 16;
  static constexpr int kThreads = 8;

  char* pinned(size_t slot) const { return pinned_[slot]; }

  // Chunks from alloc (char*(size_t), null: none) and the threads; false if
  // they are not to be had (stop() takes back what there is).
  template <typename Alloc>
  bool start(Alloc alloc) {
    for (char*& p : pinned_)
      if (!(p = alloc(kChunk))) return false;
    try {
      for (auto& t : threads_) t = std::thread([this] { run(); });
    } catch (...) {
      return false;
    }
    return true;
  }

  template <typename Free>
  void stop(Free free) {
    {
      std::lock_guard<std::mutex> lk(mu_);
      stop_ = true;
    }
    wake_.notify_all();
    for (auto& t : threads_)
      if (t.joinable()) t.join();
    for (char*& p : pinned_) {
      if (p) free(p);
      p = nullptr;
    }
  }

  // Copies `bytes` (at least 1) to `user`.  The engine:
  //   bool put(slot, offset, n)  queues source [offset, offset + n) into pinned(slot)
  //   bool wait(slot)            until what was last put into the slot is there
  //   bool go()                  asked when the first chunk is there
  //   void drain()               after it, nothing queued writes a chunk any more
  // Nothing but bytes of this copy's source reaches the buffer, also where a
  // transfer fails: the chunks may hold an earlier copy's.
  template <typename Engine>
  CopyEnd copy(char* user, size_t bytes, Engine& e) {
    const size_t n = (bytes + kChunk - 1) / kChunk;
    begin(user, bytes, n);
    CopyEnd end = CopyEnd::kDone;
    size_t queued = 0;
    for (size_t c = 0; c < n && end == CopyEnd::kDone; ++c) {
      bool ok = true;
      // the host threads run behind the engine, at most a ring behind it
      while (queued < n && queued < c + kChunks && ok) {
        if (queued >= kChunks) wait_for(queued - kChunks);  // its chunk is empty again
        const size_t off = queued * kChunk;
        ok = e.put(queued % kChunks, off, bytes - off < kChunk ? bytes - off : kChunk);
        if (ok) ++queued;
      }
      ok = ok && e.wait(c % kChunks);
      if (!ok)
        end = CopyEnd::kFailed;
      else if (c == 0 && !e.go())
        end = CopyEnd::kRefused;
      else
        ready_.store(c + 1, std::memory_order_release);
    }
    if (end != CopyEnd::kDone) {
      e.drain();
      given_up_.store(true, std::memory_order_release);
    }
    finish(n);
    return end;
  }

 private:
  // Maps the whole pages of [p, p + n) for writing in one call, where the kernel
  // can: a fresh page's fault costs about a microsecond here, one by one.
  static void populate(char* p, size_t n) {
    constexpr uintptr_t page = 4096;
    const uintptr_t lo = ((uintptr_t)p + page - 1) / page * page, hi = ((uintptr_t)p + n) / page * page;
#ifdef MADV_POPULATE_WRITE
    if (hi > lo) (void)madvise(reinterpret_cast<void*>(lo), hi - lo, MADV_POPULATE_WRITE);
#else
    (void)lo, (void)hi;
#endif
  }

  void help() {  // chunks of the current copy, until none is left
    while (true) {
      const size_t c = taken_.fetch_add(1, std::memory_order_relaxed);
      if (c >= n_) return;
      const size_t len = bytes_ - c * kChunk < kChunk ? bytes_ - c * kChunk : kChunk;
      populate(user_ + c * kChunk, len);
      while (ready_.load(std::memory_order_acquire) <= c && !given_up_.load(std::memory_order_acquire))
        std::this_thread::yield();
      if (ready_.load(std::memory_order_acquire) > c) memcpy(user_ + c * kChunk, pinned_[c % kChunks], len);
      done_[c % kChunks].fetch_add(1, std::memory_order_release);
      finished_.fetch_add(1, std::memory_order_release);
    }
  }

  void run() {
    std::unique_lock<std::mutex> lk(mu_);
    uint64_t seen = 0;
    while (true) {
      wake_.wait(lk, [&] { return stop_ || (open_ && job_ != seen); });
      if (stop_) return;
      seen = job_;
      working_.fetch_add(1);
      lk.unlock();
      help();
      working_.fetch_sub(1);
      lk.lock();
    }
  }

  void begin(char* user, size_t bytes, size_t n) {
    for (auto& d : done_) d.store(0, std::memory_order_relaxed);
    std::lock_guard<std::mutex> lk(mu_);
    user_ = user;
    bytes_ = bytes;
    n_ = n;
    ready_.store(0);
    taken_.store(0);
    finished_.store(0);
    given_up_.store(false);
    ++job_;
    open_ = true;
    wake_.notify_all();
  }

  void wait_for(size_t c) {
    while (done_[c % kChunks].load(std::memory_order_acquire) <= c / kChunks) std::this_thread::yield();
  }

  // Every chunk is copied or given up, and no thread looks at this copy any more.
  void finish(size_t n) {
    help();
    while (finished_.load(std::memory_order_acquire) < n) std::this_thread::yield();
    {
      std::lock_guard<std::mutex> lk(mu_);
      open_ = false;
    }
    while (working_.load() != 0) std::this_thread::yield();
  }

  char* pinned_[kChunks] = {};
  std::thread threads_[kThreads];
  std::mutex mu_;  // guards job_, open_, stop_ and the start of a copy
  std::condition_variable wake_;
  uint64_t job_ = 0;   // copies begun
  bool open_ = false;  // the current copy takes threads
  bool stop_ = false;
  // the current copy; threads spin on ready_ while it lasts
  char* user_ = nullptr;
  size_t bytes_ = 0, n_ = 0;
  std::atomic<size_t> ready_{0}, taken_{0}, finished_{0};
  std::atomic<size_t> done_[kChunks] = {};  // chunks taken out of each slot
  std::atomic<bool> given_up_{false};
  std::atomic<int> working_{0};
};

#endif  // DG_COPY_RING_H
