// hostcopy.hip - copies from device memory to the caller's pageable host
// buffers, through pinned memory and several host threads.
//
// The C ABI's buffers are the caller's, so their pages are not pinned, and a
// large one's are often fresh: a plain hipMemcpy pins them (0.12 ms for 256
// KB) or first touches them page by page in one thread (10 GB/s for 32 MB).
// A copy of at most a chunk goes through a pinned chunk, copied on by the
// caller's thread (256 KB: 119 -> 23 us).  For a larger one the DMA engine
// fills a ring of pinned chunks and host threads copy from it, mapping the
// buffer's pages a chunk at a time (two buffers of 32 MB: 6.7 -> 2.6 ms; 3.8 ms
// with a fault per page).
//
// One ring and its threads serve the process, since pinning it costs
// milliseconds: made at the first such copy, bounded (kChunks chunks,
// kThreads threads), given back when the last context closes.  A copy that
// finds the ring in use by another thread, or cannot get it, takes hipMemcpy.
#include <sys/mman.h>

#include <atomic>
#include <condition_variable>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "dg_internal.h"

namespace {

constexpr size_t kChunk = 1u << 20;
constexpr size_t kChunks = 16;
constexpr int kThreads = 8;
constexpr size_t kMinBytes = 1u << 10;

// Maps the whole pages of [p, p + n) for writing in one call, where the kernel
// can: a fresh page's fault costs about a microsecond here, one by one.
void populate(char* p, size_t n) {
  constexpr uintptr_t page = 4096;
  const uintptr_t lo = ((uintptr_t)p + page - 1) / page * page, hi = ((uintptr_t)p + n) / page * page;
#ifdef MADV_POPULATE_WRITE
  if (hi > lo) (void)madvise(reinterpret_cast<void*>(lo), hi - lo, MADV_POPULATE_WRITE);
#else
  (void)lo, (void)hi;
#endif
}

struct Ring {
  std::vector<char*> pinned;
  std::vector<std::thread> threads;
  std::mutex mu;  // guards the fields down to `stop`
  std::condition_variable wake;
  uint64_t job = 0;     // copies begun
  bool open = false;    // the current copy takes threads
  bool stop = false;
  // the current copy; threads spin on `ready` while it lasts
  char* user = nullptr;
  size_t bytes = 0, n = 0;
  std::atomic<size_t> ready{0}, taken{0};
  std::atomic<int> working{0};
  std::unique_ptr<std::atomic<char>[]> finished;

  void help() {  // chunks of the current copy, until none is left
    while (true) {
      const size_t c = taken.fetch_add(1, std::memory_order_relaxed);
      if (c >= n) return;
      const size_t len = bytes - c * kChunk < kChunk ? bytes - c * kChunk : kChunk;
      populate(user + c * kChunk, len);
      while (ready.load(std::memory_order_acquire) <= c) std::this_thread::yield();
      memcpy(user + c * kChunk, pinned[c % kChunks], len);
      finished[c].store(1, std::memory_order_release);
    }
  }

  void run() {
    std::unique_lock<std::mutex> lk(mu);
    uint64_t seen = 0;
    while (true) {
      wake.wait(lk, [&] { return stop || (open && job != seen); });
      if (stop) return;
      seen = job;
      working.fetch_add(1);
      lk.unlock();
      help();
      working.fetch_sub(1);
      lk.lock();
    }
  }

  bool start() {
    for (size_t i = 0; i < kChunks; ++i) {
      void* p = nullptr;
      if (hipHostMalloc(&p, kChunk, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        return false;
      }
      pinned.push_back(static_cast<char*>(p));
    }
    try {
      for (int i = 0; i < kThreads; ++i) threads.emplace_back([this] { run(); });
    } catch (...) {  // no threads to be had
      return false;
    }
    return true;
  }

  ~Ring() {
    {
      std::lock_guard<std::mutex> lk(mu);
      stop = true;
    }
    wake.notify_all();
    for (auto& t : threads) t.join();
    for (char* p : pinned) hipHostFree(p);
  }

  void begin(char* u, size_t size) {
    const size_t count = (size + kChunk - 1) / kChunk;
    finished.reset(new std::atomic<char>[count]);
    for (size_t c = 0; c < count; ++c) finished[c].store(0, std::memory_order_relaxed);
    std::lock_guard<std::mutex> lk(mu);
    user = u;
    bytes = size;
    n = count;
    ready.store(0);
    taken.store(0);
    ++job;
    open = true;
    wake.notify_all();
  }
  void wait_for(size_t c) {
    while (!finished[c].load(std::memory_order_acquire)) std::this_thread::yield();
  }
  // Every chunk is copied and no thread looks at this copy any more.
  void end() {
    ready.store(n, std::memory_order_release);
    help();
    for (size_t c = 0; c < n; ++c) wait_for(c);
    {
      std::lock_guard<std::mutex> lk(mu);
      open = false;
    }
    while (working.load() != 0) std::this_thread::yield();
  }
};

std::mutex g_mu;          // held for the length of a copy
Ring* g_ring = nullptr;
bool g_failed = false;
int g_users = 0;          // open contexts

Ring* ring_locked() {
  if (!g_ring && !g_failed) {
    Ring* r = new Ring();
    if (r->start()) {
      g_ring = r;
    } else {
      delete r;
      g_failed = true;
    }
  }
  return g_ring;
}

// The host threads run behind the DMA engine, at most a ring behind it.
int copy_by_ring(dg_ctx* ctx, Ring& r, char* dst, const char* src, size_t bytes) {
  hipEvent_t ev[kChunks] = {};
  hipError_t e = hipSuccess;
  for (auto& x : ev)
    if (e == hipSuccess) e = hipEventCreateWithFlags(&x, hipEventDisableTiming);
  const size_t n = (bytes + kChunk - 1) / kChunk;
  r.begin(dst, bytes);
  size_t queued = 0;
  for (size_t c = 0; c < n && e == hipSuccess; ++c) {
    while (queued < n && queued < c + kChunks && e == hipSuccess) {
      if (queued >= kChunks) r.wait_for(queued - kChunks);  // its pinned chunk is empty again
      const size_t off = queued * kChunk, len = bytes - off < kChunk ? bytes - off : kChunk;
      e = hipMemcpyAsync(r.pinned[queued % kChunks], src + off, len, hipMemcpyDeviceToHost, ctx->stream);
      if (e == hipSuccess) e = hipEventRecord(ev[queued % kChunks], ctx->stream);
      if (e == hipSuccess) ++queued;
    }
    if (e == hipSuccess) e = hipEventSynchronize(ev[c % kChunks]);
    if (e == hipSuccess) r.ready.store(c + 1, std::memory_order_release);
  }
  if (e != hipSuccess) hipStreamSynchronize(ctx->stream);  // nothing may write the ring after this call
  r.end();  // after an error the rest of the buffer gets what the ring holds; the call fails
  for (auto x : ev)
    if (x) hipEventDestroy(x);
  if (e != hipSuccess) return dg_fail(ctx, DG_ERR_HIP, "copy to the host: %s", hipGetErrorString(e));
  return DG_OK;
}

}  // namespace

void dg_hostcopy_open() {
  std::lock_guard<std::mutex> lk(g_mu);
  ++g_users;
}

void dg_hostcopy_close() {
  std::lock_guard<std::mutex> lk(g_mu);
  if (--g_users == 0) {
    delete g_ring;
    g_ring = nullptr;
    g_failed = false;
  }
}

int dg_copy_to_host(dg_ctx* ctx, void* dst, const void* src, size_t bytes) {
  if (bytes >= kMinBytes) {
    std::unique_lock<std::mutex> lk(g_mu, std::try_to_lock);
    if (Ring* r = lk.owns_lock() ? ring_locked() : nullptr) {
      if (bytes > kChunk) return copy_by_ring(ctx, *r, static_cast<char*>(dst), static_cast<const char*>(src), bytes);
      DG_HIP(ctx, hipMemcpyAsync(r->pinned[0], src, bytes, hipMemcpyDeviceToHost, ctx->stream));
      DG_HIP(ctx, hipStreamSynchronize(ctx->stream));
      memcpy(dst, r->pinned[0], bytes);
      return DG_OK;
    }
  }
  DG_HIP(ctx, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
  DG_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return DG_OK;
}
