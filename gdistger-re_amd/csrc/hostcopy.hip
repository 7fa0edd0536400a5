// hostcopy.hip - copies from device memory to the caller's pageable host
// buffers, through pinned memory and several host threads.
//
// The C ABI's buffers are the caller's, so their pages are not pinned, and a
// large one's are often fresh: a plain hipMemcpy first touches them page by page
// in one thread (10 GB/s for 32 MB).
//   up to 64 KB   through the context's own pinned memory, one wait in all (two
//                 tables of 32 KB: 46 -> 23 us);
//   up to 4 MB    hipMemcpy (two tables of 2 MB: 299 us, 334 by the ring; of 4
//                 MB 589 and 550; a pinned chunk for less was no faster);
//   above it      the DMA engine fills a ring of pinned chunks and host threads
//                 copy from it, mapping the buffer's pages a chunk at a time
//                 (two tables of 8 MB: 2.17 -> 0.98 ms, of 32 MB: 6.7 -> 2.6 ms;
//                 3.8 ms with a fault per page).
// One ring and its threads serve the process.  Making them costs 2.6 ms, so
// they are made when the copies without them have lost about as much, and given
// back when the last context closes (made at the first copy, they took a job of
// one small batch from 0.2 to 2.9 ms).  A copy that finds the ring in use by
// another thread, or cannot get it, takes hipMemcpy.
#include <new>

#include "dg_copy_ring.h"
#include "dg_internal.h"

namespace {

constexpr size_t kRingBytes = 4u << 20;   // copies above it take the ring,
constexpr size_t kRingAfter = 32u << 20;  // made after so many bytes without it

std::mutex g_mu;              // held for the length of a copy
CopyRing* g_ring = nullptr;
bool g_failed = false;
MadeAfter g_ring_due;
std::atomic<int> g_users{0};  // open contexts

void give_back(CopyRing* r) {
  r->stop([](char* p) { (void)hipHostFree(p); });
  delete r;
}

char* pin(size_t bytes) {
  void* p = nullptr;
  if (hipHostMalloc(&p, bytes, hipHostMallocDefault) == hipSuccess) return static_cast<char*>(p);
  (void)hipGetLastError();
  return nullptr;
}

CopyRing* ring_locked(size_t bytes) {
  if (!g_ring && !g_failed && g_ring_due.due(bytes, kRingAfter)) {
    CopyRing* r = new (std::nothrow) CopyRing();
    const bool ok = r && r->start(pin);
    if (ok)
      g_ring = r;
    else if (r)
      give_back(r);
    g_failed = !ok;
  }
  return g_ring;
}

bool is_set(const uint32_t* word) { return word && __atomic_load_n(word, __ATOMIC_ACQUIRE) != 0u; }

// The stream's transfers into the ring, an event for each slot.
struct StreamEngine {
  hipStream_t stream;
  const CopyRing& ring;
  const char* src;
  const uint32_t* refused;
  hipError_t err = hipSuccess;
  hipEvent_t ev[CopyRing::kChunks] = {};

  StreamEngine(hipStream_t s, const CopyRing& r, const char* from, const uint32_t* no)
      : stream(s), ring(r), src(from), refused(no) {
    for (auto& x : ev)
      if (err == hipSuccess) err = hipEventCreateWithFlags(&x, hipEventDisableTiming);
  }
  ~StreamEngine() {
    for (auto x : ev)
      if (x) (void)hipEventDestroy(x);
  }
  bool put(size_t slot, size_t off, size_t n) {
    err = hipMemcpyAsync(ring.pinned(slot), src + off, n, hipMemcpyDeviceToHost, stream);
    if (err == hipSuccess) err = hipEventRecord(ev[slot], stream);
    return err == hipSuccess;
  }
  bool wait(size_t slot) { return (err = hipEventSynchronize(ev[slot])) == hipSuccess; }
  bool go() const { return !is_set(refused); }
  void drain() { (void)hipStreamSynchronize(stream); }
};

}  // namespace

void dg_hostcopy_open() { g_users.fetch_add(1); }

void dg_hostcopy_close() {
  if (g_users.fetch_sub(1) != 1) return;
  std::lock_guard<std::mutex> lk(g_mu);
  if (g_users.load() != 0) return;  // opened since
  if (g_ring) give_back(g_ring);
  g_ring = nullptr;
  g_failed = false;
  g_ring_due.reset();
}

int dg_copy_to_host(dg_ctx* ctx, void* dst, const void* src, size_t bytes, const uint32_t* refused) {
  if (bytes <= kStageBytes) {
    DG_HIP(ctx, hipMemcpyAsync(ctx->h_stage, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
    DG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (!is_set(refused)) memcpy(dst, ctx->h_stage, bytes);
    return DG_OK;
  }
  if (bytes > kRingBytes) {
    std::unique_lock<std::mutex> lk(g_mu, std::try_to_lock);
    if (CopyRing* r = lk.owns_lock() ? ring_locked(bytes) : nullptr) {
      StreamEngine e(ctx->stream, *r, static_cast<const char*>(src), refused);
      if (e.err == hipSuccess && r->copy(static_cast<char*>(dst), bytes, e) != CopyEnd::kFailed) return DG_OK;
      return dg_fail(ctx, DG_ERR_HIP, "copy to the host: %s", hipGetErrorString(e.err));
    }
  }
  DG_HIP(ctx, hipStreamSynchronize(ctx->stream));
  if (is_set(refused)) return DG_OK;
  DG_HIP(ctx, hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
  return DG_OK;
}
