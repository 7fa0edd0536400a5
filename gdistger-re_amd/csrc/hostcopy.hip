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
// milliseconds: made at the first such copy, bounded, given back when the last
// context closes.  A copy that finds the ring in use by another thread, or
// cannot get it, takes hipMemcpy.
#include <new>

#include "dg_copy_ring.h"
#include "dg_internal.h"

namespace {

constexpr size_t kMinBytes = 1u << 10;

std::mutex g_mu;              // held for the length of a copy
CopyRing* g_ring = nullptr;
bool g_failed = false;
std::atomic<int> g_users{0};  // open contexts

void give_back(CopyRing* r) {
  r->stop([](char* p) { (void)hipHostFree(p); });
  delete r;
}

CopyRing* ring_locked() {
  if (!g_ring && !g_failed) {
    CopyRing* r = new (std::nothrow) CopyRing();
    const bool ok = r && r->start([](size_t bytes) {
      void* p = nullptr;
      if (hipHostMalloc(&p, bytes, hipHostMallocDefault) == hipSuccess) return static_cast<char*>(p);
      (void)hipGetLastError();
      return static_cast<char*>(nullptr);
    });
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
}

int dg_copy_to_host(dg_ctx* ctx, void* dst, const void* src, size_t bytes, const uint32_t* refused) {
  if (bytes >= kMinBytes) {
    std::unique_lock<std::mutex> lk(g_mu, std::try_to_lock);
    if (CopyRing* r = lk.owns_lock() ? ring_locked() : nullptr) {
      if (bytes > CopyRing::kChunk) {
        StreamEngine e(ctx->stream, *r, static_cast<const char*>(src), refused);
        if (e.err == hipSuccess && r->copy(static_cast<char*>(dst), bytes, e) != CopyEnd::kFailed) return DG_OK;
        return dg_fail(ctx, DG_ERR_HIP, "copy to the host: %s", hipGetErrorString(e.err));
      }
      DG_HIP(ctx, hipMemcpyAsync(r->pinned(0), src, bytes, hipMemcpyDeviceToHost, ctx->stream));
      DG_HIP(ctx, hipStreamSynchronize(ctx->stream));
      if (!is_set(refused)) memcpy(dst, r->pinned(0), bytes);
      return DG_OK;
    }
  }
  if (refused) {
    DG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (is_set(refused)) return DG_OK;
  }
  DG_HIP(ctx, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
  DG_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return DG_OK;
}
