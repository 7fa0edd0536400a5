// Copies through CopyRing with a transfer engine of plain memcpy that fails or
// refuses where it is told to.  Prints one line per case; exits 1 on a wrong one.
#include "dg_copy_ring.h"

#include <stdio.h>
#include <stdlib.h>

#include <vector>

namespace {

struct Engine {
  CopyRing& ring;
  const std::vector<char>& src;
  size_t fail_put, fail_wait;  // chunk whose put or wait fails
  bool accept;
  size_t puts = 0, waits = 0;

  bool put(size_t slot, size_t off, size_t n) {
    if (puts++ == fail_put) return false;
    memcpy(ring.pinned(slot), src.data() + off, n);
    return true;
  }
  bool wait(size_t) { return waits++ != fail_wait; }
  bool go() const { return accept; }
  void drain() {}
};

constexpr size_t kNever = ~(size_t)0, C = CopyRing::kChunk;
constexpr char kOld = 0x55;

// Chunks of the buffer that hold the source, from the front; -1 if any byte is
// neither the source's nor the buffer's own.
long copied(const std::vector<char>& buf, const std::vector<char>& src) {
  const size_t bytes = src.size();
  long n = 0;
  bool more = true;
  for (size_t o = 0; o < bytes; o += C) {
    const size_t len = bytes - o < C ? bytes - o : C;
    if (memcmp(buf.data() + o, src.data() + o, len) == 0) {
      if (!more) return -1;
      ++n;
      continue;
    }
    more = false;
    for (size_t i = 0; i < len; ++i)
      if (buf[o + i] != kOld) return -1;
  }
  return n;
}

}  // namespace

int main() {
  CopyRing ring;
  if (!ring.start([](size_t n) { return (char*)malloc(n); })) return 2;
  int bad = 0;
  auto check = [&](const char* what, size_t bytes, size_t fail_put, size_t fail_wait, bool accept, CopyEnd end,
                   long lo, long hi) {
    static unsigned seed = 1;
    std::vector<char> src(bytes), buf(bytes + 64, kOld);
    for (auto& x : src) x = (char)((seed = seed * 1664525u + 1013904223u) >> 24 | 0x80);  // never kOld
    Engine e{ring, src, fail_put, fail_wait, accept};
    const CopyEnd got = ring.copy(buf.data(), bytes, e);
    const long n = copied(buf, src);
    bool past = false;
    for (size_t i = bytes; i < buf.size(); ++i) past |= buf[i] != kOld;
    const bool ok = got == end && n >= lo && n <= hi && !past;
    printf("%s %s: %zu bytes, ended %d, %ld chunks\n", ok ? "ok" : "WRONG", what, bytes, (int)got, n);
    fflush(stdout);
    bad += !ok;
  };
  // what the ring holds between the cases is an earlier copy's
  for (size_t bytes : {(size_t)1, C - 1, C, C + 1, 5 * C + 17, 16 * C, 16 * C + 1, 50 * C + 12345})
    check("whole", bytes, kNever, kNever, true, CopyEnd::kDone, (long)((bytes + C - 1) / C), (long)((bytes + C - 1) / C));
  check("first put fails", 40 * C, 0, kNever, true, CopyEnd::kFailed, 0, 0);
  check("a put of the first ring fails", 40 * C, 7, kNever, true, CopyEnd::kFailed, 0, 0);
  check("a later put fails", 40 * C, 20, kNever, true, CopyEnd::kFailed, 0, 20);
  check("first wait fails", 40 * C, kNever, 0, true, CopyEnd::kFailed, 0, 0);
  check("a later wait fails", 40 * C + 3, kNever, 23, true, CopyEnd::kFailed, 0, 23);
  check("last wait fails", 18 * C + 3, kNever, 18, true, CopyEnd::kFailed, 0, 18);
  check("refused", 40 * C, kNever, kNever, false, CopyEnd::kRefused, 0, 0);
  check("refused, one chunk", 100, kNever, kNever, false, CopyEnd::kRefused, 0, 0);
  check("whole again", 33 * C + 5, kNever, kNever, true, CopyEnd::kDone, 34, 34);
  ring.stop([](char* p) { free(p); });
  // memory for faster copies: not for a few small ones, and after so many bytes without it
  MadeAfter made;
  int without = 0;
  while (!made.due(100, 1000)) ++without;
  bool late = made.due(1, 1000);
  made.reset();
  const bool again = made.due(5000, 1000), then = made.due(1, 1000);
  const bool ok = without == 10 && late && !again && then;
  printf("%s made after 10 of 100 bytes, at once later, anew after the last user\n", ok ? "ok" : "WRONG");
  return bad || !ok ? 1 : 0;
}
