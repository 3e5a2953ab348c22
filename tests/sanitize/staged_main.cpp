// The ring of host copies (rtnn_amd/csrc/staged.h) without a device: chunks arrive
// by memcpy, some of them late; every byte must arrive, and an error must end the
// copy with all threads joined.  Built with -fsanitize=thread.
#include <chrono>
#include <cstdio>
#include <vector>

#include "../../rtnn_amd/csrc/staged.h"

namespace {

__attribute__((no_sanitize("thread"))) void fill(std::vector<char>& v, int seed) {
  for (size_t j = 0; j < v.size(); ++j) v[j] = (char)(j * 31 + (j >> 12) + seed);
}

// Copies two pieces of `bytes` (or one); fail_at: the send that fails (-1: none).
// `late` sends (and waits) take a while.  Returns the pieces that differ, or -1
// where the error was not reported.
long run(uint64_t bytes, int npieces, int fail_at, bool late, bool fail_wait) {
  const uint64_t total = bytes * (uint64_t)npieces;
  std::vector<char> src[2], dst[2], ring(rtnn::kCopySlots * rtnn::copy_slot_bytes(total));
  rtnn::HostPiece piece[2];
  for (int i = 0; i < npieces; ++i) {
    src[i].resize(bytes);
    fill(src[i], i + 1);
    dst[i].assign(bytes, 0);
    piece[i] = {dst[i].data(), src[i].data(), bytes};
  }
  int sends = 0, waits = 0;
  const int e = rtnn::copy_staged(
      piece, npieces, total, ring.data(),
      [&](int, void* to, const void* from, uint64_t n) {
        if (!fail_wait && sends++ == fail_at) return 7;
        std::memcpy(to, from, n);
        return 0;
      },
      [&](int) {
        if (late && waits % 3 == 0) std::this_thread::sleep_for(std::chrono::milliseconds(2));
        return fail_wait && waits++ == fail_at ? 7 : 0;
      });
  if (fail_at >= 0) return e == 7 ? 0 : -1;
  if (e != 0) return -1;
  long bad = 0;  // pieces
  for (int i = 0; i < npieces; ++i) bad += std::memcmp(dst[i].data(), src[i].data(), bytes) != 0;
  return bad;
}

}  // namespace

int main() {
  const uint64_t mb = 1ull << 20;
  for (uint64_t bytes : {(uint64_t)1000, mb, 9 * mb + 4})
    for (int np : {1, 2})
      for (bool late : {false, true})
        if (const long bad = run(bytes, np, -1, late, false)) {
          std::printf("%llu bytes, %d pieces: %ld wrong\n", (unsigned long long)bytes, np, bad);
          return 1;
        }
  for (int at : {0, 1, 5, 7})
    for (bool wait : {false, true})
      if (run(5 * mb, 2, at, true, wait) != 0) {
        std::printf("error at %d not reported\n", at);
        return 1;
      }
  std::printf("staged copies passed\n");
  return 0;
}
