// Copies from a device to ordinary host memory through a ring of pinned slots, the
// host's side of it: no HIP here, so that it also builds under a thread sanitizer.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>

namespace rtnn {

// Device memory to the caller's pageable host memory.  The runtime's own copy
// moves it at 17 GB/s, one thread copying from a pinned buffer; here chunks
// travel through a ring of pinned slots (8 to 32 MiB, kept by the context), and
// threads of this call, started while the search still runs, copy each from its
// slot as it lands.  Each chunk costs the queue about 20 us, each thread copies
// about 12 GB/s.  Search and copy of 61 MB of rows: 3424 -> 1588 us (1 MiB
// chunks 2138; 6 or 8 threads no better), 410 MB: 23.5 -> 9.4 ms, 16 MB: 1044 ->
// 582 us, 8 MB: 552 -> 392, 5 MB: 395 -> 308; below 4 MB the threads' start
// costs what they win.
struct HostPiece {
  void* dst;
  const void* src;
  uint64_t bytes;
};
constexpr int kCopySlots = 8, kCopyDepth = 3, kCopyThreads = 4;
constexpr uint64_t kStagedBytes = 4ull << 20;

inline uint64_t copy_slot_bytes(uint64_t total) {
  return std::min<uint64_t>(4ull << 20,
                            std::max<uint64_t>(1ull << 20, (total / 8 + 65535) & ~65535ull));
}

// Copies npieces (at most two) through `ring`, kCopySlots slots of
// copy_slot_bytes(total).  send(slot, dst, src, bytes) starts the copy of a chunk
// into its slot, wait(slot) waits for it; both return 0, or an error that ends the
// copy and is returned.
template <class Send, class Wait>
int copy_staged(const HostPiece* piece, int npieces, uint64_t total, void* ring, Send send,
                Wait wait) {
  const uint64_t slot_bytes = copy_slot_bytes(total);
  uint64_t first[3] = {0, 0, 0};  // first chunk of each piece
  for (int i = 0; i < npieces; ++i)
    first[i + 1] = first[i] + (piece[i].bytes + slot_bytes - 1) / slot_bytes;
  const uint64_t chunks = first[npieces];
  char* const slots = static_cast<char*>(ring);
  auto chunk = [&](uint64_t j) {
    const int i = npieces > 1 && j >= first[1] ? 1 : 0;
    const uint64_t off = (j - first[i]) * slot_bytes;
    return HostPiece{static_cast<char*>(piece[i].dst) + off,
                     static_cast<const char*>(piece[i].src) + off,
                     std::min(slot_bytes, piece[i].bytes - off)};
  };
  auto unload = [&](uint64_t j) {
    const HostPiece c = chunk(j);
    std::memcpy(c.dst, slots + (j % kCopySlots) * slot_bytes, c.bytes);
  };
  // Chunk j is thread (j mod threads)'s, in order: it waits until `landed`
  // passes j.  A slot is free again once its chunk's thread has passed it.
  std::atomic<uint64_t> landed{0};
  std::atomic<uint64_t> passed[kCopyThreads];  // chunks each thread has copied
  for (auto& x : passed) x.store(0);
  std::atomic<bool> stop{false};
  int nth = 0;
  std::thread th[kCopyThreads];
  auto work = [&](int w, int of) {
    for (uint64_t j = (uint64_t)w; j < chunks; j += (uint64_t)of) {
      while (landed.load(std::memory_order_acquire) <= j) {
        if (stop.load(std::memory_order_relaxed)) return;
        std::this_thread::yield();
      }
      unload(j);
      passed[w].fetch_add(1, std::memory_order_release);
    }
  };
  // The threads sleep until the first chunk has landed (the search may take
  // long), then poll.  of: how many of them there are.
  std::mutex mu;
  std::condition_variable cv;
  bool go = false;
  int of = 1;
  auto start = [&](int w) {
    {
      std::unique_lock<std::mutex> lk(mu);
      cv.wait(lk, [&] { return go; });
    }
    work(w, of);
  };
  auto release = [&] {
    std::lock_guard<std::mutex> lk(mu);
    if (go) return;  // the threads read `of` from here on
    of = nth > 0 ? nth : 1;
    go = true;
    cv.notify_all();
  };
  try {
    for (; nth < kCopyThreads; ++nth) th[nth] = std::thread(start, nth);
  } catch (...) {  // as many as there are; none: this thread copies
  }
  int e = 0;
  uint64_t sent = 0;
  for (uint64_t j = 0; j < chunks && e == 0; ++j) {
    for (; sent < chunks && sent < j + kCopyDepth && e == 0; ++sent) {
      if (sent >= kCopySlots && nth > 0) {  // the slot's last chunk: o
        const uint64_t o = sent - kCopySlots;
        while (passed[o % nth].load(std::memory_order_acquire) <= o / nth) std::this_thread::yield();
      }
      const HostPiece c = chunk(sent);
      const int slot = (int)(sent % kCopySlots);
      e = send(slot, slots + (uint64_t)slot * slot_bytes, c.src, c.bytes);
    }
    if (e == 0) e = wait((int)(j % kCopySlots));
    if (e != 0) break;
    if (nth == 0) unload(j);
    landed.store(j + 1, std::memory_order_release);
    if (j == 0) release();
  }
  if (e != 0) stop.store(true);
  release();
  for (int w = 0; w < nth; ++w) th[w].join();
  return e;
}

}  // namespace rtnn
