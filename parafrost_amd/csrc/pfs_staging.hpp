// Moves a large download through a ring of slots: the calling thread keeps
// the copies into the slots going, threads that live as long as the call move
// their share of every slot that has arrived to the caller's memory.  Host
// code without device calls: the ring and its copies are the caller's R.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <thread>
#include <vector>

namespace pfs {

struct StagedPiece {  // at most a slot
  char* dst;
  const char* src;
  size_t bytes;
};
enum class Staged { DONE, NOT_STARTED, FAILED };

// R: slots, their number; slot(k), the memory of one; queue(k, piece), starts
// its copy there and returns whether that went well; arrived(k), waits for the
// copy queued last into a slot, from any thread; run(f), a thread that runs f
// (may throw).  Piece i sits in slot i % slots.  NOT_STARTED: nothing was
// queued or written.  FAILED: copies may still be running into the slots.
template <class R>
Staged staged_copy(const std::vector<StagedPiece>& pc, uint32_t nthr, R& ring) {
  const uint32_t np = (uint32_t)pc.size(), slots = ring.slots;
  std::vector<std::atomic<uint32_t>> done(np);  // threads that have moved their share of a piece
  for (auto& d : done) d.store(0, std::memory_order_relaxed);
  std::atomic<uint32_t> queued{0};
  std::atomic<bool> failed{false};
  auto mover = [&](uint32_t t) {
    for (uint32_t i = 0; i < np; i++) {
      while (queued.load(std::memory_order_acquire) <= i) {
        if (failed.load(std::memory_order_relaxed)) return;
        std::this_thread::yield();
      }
      if (!ring.arrived(i % slots)) {
        failed.store(true);
        return;
      }
      const size_t n = pc[i].bytes, share = (n / nthr + 63) & ~(size_t)63;
      const size_t a = std::min(n, t * share), b = t + 1 == nthr ? n : std::min(n, a + share);
      memcpy(pc[i].dst + a, ring.slot(i % slots) + a, b - a);
      done[i].fetch_add(1, std::memory_order_release);
    }
  };
  std::vector<std::thread> thr;
  try {
    thr.reserve(nthr);
    for (uint32_t t = 0; t < nthr; t++) thr.push_back(ring.run([&mover, t] { mover(t); }));
  } catch (...) {  // no thread to be had: the ones that were started return
    failed.store(true);
    for (std::thread& t : thr) t.join();
    return Staged::NOT_STARTED;
  }
  for (uint32_t i = 0; i < np; i++) {
    // the slot is free once every thread has moved its piece before
    while (i >= slots && done[i - slots].load(std::memory_order_acquire) < nthr &&
           !failed.load(std::memory_order_relaxed))
      std::this_thread::yield();
    if (failed.load(std::memory_order_relaxed)) break;  // a thread may still read the slot
    if (ring.queue(i % slots, pc[i])) queued.store(i + 1, std::memory_order_release);
    else failed.store(true);
  }
  for (std::thread& t : thr) t.join();
  return failed.load() ? Staged::FAILED : Staged::DONE;
}

}  // namespace pfs
