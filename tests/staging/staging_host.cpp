// Host build of the staged download (parafrost_amd/csrc/pfs_staging.hpp) for
// the CPU tests.  TEST INFRASTRUCTURE ONLY.
//
// A ring in ordinary memory whose copies run in a thread of its own, in order
// and late, as a stream's do; threads that cannot be started, copies that
// cannot be queued and waits that fail are forced by counters.
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <deque>
#include <mutex>
#include <random>
#include <system_error>

#include "../../parafrost_amd/csrc/pfs_staging.hpp"

using namespace pfs;
constexpr size_t SLOT = 4096;

struct Ring {
  uint32_t slots;
  std::vector<std::vector<unsigned char>> mem;
  std::vector<uint32_t> queued, ran;  // copies per slot
  std::deque<std::pair<uint32_t, StagedPiece>> q;
  std::mutex m;
  std::condition_variable cv;
  bool stop = false;
  int threads_left = 1 << 30, copies_left = 1 << 30, waits_left = 1 << 30;
  uint32_t started = 0, copies = 0;
  std::thread stream;

  explicit Ring(uint32_t n) : slots(n), mem(n, std::vector<unsigned char>(SLOT)), queued(n, 0), ran(n, 0) {
    stream = std::thread([this] {
      std::unique_lock<std::mutex> lk(m);
      while (true) {
        cv.wait(lk, [this] { return stop || !q.empty(); });
        if (q.empty()) return;
        const auto c = q.front();
        q.pop_front();
        memcpy(mem[c.first].data(), c.second.src, c.second.bytes);
        ran[c.first]++;
        cv.notify_all();
      }
    });
  }
  ~Ring() {
    {
      std::lock_guard<std::mutex> lk(m);
      stop = true;
    }
    cv.notify_all();
    stream.join();
  }
  const unsigned char* slot(uint32_t k) { return mem[k].data(); }
  bool queue(uint32_t k, const StagedPiece& p) {
    std::lock_guard<std::mutex> lk(m);
    if (copies_left-- <= 0) return false;
    copies++;
    queued[k]++;
    q.emplace_back(k, p);
    cv.notify_all();
    return true;
  }
  bool arrived(uint32_t k) {
    std::unique_lock<std::mutex> lk(m);
    if (waits_left-- <= 0) return false;
    const uint32_t n = queued[k];
    cv.wait(lk, [&] { return ran[k] >= n; });
    return true;
  }
  template <class F>
  std::thread run(F f) {
    if (threads_left-- <= 0) throw std::system_error(std::make_error_code(std::errc::resource_unavailable_try_again));
    started++;
    return std::thread(f);
  }
};

int main(int argc, char** argv) {
  std::mt19937 rng(1);
  const int trials = argc > 1 ? atoi(argv[1]) : 100;
  int done = 0, refused = 0, failed = 0;
  for (int t = 0; t < trials; t++) {
    const uint32_t np = 1 + rng() % 20, nthr = 1 + rng() % 5;
    std::vector<std::vector<char>> src(np), dst(np);
    std::vector<StagedPiece> pc;
    for (uint32_t i = 0; i < np; i++) {
      const size_t n = rng() % 3 ? SLOT : 1 + rng() % SLOT;
      src[i].resize(n), dst[i].assign(n, 0);
      for (char& c : src[i]) c = (char)(1 + rng() % 255);
      pc.push_back(StagedPiece{dst[i].data(), src[i].data(), n});
    }
    Ring ring(1 + rng() % 4);
    const int kind = t % 4;
    if (kind == 1) ring.threads_left = (int)(rng() % nthr);
    if (kind == 2) ring.copies_left = (int)(rng() % np);
    if (kind == 3) ring.waits_left = (int)(rng() % (np * nthr));
    Staged r;
    try {
      r = staged_copy(pc, nthr, ring);
    } catch (std::exception& e) {
      return fprintf(stderr, "trial %d: %s\n", t, e.what()), 1;
    }
    const Staged want = kind == 0 ? Staged::DONE : kind == 1 ? Staged::NOT_STARTED : Staged::FAILED;
    if (r != want) return fprintf(stderr, "trial %d kind %d: %d\n", t, kind, (int)r), 1;
    if (r == Staged::NOT_STARTED) {
      for (const auto& d : dst)
        for (char c : d)
          if (c) return fprintf(stderr, "trial %d: written\n", t), 1;
      if (ring.copies) return fprintf(stderr, "trial %d: queued\n", t), 1;
      refused++;
    } else if (r == Staged::DONE) {
      if (src != dst) return fprintf(stderr, "trial %d: bytes differ\n", t), 1;
      done++;
    } else {
      failed++;
    }
  }
  printf("{\"done\": %d, \"not_started\": %d, \"failed\": %d}\n", done, refused, failed);
  return 0;
}
