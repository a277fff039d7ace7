// Host build of the passes that append a batch of clauses on the device
// (append_pass and append_write, parafrost_amd/csrc/pfs_items.hpp) for the CPU
// tests.  TEST INFRASTRUCTURE ONLY.
//
// Random batches over few or many variables, with units, empty clauses, tautologies,
// duplicates, root assignments, and in half of them one clause that the device
// has to refuse (a literal out of range alone or among others, an over-long
// clause, decreasing offsets) at the start, in the middle or at the end.  The
// passes run as the driver queues them, eight before a look at the flags, the
// clauses of a pass in random order, on arrays of exactly the sizes that the
// driver allocates, so that the sanitizers see every access.  A batch is
// refused exactly where it holds such a clause; any other one leaves the
// clauses, units and status of a sequential loop.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <memory>
#include <random>
#include <vector>

#include "../../parafrost_amd/csrc/pfs_items.hpp"

using namespace pfs;

static std::mt19937_64 g_rng;
static u32 below(u32 n) { return (u32)(g_rng() % n); }

template <class T>
static std::unique_ptr<T[]> heap(size_t n, T v) {
  std::unique_ptr<T[]> p(new T[n]);
  std::fill(p.get(), p.get() + n, v);
  return p;
}

struct Counts {
  unsigned refused = 0, taken = 0, units = 0, refuted = 0, kept = 0;
};

static bool trial(Counts& cnt) {
  const u32 nvars = 1 + below(below(2) ? 40 : 900), n = 1 + below(60);
  std::vector<std::vector<u32>> cls(n);
  const u32 kind = below(10);  // 0-4: refused
  const u32 at = below(3) == 0 ? 0 : below(2) ? n - 1 : n / 2;
  for (auto& c : cls) {
    const u32 k = below(8) == 0 ? below(2) : 1 + below(5);
    for (u32 q = 0; q < k; q++) c.push_back(2 * (1 + below(nvars)) + below(2));
  }
  static const u32 BAD[] = {0, 1, 0xFFFFFFFFu, 0xFFFFFFFEu, 0x80000000u};
  const u32 bad = below(2) ? BAD[below(5)] : 2 * (nvars + 1 + below(1000000)) + below(2);
  bool refuse = false;
  if (kind < 3) {
    if (kind == 0) cls[at].clear();  // alone in its clause
    cls[at].insert(cls[at].begin() + below((u32)cls[at].size() + 1), bad);
    refuse = true;
  } else if (kind == 3) {
    while (cls[at].size() <= AP_LONG) cls[at].push_back(2 * (1 + below(nvars)) + below(2));
    refuse = true;
  }
  std::vector<u64> off(1, below(3));  // a batch may start inside the caller's arrays
  std::vector<u32> lits;
  for (const auto& c : cls) {
    lits.insert(lits.end(), c.begin(), c.end());
    off.push_back(off.back() + c.size());
  }
  if (kind == 4 && n > 1) {
    const u32 q = 1 + below(n - 1);
    off[q] = below(2) ? ~0ull - below(9) : off[n] + 1 + below(5);
    refuse = true;
  }
  const u32 nl = (u32)lits.size();
  auto o = heap<u64>(n + 1, 0);
  std::copy(off.begin(), off.end(), o.get());
  auto l = heap<u32>(nl, 0);
  std::copy(lits.begin(), lits.end(), l.get());
  auto assign = heap<u32>(nvars + 1, 0);
  for (u32 v = 1; v <= nvars; v++)
    if (below(12) == 0) assign[v] = 2 * v + below(2) + 1;
  auto s0 = heap<u64>(nvars + 1, ~0ull), s1 = heap<u64>(nvars + 1, ~0ull), units = heap<u64>(n, 0);
  auto res = heap<u32>(n, 0xABABABABu), kept = heap<u32>(n, 0), words = heap<u32>(n, 0), fl = heap<u32>(AP_FLAGS, 0);
  auto pool = heap<u32>(nl + CL_HDR * n, 0), c_off = heap<u32>(n, 0);
  DB db{};
  db.lits = pool.get();
  db.c_off = c_off.get();
  db.assign = assign.get();
  db.nvars = nvars;
  AppendArgs a{};
  a.off = o.get(), a.lits = l.get(), a.n = n, a.nl = nl;
  a.seen[0] = s0.get(), a.seen[1] = s1.get();
  a.res = res.get(), a.kept = kept.get(), a.words = words.get(), a.fl = fl.get(), a.units = units.get();

  std::vector<u32> order(n);
  for (u32 i = 0; i < n; i++) order[i] = i;
  u32 done = 0, last = AP_PASSES;
  while (last == AP_PASSES && done < AP_PASSES) {
    for (const u32 to = done + 8; done < to; done++) {
      if (!append_runs(a, done)) continue;  // the whole launch, as the flags are an earlier launch's
      std::shuffle(order.begin(), order.end(), g_rng);
      bool any = false;
      for (u32 i : order) any |= append_pass(db, a, i, done);
      if (any) fl[AP_CHANGED + done] = 1;
    }
    if (fl[0]) break;
    for (u32 p = 0; p < done && last == AP_PASSES; p++)
      if (!fl[AP_CHANGED + p]) last = p;
  }
  if ((fl[0] != 0) != refuse) return fprintf(stderr, "kind %u refused %u\n", kind, fl[0]), false;
  if (refuse) return cnt.refused++, true;
  if (last == AP_PASSES) return true;  // a long chain of units is the host's
  u32 nk = 0, nw = 0;
  for (u32 i = 0; i < n; i++) {
    const u32 k = kept[i], w = words[i];
    kept[i] = nk, words[i] = nw;
    nk += k, nw += w;
  }
  fl[4] = nk, fl[5] = nw;
  for (u32 i : order) append_write(db, a, i, last, 0, 0);
  std::sort(units.get(), units.get() + fl[2]);

  // the sequential loop
  std::vector<u64> want_units;
  std::vector<std::vector<u32>> want;
  bool refuted = false;
  for (u32 i = 0; i < n; i++) {
    std::vector<u32> c;
    bool sat = false;
    for (u32 x : cls[i]) {
      if (const u32 t = assign[ABS(x)]) {
        sat |= t - 1 == x;
        continue;
      }
      sat |= std::count(c.begin(), c.end(), FLIP(x)) != 0;
      if (!std::count(c.begin(), c.end(), x)) c.push_back(x);
    }
    if (sat) continue;
    if (c.empty()) {
      refuted = true;
    } else if (c.size() == 1) {
      assign[ABS(c[0])] = c[0] + 1;
      want_units.push_back((u64)i << 32 | c[0]);
    } else {
      std::sort(c.begin(), c.end());
      want.push_back(c);
    }
  }
  bool ok = nk == want.size() && fl[2] == want_units.size() && (fl[1] != 0) == refuted;
  ok = ok && std::equal(want_units.begin(), want_units.end(), units.get());
  for (u32 k = 0; ok && k < nk; k++) {
    const u32* h = pool.get() + c_off[k];
    ok = hdr_size(h[0]) == want[k].size() && std::equal(want[k].begin(), want[k].end(), h + CL_HDR) &&
         h[1] == calc_sig(h + CL_HDR, hdr_size(h[0]));
  }
  cnt.taken++, cnt.units += fl[2], cnt.refuted += refuted, cnt.kept += nk;
  return ok;
}

int main(int argc, char** argv) {
  const unsigned seeds = argc > 1 ? (unsigned)atoi(argv[1]) : 1, trials = argc > 2 ? (unsigned)atoi(argv[2]) : 100;
  Counts c;
  for (unsigned s = 0; s < seeds; s++) {
    g_rng.seed(s + 1);
    for (unsigned t = 0; t < trials; t++)
      if (!trial(c)) return fprintf(stderr, "seed %u trial %u\n", s + 1, t), 1;
  }
  printf("{\"refused\": %u, \"taken\": %u, \"units\": %u, \"refuted\": %u, \"kept\": %u}\n", c.refused, c.taken, c.units,
         c.refuted, c.kept);
  return 0;
}
