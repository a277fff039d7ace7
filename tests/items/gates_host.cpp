// Host build of the equivalence and AND/OR gate searches
// (parafrost_amd/csrc/pfs_items.hpp) for the CPU tests.  TEST INFRASTRUCTURE
// ONLY.
//
// Random clause lists of one variable, of few other variables so that gates
// are frequent, with repeated binary clauses, learnt ones and clauses that
// hold a literal twice, against the definitions written out: an equivalence is
// the only original binary clause of x with its converse in the list of -x; an
// AND/OR gate of dx is the literals that its original binary clauses imply,
// with -dx, as one multiset the literals of an original clause of -dx, if
// substituting it adds no more clauses than it takes away.  Exactly a gate's
// clauses are molten afterwards.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <set>
#include <vector>

#include "../../parafrost_amd/csrc/pfs_items.hpp"

using namespace pfs;

static std::mt19937_64 g_rng;
static u32 below(u32 n) { return (u32)(g_rng() % n); }

struct Lists {
  std::vector<u32> pool = {0}, refs;
  u32 off[5] = {0}, size[4] = {0};
  u32 add(std::vector<u32> l, bool learnt) {
    std::sort(l.begin(), l.end());
    const u32 c = (u32)pool.size();
    pool.push_back(make_hdr((u32)l.size(), learnt ? ST_LEARNT : ST_ORIGINAL));
    pool.push_back(calc_sig(l.data(), (u32)l.size()));
    pool.push_back(0);
    pool.insert(pool.end(), l.begin(), l.end());
    return c;
  }
  DB db() {
    DB d{};
    d.lits = pool.data(), d.ot_off = off, d.ot_size = size, d.ot_refs = refs.data(), d.nvars = 15;
    return d;
  }
};

// the resolvents on variable 1 of gate clauses with the others
static int resolvents(const DB& db, u32 p, const std::set<u32>& gate) {
  int n = 0;
  const OLV a = olist(db, p), b = olist(db, FLIP(p));
  for (u32 i = 0; i < a.n; i++)
    for (u32 j = 0; j < b.n; j++) {
      const u32 c = a.r[i], d = b.r[j];
      if (!is_original(db, c) || !is_original(db, d) || gate.count(c) == gate.count(d)) continue;
      n += merge_len(ABS(p), clause(db, c), clause(db, d)) > 1;
    }
  return n;
}

int main(int argc, char** argv) {
  const int trials = argc > 1 ? atoi(argv[1]) : 1000;
  g_rng.seed(3);
  int equ = 0, ao = 0, refused = 0, repeated = 0;
  for (int t = 0; t < trials; t++) {
    Lists f;
    const u32 vars = 2 + below(4);
    const auto lit = [&] { return 2 * (2 + below(vars)) + below(2); };
    std::vector<std::vector<u32>> gate;  // a gate to be found, in half of the trials
    if (below(2)) {
      const u32 k = 1 + below(3), dx = 2 + below(2);
      std::vector<u32> out = {FLIP(dx)};
      for (u32 q = 0; q < k; q++) out.push_back(lit());
      for (u32 q = 1; q <= k; q++) gate.push_back({dx, FLIP(out[q])});
      if (below(3) == 0) out[1 + below(k)] = out[1 + below(k)];  // a literal twice, one missing
      gate.push_back(out);
    }
    for (u32 s = 0; s < 2; s++) {
      f.off[2 + s] = (u32)f.refs.size();
      for (const auto& c : gate)
        if (std::count(c.begin(), c.end(), 2 + s)) f.refs.push_back(f.add(c, below(12) == 0));
      for (u32 n = below(5); n; n--) {
        std::vector<u32> c = {2 + s};
        for (u32 k = 1 + below(3); k; k--) c.push_back(lit());
        f.refs.push_back(f.add(c, below(5) == 0));
      }
      f.size[2 + s] = (u32)f.refs.size() - f.off[2 + s];
    }
    f.off[4] = (u32)f.refs.size();
    DB db = f.db();
    const auto molten = [&] {
      std::set<u32> m;
      for (u32 c : f.refs)
        if (is_molten(db, c)) m.insert(c);
      return m;
    };
    const auto thaw = [&] {
      for (u32 c : f.refs)
        if (is_molten(db, c)) freeze(db, c);
    };
    const auto binaries = [&](u32 dx) {
      std::vector<u32> b;
      const OLV ol = olist(db, dx);
      for (u32 i = 0; i < ol.n; i++)
        if (is_original(db, ol.r[i]) && csize(db, ol.r[i]) == 2) b.push_back(ol.r[i]);
      return b;
    };
    const auto other = [&](u32 c, u32 dx) { return clits(db, c)[0] == dx ? clits(db, c)[1] : clits(db, c)[0]; };
    int orgs = 0;
    for (u32 c : f.refs) orgs += is_original(db, c);

    // equivalence of x
    u32 def = 0;
    std::set<u32> want;
    const std::vector<u32> bx = binaries(2), bn = binaries(3);
    if (bx.size() == 1)
      for (u32 c : bn) {
        std::vector<u32> conv = {3, FLIP(other(bx[0], 2))};
        std::sort(conv.begin(), conv.end());
        if (def || !std::equal(conv.begin(), conv.end(), clits(db, c))) continue;
        def = FLIP(other(bx[0], 2));
        want = {bx[0], c};
      }
    if (find_equ_gate(db, 2) != def || molten() != want) return fprintf(stderr, "trial %d: equivalence\n", t), 1;
    equ += def != 0;
    thaw();

    for (u32 dx = 2; dx < 4; dx++) {
      std::vector<u32> out = {FLIP(dx)};
      const std::vector<u32> b = binaries(dx);
      for (u32 c : b) out.push_back(FLIP(other(c, dx)));
      std::sort(out.begin(), out.end());
      bool found = false, counted = false;
      want.clear();
      const OLV ol = olist(db, FLIP(dx));
      for (u32 i = 0; i < ol.n && b.size() > 1 && !counted; i++) {
        const u32 c = ol.r[i], *l = clits(db, c);
        if (!is_original(db, c) || !std::equal(l, l + csize(db, c), out.begin(), out.end())) continue;
        std::set<u32> g(b.begin(), b.end());
        g.insert(c);
        counted = true;
        found = resolvents(db, dx, g) <= orgs;
        if (found) want = g;
        repeated += std::set<u32>(out.begin(), out.end()).size() < out.size();
      }
      Options o;
      o.ve_clause_limit = 0;
      o.ve_lbound_en = false;
      int added = 0;
      u32 lits = 0;
      const bool got = find_ao_gate(db, o, dx, orgs, added, lits);
      if (got != found || molten() != want)
        return fprintf(stderr, "trial %d: AND/OR of %u found %d, is %d\n", t, dx, (int)got, (int)found), 1;
      ao += found;
      refused += counted && !found;
      thaw();
    }
  }
  printf("{\"equivalences\": %d, \"gates\": %d, \"too_many\": %d, \"repeated\": %d}\n", equ, ao, refused, repeated);
  return 0;
}
