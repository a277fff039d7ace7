// Host build of the elimination of one variable (ve_apply,
// parafrost_amd/csrc/pfs_items.hpp) for the CPU tests.  TEST INFRASTRUCTURE
// ONLY.
//
// "pairs": a variable with 65,536 entries in one list and 65,537 in the other,
// 2^32 + 65,536 pairs, nearly all of them of one learnt clause that gives no
// resolvent; the originals come last in both lists.  Every resolvent has to be
// there.  "few": the decision counted a resolvent more than there are; the
// error counter has to say so.
#include <cstdio>
#include <cstring>
#include <vector>

#include "../../parafrost_amd/csrc/pfs_items.hpp"

using namespace pfs;

struct Formula {
  std::vector<u32> pool, lists[2];
  u32 add(const std::vector<u32>& l, u8 flags) {
    const u32 c = (u32)pool.size();
    pool.push_back(make_hdr((u32)l.size(), flags));
    pool.push_back(calc_sig(l.data(), (u32)l.size()));
    pool.push_back(0);
    pool.insert(pool.end(), l.begin(), l.end());
    return c;
  }
};

// eliminates variable 1; the resolvents in order, the errors in *error
static std::vector<std::vector<u32>> eliminate(Formula& f, u32 ncls, u32 nlits, u32* error) {
  const u32 n0 = (u32)f.pool.size(), room = nlits + CL_HDR * ncls;
  f.pool.resize(n0 + room, 0);
  std::vector<u32> c_off(ncls, 0), refs = f.lists[0], stack(1u << 12), recs(64);
  refs.insert(refs.end(), f.lists[1].begin(), f.lists[1].end());
  u32 ot_off[5] = {0, 0, 0, (u32)f.lists[0].size(), (u32)refs.size()};
  u32 ot_size[4] = {0, 0, (u32)f.lists[0].size(), (u32)f.lists[1].size()};
  std::vector<u32> assign(64, 0), vorg(64);
  std::vector<u8> vstate(64, 0);
  for (u32 v = 0; v < 64; v++) vorg[v] = v;
  DB db{};
  db.lits = f.pool.data();
  db.c_off = c_off.data();
  db.ot_off = ot_off, db.ot_size = ot_size, db.ot_refs = refs.data();
  db.assign = assign.data(), db.vstate = vstate.data(), db.vorg = vorg.data();
  db.nvars = 63;
  u32 type = VT_RES, def = 0, words = nlits + CL_HDR * ncls, nstack = 64, zero = 0, units = 0;
  const VeDecision d{&type, &def, &ncls, &words, &nstack};
  VeApply a{};
  a.cls_base = a.lit_base = a.stack_base = &zero;
  a.cls0 = 0, a.lit0 = n0, a.stack0 = 0;
  a.cls_cap = ncls, a.lit_cap = n0 + room, a.stack_cap = (u32)stack.size();
  a.stack = stack.data();
  a.units = UnitOut{recs.data(), &units, 16};
  a.error = error;
  ve_apply(db, db, 1, 0, d, a);
  std::vector<std::vector<u32>> out;
  for (u32 c : c_off)
    out.emplace_back(f.pool.data() + c + CL_HDR, f.pool.data() + c + CL_HDR + (c ? csize(db, c) : 0u));
  return out;
}

int main(int argc, char** argv) {
  const bool few = argc > 1 && !strcmp(argv[1], "few");
  const u32 np = few ? 3 : 65536, nn = few ? 4 : 65537;
  Formula f;
  f.add({60}, ST_DELETED);  // no clause has handle 0
  const u32 lp = f.add({2, 40}, ST_LEARNT), ln = f.add({3, 42}, ST_LEARNT);
  f.lists[0].assign(np, lp);
  f.lists[1].assign(nn, ln);
  f.lists[0][np - 2] = f.add({2, 4, 6}, ST_ORIGINAL);
  f.lists[0][np - 1] = f.add({2, 8}, ST_ORIGINAL);
  f.lists[1][nn - 3] = f.add({3, 10}, ST_ORIGINAL);
  f.lists[1][nn - 2] = f.add({3, 5, 12}, ST_ORIGINAL);  // a tautology with the first
  f.lists[1][nn - 1] = f.add({3, 8, 14}, ST_ORIGINAL);
  u32 error = 0;
  const std::vector<std::vector<u32>> want = {{4, 6, 10}, {4, 6, 8, 14}, {8, 10}, {5, 8, 12}, {8, 14}};
  const auto got = eliminate(f, few ? 6 : 5, few ? 16 : 14, &error);
  if (few) return printf("errors %u\n", error), error ? 0 : 1;
  printf("resolvents right: %d, errors %u\n", (int)(got == want), error);
  return got == want && !error ? 0 : 1;
}
