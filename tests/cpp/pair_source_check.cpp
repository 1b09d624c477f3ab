// The pair tables' source slots (PairPlan::tsrc): with a copy list every entry
// is the table of slots with each listed ghost replaced by the active U point
// that it copies, and only those; without one there are none; check_pairs
// reports a source dropped, one that a plain ghost is given, and a table cut
// short.  Input file as for pair_plan_check.cpp.
#include "evp1d_tiles.hpp"
#include <cstdio>
#include <map>
#include <vector>

int main(int argc, char **argv) {
  if (argc < 2) return 2;
  FILE *f = fopen(argv[1], "rb");
  if (!f) return 2;
  int hdr[2];
  if (fread(hdr, 4, 2, f) != 2) return 2;
  const int na = hdr[0], navel = hdr[1];
  std::vector<std::vector<int32_t>> idx(6, std::vector<int32_t>(na));
  const int32_t *ip[6];
  for (int k = 0; k < 6; ++k) {
    if (fread(idx[k].data(), 4, na, f) != (size_t)na) return 2;
    ip[k] = idx[k].data();
  }
  std::vector<uint8_t> skip(na);
  if (fread(skip.data(), 1, na, f) != (size_t)na) return 2;
  fclose(f);
  int fails = 0;
  const int shapes[3][2] = {{31, 19}, {15, 11}, {5, 7}};
  for (const auto &sh : shapes) {
    const evp1d::TilePlan p = evp1d::plan_tiles(na, navel, ip, skip.data(), sh[0], sh[1], 2560);
    const int u_begin = p.cnt[0], u_end = p.cnt[0] + p.cnt[1] + p.cnt[2];
    std::vector<int32_t> hd, hs;   // every third ghost: an active U point, another point, zero
    for (int g = na, k = 0; g < navel; g += 3, ++k) {
      hd.push_back(g);
      hs.push_back(k % 3 == 0 ? u_begin + (k * 7919) % (u_end - u_begin)
                              : k % 3 == 1 ? (k * 31) % (p.cnt[0] > 0 ? p.cnt[0] : 1) : -1);
    }
    std::map<int32_t, int32_t> copy;
    for (size_t k = 0; k < hd.size(); ++k) copy[hd[k]] = hs[k];
    evp1d::HaloList hl;
    hl.n = (int)hd.size();
    hl.dst = hd.data();
    hl.src = hs.data();
    auto check = [&](const evp1d::PairPlan &q, const evp1d::HaloList &h) {
      return evp1d::check_pairs(q, p, na, navel, ip, skip.data(), h);
    };
    const evp1d::PairPlan none = evp1d::plan_pairs(p, na, navel, ip, skip.data(), 4096, 4096, 1024);
    const evp1d::PairPlan q = evp1d::plan_pairs(p, na, navel, ip, skip.data(), 4096, 4096, 1024, hl);
    fails += !none.ok || !q.ok || !none.tsrc.empty() || q.tsrc.size() != q.tnbr.size() || !check(q, hl).empty();
    size_t named = 0, plain = q.tsrc.size(), source = q.tsrc.size();
    for (size_t j = 0; j < q.tsrc.size(); ++j) {
      const auto c = copy.find(q.tnbr[j]);
      const bool active = c != copy.end() && c->second >= u_begin && c->second < u_end;
      fails += q.tsrc[j] != (active ? c->second : q.tnbr[j]);
      named += active;
      if (active) source = j;
      else if (q.tnbr[j] >= na) plain = j;
    }
    fails += named == 0 || plain == q.tsrc.size();
    evp1d::PairPlan a = q, b = q, c = q;
    a.tsrc[source] = a.tnbr[source];
    b.tsrc[plain] = u_begin;
    c.tsrc.resize(c.tsrc.size() - 4);
    fails += check(a, hl).empty() + check(b, hl).empty() + check(c, hl).empty();
    printf("tile %dx%d: %zu of %zu entries name a source; failures so far %d\n", sh[0], sh[1], named, q.tsrc.size(), fails);
  }
  return fails;
}
extern "C" int evp1d__set_error(int c, const char *) { return c; }
