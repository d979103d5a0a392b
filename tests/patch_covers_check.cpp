// Models that share patch covers (PatchCovers, cemc_amd/csrc/ce_patches.h):
// reads sub-cluster sets from standard input, looks each up from four threads
// at once, then many sets that differ in one block.  Prints the searches that
// the sets took, whether every cover is the search's own, the covers kept at the
// end and whether the newest is among them; driven by test_patch_covers.py.
#include <cstdio>
#include <thread>

#include "../cemc_amd/csrc/ce_patches.h"

using namespace cemc;

static bool same(const PatchCover& a, const PatchCover& b) {
  if (a.patches.size() != b.patches.size() || a.tables.size() != b.tables.size()) return false;
  for (size_t i = 0; i < a.patches.size(); ++i)
    if (a.patches[i].site != b.patches[i].site || a.patches[i].table != b.patches[i].table) return false;
  for (size_t t = 0; t < a.tables.size(); ++t) {
    if (a.tables[t].size() != b.tables[t].size()) return false;
    for (size_t k = 0; k < a.tables[t].size(); ++k) {
      const PatchTerm &x = a.tables[t][k], &y = b.tables[t][k];
      if (x.block != y.block || x.n != y.n || x.share != y.share || !std::equal(x.place, x.place + x.n, y.place))
        return false;
    }
  }
  return true;
}

int main() {
  int n_sets;
  if (std::scanf("%d", &n_sets) != 1) return 1;
  PatchCovers covers;
  bool good = true;
  std::vector<PatchInput> in;
  int n_sites = 0, q = 0;
  for (int i = 0; i < n_sets; ++i) {
    int n_rec;
    if (std::scanf("%d %d %d", &n_sites, &n_rec, &q) != 3) return 1;
    in.assign(n_rec, PatchInput());
    for (auto& r : in) {
      if (std::scanf("%d %d %d %d %u", &r.n, &r.site[0], &r.site[1], &r.site[2], &r.block) != 5) return 1;
      r.orders.assign(1, {0, 1, 2});
    }
    PatchCover own;
    PatchSearch(n_sites, in, q).run(&own);
    covers.get(n_sites, in, q);
    std::vector<std::thread> threads;
    std::vector<char> ok(4, 0);
    for (int t = 0; t < 4; ++t) threads.emplace_back([&, t] { ok[t] = same(*covers.get(n_sites, in, q), own); });
    for (auto& t : threads) t.join();
    for (char c : ok) good = good && c;
  }
  const int searches = covers.searches();
  for (uint32_t k = 0; k < 2 * PatchCovers::kKept; ++k) {
    in[0].block += 1000000;
    covers.get(n_sites, in, q);
  }
  const int before = covers.searches();
  covers.get(n_sites, in, q);
  std::printf("%d %d %zu %d\n", searches, int(good), covers.size(), int(covers.searches() == before));
  return 0;
}
