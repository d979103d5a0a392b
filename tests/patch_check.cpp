// Runs the patch search (cemc_amd/csrc/ce_patches.h) on sub-clusters read from
// standard input and writes the patches and their tables; driven by
// test_patches.py.
#include <cstdio>

#include "../cemc_amd/csrc/ce_patches.h"

using namespace cemc;

int main() {
  int n_sites, n_rec, q, n_species, bits, n_tab;
  if (std::scanf("%d %d %d %d %d %d", &n_sites, &n_rec, &q, &n_species, &bits, &n_tab) != 6) return 1;
  std::vector<PatchInput> in(n_rec);
  for (auto& r : in) {
    int n_orders;
    if (std::scanf("%d %d %d %d %u %d", &r.n, &r.site[0], &r.site[1], &r.site[2], &r.block, &n_orders) != 6) return 1;
    r.orders.resize(n_orders);
    for (auto& o : r.orders)
      if (std::scanf("%d %d %d", &o[0], &o[1], &o[2]) != 3) return 1;
  }
  std::vector<double> rec(n_tab);
  for (double& v : rec)
    if (std::scanf("%lf", &v) != 1) return 1;
  PatchCover cover;
  if (!PatchSearch(n_sites, in, q).run(&cover)) {
    std::printf("0 0\n");
    return 0;
  }
  const int slices = n_species - 1;
  int codes = 1;
  for (int i = 0; i < q; ++i) codes *= n_species;
  std::printf("%zu %zu\n", cover.patches.size(), cover.tables.size());
  for (const auto& p : cover.patches) {
    for (int i = 0; i < q; ++i) std::printf("%d ", p.site[i]);
    std::printf("%d\n", p.table);
  }
  std::vector<double> t(size_t(codes) * slices);
  for (const auto& terms : cover.tables) {
    patch_table(terms, n_species, q, slices, slices, bits, rec.data(), t.data());
    for (double v : t) std::printf("%.17g ", v);
    std::printf("\n");
  }
  return 0;
}
