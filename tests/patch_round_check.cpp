// The index arithmetic of a round of the patch kernel (ce_patch_kernel.h) on a
// small periodic lattice, with random rounds of 1 to 16 open swaps: a slot
// past the last open move keeps the swap of an earlier round, and every slot
// is evaluated.  Reads the lattice and its sub-clusters from standard input,
// prints the evaluations and how many of them leave their patch's table;
// driven by test_patch_rounds.py.
#include <cstdio>
#include <cstdlib>
#include <random>

#include "../cemc_amd/csrc/ce_patches.h"

using namespace cemc;

int main() {
  int L[3], S, q, n_cols, n_rec, rounds;
  if (std::scanf("%d %d %d %d %d %d %d %d", &L[0], &L[1], &L[2], &S, &q, &n_cols, &n_rec, &rounds) != 8) return 1;
  std::vector<std::array<int, 3>> off(n_cols);
  for (auto& o : off)
    if (std::scanf("%d %d %d", &o[0], &o[1], &o[2]) != 3) return 1;
  std::vector<PatchInput> in(n_rec);
  for (auto& r : in) {
    if (std::scanf("%d %d %d %d %u", &r.n, &r.site[0], &r.site[1], &r.site[2], &r.block) != 5) return 1;
    r.orders.assign(1, {0, 1, 2});
  }
  PatchCover cover;
  if (!PatchSearch(n_cols, in, q).run(&cover)) return 1;
  // a table holds the last place's codes where a term uses that place
  std::vector<char> full(cover.tables.size(), 0);
  for (size_t t = 0; t < full.size(); ++t)
    for (const auto& term : cover.tables[t])
      for (int m = 0; m < term.n; ++m) full[t] |= term.place[m] == q - 1;
  const int n_patch = int(cover.patches.size());
  const int N = L[0] * L[1] * L[2];
  auto at = [&](int site, const std::array<int, 3>& o) {
    const int x = site / (L[1] * L[2]), y = site / L[2] % L[1], z = site % L[2];
    auto wrap = [](int v, int n) { return ((v % n) + n) % n; };
    return (wrap(x + o[0], L[0]) * L[1] + wrap(y + o[1], L[1])) * L[2] + wrap(z + o[2], L[2]);
  };
  std::mt19937 rng(3);
  std::vector<int> occ(N);
  for (int& s : occ) s = int(rng() % S);
  constexpr int kK = 16;
  struct Slot {
    int i = 0, j = 0;
    uint32_t w = 0;
  } slots[kK];
  long n_eval = 0, n_out = 0;
  for (int r = 0; r < rounds; ++r) {
    const int n = 1 + int(rng() % kK);
    std::vector<char> touched(N, 0);
    for (int k = 0; k < n; ++k) {
      int i, j;
      do {
        i = int(rng() % N);
        // half of the swaps between sites that interact
        j = (rng() & 1) ? at(i, off[rng() % n_cols]) : int(rng() % N);
      } while (i == j || occ[i] == occ[j]);
      slots[k] = Slot{i, j, uint32_t(occ[i]) | (uint32_t(occ[j]) << 8) | (uint32_t(k) << 16)};
    }
    for (int k = 0; k < kK; ++k) {
      const uint32_t sw = slot_swap(slots[k].w, k, n);
      const int ds = int(sw >> 8) - int(sw & 255u);  // site i, already changed
      for (int p = 0; p < n_patch; ++p) {
        int code = 0, weight = 1, codes = 1;
        for (int m = 0; m < q; ++m, weight *= S) {
          const int member = cover.patches[p].site[m];
          const bool held = m < q - 1 || full[cover.patches[p].table];
          const int site = member >= 0 ? at(slots[k].j, off[member]) : slots[k].j;
          codes *= held ? S : 1;
          code += (held ? weight : 0) * (occ[site] + (member >= 0 && site == slots[k].i ? ds : 0));
        }
        ++n_eval;
        n_out += code < 0 || code >= codes;
      }
    }
    for (int k = 0; k < n; ++k) {  // most swaps are made, those that earlier ones left valid
      if (touched[slots[k].i] || touched[slots[k].j] || rng() % 4 == 0) continue;
      std::swap(occ[slots[k].i], occ[slots[k].j]);
      touched[slots[k].i] = touched[slots[k].j] = 1;
    }
  }
  std::printf("%ld %ld\n", n_eval, n_out);
  return 0;
}
