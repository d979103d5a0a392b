// Patches: the sub-clusters of a site regrouped so that one table read covers
// many of them.  No HIP in here, so that it can be checked on the CPU.
//
// A flip of a site sums one table entry per sub-cluster that holds the site,
// each chosen by the species of at most three other members.  Sub-clusters
// overlap heavily: on FCC the 78 pairs and triplets within the second shell
// lie inside the six octahedra around the site, five other members each.  A
// patch is such a set of up to kQ member sites whose table, indexed by all
// their species at once, holds the sum over the sub-clusters inside it.
//
// The patches come in families: the images of one site set under the
// symmetries of the sub-clusters (site permutations that keep blocks and
// places).  A sub-cluster inside several patches of its family
// enters each with weight 1 / (their number), so the patches of a family
// have one table.  Families are chosen greedily by the sub-clusters that they
// newly cover per patch; what remains are pairs, packed kQ sites to a patch.
// The result is an exact regrouping: for every lattice the patch entries sum
// to the sub-clusters' entries (up to rounding).
#pragma once

#include <stdint.h>

#include <algorithm>
#include <array>
#include <map>
#include <memory>
#include <mutex>
#include <tuple>
#include <unordered_map>
#include <vector>

namespace cemc {

constexpr int kPatchMembers = 6;   // most members of a patch
constexpr int kPatchSites = 96;    // most distinct member sites the search takes

// Members per patch by species count: tables of S^q codes, 64 (two species),
// 243 (three) and 256 (four), which keep every table of a model in LDS.
inline int patch_members(int n_species) { return n_species == 2 ? 6 : (n_species == 3 ? 5 : (n_species == 4 ? 4 : 0)); }

// Species a | b << 8 of the swap in slot `slot` of a round of n moves; `w` is
// what the slot holds.  Slots past the last move hold a swap of an earlier
// round: made since, it would shift its first site's species a second time and
// index past the patch's table, so it counts as no swap.  (constexpr: the
// kernel calls it too.)
constexpr uint32_t slot_swap(uint32_t w, int slot, int n) { return slot < n ? w & 0xFFFFu : 0u; }

// One sub-cluster as seen from the reference site: its other members (site
// ids 0 .. n_sites-1 of the search) in code order, its table block, and the
// orders of the members that the block reads the same way (order o: member m
// stands where member o[m] stood; the identity always among them).
struct PatchInput {
  int n;
  int site[3];
  uint32_t block;
  std::vector<std::array<int, 3>> orders;
};

struct PatchTerm {
  uint32_t block;  // table block of the sub-cluster
  int n;
  int place[3];    // members' places in the patch, code order
  int share;       // patches of the family that hold the sub-cluster: weight 1 / share
};

struct PatchCover {
  struct Patch {
    std::array<int, kPatchMembers> site;  // member sites, -1 for unused places
    int table;
  };
  std::vector<Patch> patches;
  std::vector<std::vector<PatchTerm>> tables;
};

class PatchSearch {
 public:
  PatchSearch(int n_sites, const std::vector<PatchInput>& in, int q) : n_(n_sites), in_(in), q_(q) {}

  // false: more sites than the search takes (no patches)
  bool run(PatchCover* out) {
    if (n_ < 1 || n_ > kPatchSites || q_ < 1 || q_ > kPatchMembers) return false;
    index_inputs();
    find_symmetries();
    while (left_multi_ > 0) {
      const int f = best_family();
      if (f < 0) return false;
      take(families_[f], out);
    }
    pack_singles(out);
    return true;
  }

 private:
  using Tuple = std::array<int, kPatchMembers>;
  struct Family {
    int size;                   // members per patch
    std::vector<Tuple> images;  // members in corresponding order
    std::vector<int> holds;     // sub-clusters inside its patches, each once
  };

  static uint64_t key_of(const int* s, int k) {
    std::array<int, kPatchMembers> v;
    std::copy(s, s + k, v.begin());
    std::sort(v.begin(), v.begin() + k);
    uint64_t key = 0;
    for (int i = 0; i < k; ++i) key = (key << 8) | uint64_t(v[i] + 1);
    return key;
  }
  size_t at2(int a, int b) const { return size_t(a) * n_ + b; }
  size_t at3(int a, int b, int c) const { return (size_t(a) * n_ + b) * n_ + c; }

  void index_inputs() {
    const int R = int(in_.size());
    left_.assign(R, 1);
    w1_.assign(n_, 0);
    w2_.assign(size_t(n_) * n_, 0);
    w3_.assign(size_t(n_) * n_ * n_, 0);
    s1_.assign(n_, 0);
    s2_.assign(size_t(n_) * n_, 0);
    s3_.assign(size_t(n_) * n_ * n_, 0);
    set1_ = s1_;
    set2_ = s2_;
    set3_ = s3_;
    std::map<uint64_t, std::vector<int>> by_set;
    for (int r = 0; r < R; ++r) {
      by_set[key_of(in_[r].site, in_[r].n)].push_back(r);
      if (in_[r].n > 1) ++left_multi_;
      add_weight(r, weight_of(r));
    }
    // what lies on an ordered set of one, two or three sites: sub-clusters'
    // blocks with the places of their members, as an id (0: nothing)
    std::map<std::vector<uint64_t>, int> ids;
    sets_.assign(1, {});
    for (const auto& kv : by_set) {
      sets_.push_back(kv.second);
      const PatchInput& any = in_[kv.second[0]];
      const int k = any.n;
      int perm[3] = {0, 1, 2};
      int base[3];
      std::copy(any.site, any.site + k, base);
      std::sort(base, base + k);
      do {
        int o[3] = {0, 0, 0};
        for (int i = 0; i < k; ++i) o[i] = base[perm[i]];
        std::vector<uint64_t> sig;
        for (int r : kv.second) {
          const std::array<int, 3> at = places(r, o, k);
          uint64_t v = in_[r].block;
          for (int m = 0; m < k; ++m) v = v * 4 + uint64_t(at[m]);
          sig.push_back(v);
        }
        std::sort(sig.begin(), sig.end());
        sig.push_back(uint64_t(k));
        const int id = ids.emplace(sig, int(ids.size()) + 1).first->second;
        const int set = int(sets_.size()) - 1;
        if (k == 1) s1_[o[0]] = id, set1_[o[0]] = set;
        if (k == 2) s2_[at2(o[0], o[1])] = id, set2_[at2(o[0], o[1])] = set;
        if (k == 3) s3_[at3(o[0], o[1], o[2])] = id, set3_[at3(o[0], o[1], o[2])] = set;
      } while (std::next_permutation(perm, perm + k));
    }
  }

  // places of the members of r among the k sites s, the smallest of the
  // equivalent orders
  std::array<int, 3> places(int r, const int* s, int k) const {
    std::array<int, 3> best{9, 9, 9};
    for (const auto& o : in_[r].orders) {
      std::array<int, 3> at{0, 0, 0};
      for (int m = 0; m < in_[r].n; ++m) at[m] = int(std::find(s, s + k, in_[r].site[o[m]]) - s);
      best = std::min(best, at);
    }
    return best;
  }

  // covering a sub-cluster of more members saves more reads
  int weight_of(int r) const { return in_[r].n == 1 ? 1 : (in_[r].n == 2 ? 2 : 4); }
  void add_weight(int r, int w) {
    const int* s = in_[r].site;
    if (in_[r].n == 1) {
      w1_[s[0]] += w;
    } else if (in_[r].n == 2) {
      w2_[at2(s[0], s[1])] += w;
      w2_[at2(s[1], s[0])] += w;
    } else {
      int p[3] = {0, 1, 2};
      do w3_[at3(s[p[0]], s[p[1]], s[p[2]])] += w;
      while (std::next_permutation(p, p + 3));
    }
  }

  // uncovered weight that adding x to the first k sites of s brings
  int gain(const Tuple& s, int k, int x) const {
    int g = w1_[x];
    for (int i = 0; i < k; ++i) {
      g += w2_[at2(x, s[i])];
      for (int j = i + 1; j < k; ++j) g += w3_[at3(x, s[i], s[j])];
    }
    return g;
  }
  bool linked(const Tuple& s, int k, int x) const {
    for (int i = 0; i < k; ++i) {
      if (s2_[at2(x, s[i])]) return true;
      for (int j = i + 1; j < k; ++j)
        if (s3_[at3(x, s[i], s[j])]) return true;
    }
    return false;
  }

  // Symmetries: permutations of the sites that share a sub-cluster with
  // another member, found site by site, each keeping what lies on every site
  // and pair.  Whether a patch and its image have one table is decided by
  // their terms (take), so a permutation that breaks a triple only costs a
  // table, and the search may stop early.
  void find_symmetries() {
    std::vector<int> who;
    for (int x = 0; x < n_; ++x) {
      bool multi = false;
      for (int y = 0; !multi && y < n_; ++y) {
        multi = w2_[at2(x, y)] != 0;
        for (int z = 0; !multi && z < n_; ++z) multi = w3_[at3(x, y, z)] != 0;
      }
      if (multi) who.push_back(x);
    }
    std::vector<int> to(n_);
    for (int x = 0; x < n_; ++x) to[x] = x;
    syms_.assign(1, to);
    std::vector<char> used(n_, 0);
    budget_ = 400000;
    extend(who, 0, to, used);
  }
  void extend(const std::vector<int>& who, size_t k, std::vector<int>& to, std::vector<char>& used) {
    if (syms_.size() >= kMaxSyms || budget_ < 0) return;
    if (k == who.size()) {
      if (to != syms_[0]) syms_.push_back(to);
      return;
    }
    const int s = who[k];
    for (int x : who) {
      if (used[x] || s1_[x] != s1_[s]) continue;
      bool ok = true;
      for (size_t i = 0; ok && i < k; ++i) {
        --budget_;
        ok = s2_[at2(to[who[i]], x)] == s2_[at2(who[i], s)];
      }
      for (size_t i = 1; ok && i < k && i < 8; ++i)
        ok = s3_[at3(to[who[i - 1]], to[who[i]], x)] == s3_[at3(who[i - 1], who[i], s)];
      if (!ok) continue;
      to[s] = x;
      used[x] = 1;
      extend(who, k + 1, to, used);
      used[x] = 0;
    }
    to[s] = s;
  }

  // a set of sites as a bit mask
  using SetKey = std::pair<uint64_t, uint64_t>;
  struct SetHash {
    size_t operator()(const SetKey& k) const {
      return size_t((k.first * 0x9E3779B97F4A7C15ull) ^ (k.second * 0xC2B2AE3D27D4EB4Full));
    }
  };
  static SetKey mask_of(const Tuple& s, int size) {
    uint64_t m[2] = {0, 0};
    for (int i = 0; i < size; ++i) m[s[i] >> 6] |= uint64_t(1) << (s[i] & 63);
    return {m[0], m[1]};
  }
  int family_of(const Tuple& s, int size) {
    auto it = family_at_.find(mask_of(s, size));
    if (it != family_at_.end()) return it->second;
    const int id = int(families_.size());
    families_.emplace_back();
    Family& f = families_.back();
    f.size = size;
    held_.assign(in_.size(), 0);
    for (const auto& to : syms_) {
      Tuple v;
      v.fill(-1);
      for (int i = 0; i < size; ++i) v[i] = to[s[i]];
      if (!family_at_.emplace(mask_of(v, size), id).second) continue;  // the same set in another order
      f.images.push_back(v);
      inside(v, size, [&](int r) {
        if (!held_[r]) f.holds.push_back(r);
        held_[r] = 1;
      });
    }
    return id;
  }

  // sub-clusters inside the patch `s`: fn(record id)
  template <class Fn>
  void inside(const Tuple& s, int size, Fn fn) const {
    for (int a = 0; a < size; ++a) {
      for (int r : sets_[set1_[s[a]]]) fn(r);
      for (int b = a + 1; b < size; ++b) {
        for (int r : sets_[set2_[at2(s[a], s[b])]]) fn(r);
        for (int c = b + 1; c < size; ++c)
          for (int r : sets_[set3_[at3(s[a], s[b], s[c])]]) fn(r);
      }
    }
  }

  // one uncovered sub-cluster of each block grows site by site by what the
  // sites newly cover (the kBranch best at each step, equals taken once per
  // family); every set on the way is a candidate
  int best_family() {
    std::map<uint32_t, int> seeds;
    for (int r = 0; r < int(in_.size()); ++r)
      if (left_[r] && in_[r].n > 1) seeds.emplace(in_[r].block, r);
    best_ = -1;
    best_score_ = 0.0;
    scored_.assign(families_.size(), 0);
    for (const auto& kv : seeds) {
      Tuple s;
      s.fill(-1);
      std::copy(in_[kv.second].site, in_[kv.second].site + in_[kv.second].n, s.begin());
      if (in_[kv.second].n <= q_) grow(s, in_[kv.second].n);
    }
    return best_;
  }

  void grow(const Tuple& s, int k) {
    const int f = family_of(s, k);
    if (f >= int(scored_.size())) scored_.resize(f + 1, 0);
    if (scored_[f]) return;
    scored_[f] = 1;
    const double sc = score(families_[f]);
    if (sc > best_score_ * (1.0 + 1e-12)) {
      best_score_ = sc;
      best_ = f;
    }
    if (k == q_) return;
    std::vector<std::pair<int, int>> next;  // (-gain, site)
    for (int y = 0; y < n_; ++y) {
      if (std::find(s.begin(), s.begin() + k, y) != s.begin() + k || !linked(s, k, y)) continue;
      const int g = gain(s, k, y);
      if (g > 0) next.emplace_back(-g, y);
    }
    std::sort(next.begin(), next.end());
    if (int(next.size()) > kBranch) next.resize(kBranch);
    for (const auto& gy : next) {
      Tuple t = s;
      t[k] = gy.second;
      grow(t, k + 1);
    }
  }

  double score(const Family& f) const {
    int64_t w = 0;
    for (int r : f.holds) w += left_[r] ? weight_of(r) : 0;
    return double(w) / double(f.images.size());
  }

  void take(Family& f, PatchCover* out) {
    // patches of neighbouring lanes read neighbouring members (128 quaternary
    // 32^3 replicas: 16.5 ms, in the symmetries' order 17.3)
    std::sort(f.images.begin(), f.images.end(), [&](const Tuple& x, const Tuple& y) {
      return key_of(x.data(), f.size) < key_of(y.data(), f.size);
    });
    std::vector<int> share(in_.size(), 0);
    for (const Tuple& s : f.images)
      inside(s, f.size, [&](int r) { share[r] += left_[r]; });
    std::map<std::vector<int64_t>, int> table_of;  // terms -> table (one, unless the shares differ)
    for (const Tuple& s : f.images) {
      std::vector<PatchTerm> terms;
      inside(s, f.size, [&](int r) {
        if (!left_[r]) return;
        const std::array<int, 3> at = places(r, s.data(), f.size);
        terms.push_back(PatchTerm{in_[r].block, in_[r].n, {at[0], at[1], at[2]}, share[r]});
      });
      if (terms.empty()) continue;
      add_patch(s, terms, table_of, out);
    }
    for (int r = 0; r < int(in_.size()); ++r)
      if (share[r] > 0) cover(r);
  }

  void cover(int r) {
    left_[r] = 0;
    add_weight(r, -weight_of(r));
    if (in_[r].n > 1) --left_multi_;
  }

  static void add_patch(const Tuple& s, std::vector<PatchTerm>& terms, std::map<std::vector<int64_t>, int>& table_of,
                        PatchCover* out) {
    std::sort(terms.begin(), terms.end(), [](const PatchTerm& x, const PatchTerm& y) {
      return std::make_tuple(x.n, x.place[0], x.place[1], x.place[2], x.block, x.share) <
             std::make_tuple(y.n, y.place[0], y.place[1], y.place[2], y.block, y.share);
    });
    std::vector<int64_t> key;
    for (const PatchTerm& t : terms)
      for (int64_t v : {int64_t(t.n), int64_t(t.place[0]), int64_t(t.place[1]), int64_t(t.place[2]), int64_t(t.block),
                        int64_t(t.share)})
        key.push_back(v);
    auto it = table_of.find(key);
    if (it == table_of.end()) {
      it = table_of.emplace(key, int(out->tables.size())).first;
      out->tables.push_back(terms);
    }
    out->patches.push_back(PatchCover::Patch{s, it->second});
  }

  // pairs left over: sites with the same blocks share one table
  void pack_singles(PatchCover* out) {
    std::map<std::vector<uint32_t>, std::vector<int>> like;
    for (int x = 0; x < n_; ++x) {
      std::vector<uint32_t> blocks;
      for (int r : sets_[set1_[x]])
        if (left_[r]) blocks.push_back(in_[r].block);
      std::sort(blocks.begin(), blocks.end());
      if (!blocks.empty()) like[blocks].push_back(x);
    }
    std::map<std::vector<int64_t>, int> table_of;
    for (const auto& kv : like) {
      const int n = int(kv.second.size()), chunks = (n + q_ - 1) / q_, per = (n + chunks - 1) / chunks;
      for (int i = 0; i < n; i += per) {
        Tuple s;
        s.fill(-1);
        std::vector<PatchTerm> terms;
        for (int k = 0; k < per && i + k < n; ++k) {
          s[k] = kv.second[i + k];
          for (uint32_t b : kv.first) terms.push_back(PatchTerm{b, 1, {k, 0, 0}, 1});
        }
        add_patch(s, terms, table_of, out);
      }
    }
  }

  const int n_;
  const std::vector<PatchInput>& in_;
  const int q_;
  int left_multi_ = 0;
  std::vector<int> left_;
  std::vector<std::vector<int>> sets_;  // sub-clusters on one site set ([0]: none)
  // by ordered sites: uncovered weight, what lies there (0: nothing), index into sets_
  std::vector<int> w1_, w2_, w3_, s1_, s2_, s3_, set1_, set2_, set3_;
  std::vector<std::vector<int>> syms_;  // [0]: the identity
  int64_t budget_ = 0;
  std::vector<Family> families_;
  std::unordered_map<SetKey, int, SetHash> family_at_;
  std::vector<char> held_;
  static constexpr int kBranch = 4;
  static constexpr size_t kMaxSyms = 96;
  int best_ = -1;
  double best_score_ = 0.0;
  std::vector<char> scored_;
};

// The covers of the cluster sets seen last.  A search takes 0.5 to 20 ms; models
// of one cluster set at several sizes, or made one after the other, share its
// outcome, which depends on the whole key.  Safe for several threads; at most
// kKept covers, of some 100 KB with their keys, stay.
class PatchCovers {
 public:
  static constexpr size_t kKept = 16;
  // nullptr: the search does not take the input
  std::shared_ptr<const PatchCover> get(int n_sites, const std::vector<PatchInput>& in, int q) {
    std::vector<uint32_t> key{uint32_t(n_sites), uint32_t(q)};
    for (const PatchInput& r : in) {
      for (int v : {r.n, r.site[0], r.site[1], r.site[2], int(r.orders.size())}) key.push_back(uint32_t(v));
      key.push_back(r.block);
      for (const auto& o : r.orders) key.push_back(uint32_t(o[0] | (o[1] << 8) | (o[2] << 16)));
    }
    {
      std::lock_guard<std::mutex> lock(mutex_);
      for (size_t i = 0; i < kept_.size(); ++i)
        if (kept_[i].first == key) {
          std::rotate(kept_.begin(), kept_.begin() + i, kept_.begin() + i + 1);  // to the front
          return kept_[0].second;
        }
    }
    auto cover = std::make_shared<PatchCover>();
    if (!PatchSearch(n_sites, in, q).run(cover.get())) cover.reset();
    std::lock_guard<std::mutex> lock(mutex_);
    ++searches_;
    kept_.insert(kept_.begin(), std::make_pair(std::move(key), std::shared_ptr<const PatchCover>(cover)));
    if (kept_.size() > kKept) kept_.pop_back();
    return cover;
  }
  int searches() const {
    std::lock_guard<std::mutex> lock(mutex_);
    return searches_;
  }
  size_t size() const {
    std::lock_guard<std::mutex> lock(mutex_);
    return kept_.size();
  }

 private:
  mutable std::mutex mutex_;
  int searches_ = 0;
  std::vector<std::pair<std::vector<uint32_t>, std::shared_ptr<const PatchCover>>> kept_;  // newest first
};

// Adds the patch table of `terms` to dst: entry (code, d) at dst[stride * code
// + d], code = sum over places of species * S^place.  `rec` holds the
// sub-clusters' tables: entry (code, d) of a block at rec[block + d * 2^(3
// bits) + code], `bits` code bits per species.
inline void patch_table(const std::vector<PatchTerm>& terms, int n_species, int q, int slices, int stride, int bits,
                        const double* rec, double* dst) {
  int n_codes = 1;
  for (int i = 0; i < q; ++i) n_codes *= n_species;
  for (int code = 0; code < n_codes; ++code) {
    int sp[kPatchMembers];
    for (int i = 0, c = code; i < q; ++i, c /= n_species) sp[i] = c % n_species;
    for (int d = 0; d < slices; ++d) {
      long double sum = 0.0L;  // rounded once: no less exact than the terms' own sum
      for (const PatchTerm& t : terms) {
        int rc = 0;
        for (int m = 0; m < t.n; ++m) rc |= sp[t.place[m]] << (bits * m);
        const long double x = rec[t.block + (uint32_t(d) << (3 * bits)) + rc];
        sum += t.share == 1 ? x : x / t.share;
      }
      dst[size_t(stride) * code + d] = double(sum);
    }
  }
}

}  // namespace cemc
