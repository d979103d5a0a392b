// Patch kernel of the cluster-expansion Metropolis engine (gfx950): the sweep
// of one chain with the sub-clusters of a site regrouped into patches
// (ce_patches.h).  Instantiations: ce_patch_inst.hip.
//
// One workgroup of kW waves owns one chain on a closed-form periodic lattice
// with one translation group; the padded occupation box, the species tracker
// and the patch tables stay in LDS for the launch.
//
// Rounds.  The first kK moves of the 64-move block that are still open are
// evaluated against the same state.  A move that an accepted earlier one of
// the round reaches (reads a site or shares a tracker slot with) is blocked,
// and so is one that a blocked one reaches; the others are made at once, in
// any order, since none reads what another writes (interactions are mutual:
// models where they are not have no patches).  Blocked moves stay open for the
// next round.  (Ending the round at the first blocked move instead made 5.6
// moves of eight for hot flips on 10^3 sites, now about 11 of 16; swaps there at
// acceptance 0.7 make 4.2.  Where most moves conflict the host keeps a chain off
// this kernel, conflict_chance.)
//
// Work split.  A flip needs 12 (two species, pairs to the 4th shell and
// triplets to the 2nd), 59 (three species, four-body clusters) or 426 (four
// species, four-body to the 3rd shell) patch entries where it needed 114, 494
// and 1746 sub-cluster entries.  One wave takes 16 moves at once, a quad of
// lanes each; several waves take a row of 16 lanes per move, or a wave per
// move above 64 patches.
//
// What bounds it: instruction issue and LDS latency of the dependent chain of
// a round, not bandwidth (binary SGC chains, counters per move: 18 VALU, 4
// LDS and 3 scalar instructions, 27 of 42 quad-cycles issuing, 11 waiting; the
// sweep kernel's rounds of eight: 37 VALU, 8 LDS and 9 scalar, 60 of 90
// issuing).  So the loads of a phase are issued together before the first wait
// (one binary chain, 40000 swaps: 14.6 -> 12.0 ms by that and by reading the
// tracker in the round instead of comparing every commit with every lane);
// which moves reach which is tested while the members are in flight; and what
// the next round does not need is put off to the end of the block, where lane l
// holds move l: energies by one prefix sum over the lanes, sample sums in
// per-lane accumulators added up once per launch.  Blocks are the 64-move blocks
// of the chain's stream, and a launch that ends inside one leaves its energy
// changes to the next, so energies do not depend on where launches end.
// Four-species models are bound by LDS reads instead: 125 a swap, three
// bank-conflict cycles each, 28 % of the cycles issuing at eight waves.
//
// Measured against the sweep kernel's automatic shapes, per pass with its reads
// of the results: 1024 binary SGC chains of 500 sweeps 149 -> 63 ms (the
// kernel 133 -> 53), 256 ternary chains of 512-4096 sites 56 -> 18 ms, a mix of
// 48 binary and ternary chains 5.8 -> 1.6 ms, 128 quaternary 32^3 replicas 56.3
// -> 16.3 ms, one binary chain 23.9 -> 11.8 ms, 128 quaternary 8^3 chains 5.4 ->
// 2.3 ms (1.24 ms of it the kernel), 64 binary walkers 44.5 -> 24.1 ms.
#pragma once

#include "ce_patches.h"
#include "ce_wl.h"

namespace cemc {

// Dynamic LDS: padded occupation | tracker (canonical, when held in LDS) |
// patch tables | weights of the members by offset (canonical, near_cells x slots).
struct PatchLayout {
  uint32_t trk, tab, near, total;
};
__host__ __device__ inline PatchLayout patch_layout(int occ_bytes, int trk_sites, int tab_doubles, int near_bytes) {
  PatchLayout L;
  L.trk = align16(uint32_t(occ_bytes));
  L.tab = L.trk + align16(uint32_t(trk_sites) * 2u);
  L.near = L.tab + uint32_t(tab_doubles) * 8u;
  L.total = L.near + align16(uint32_t(near_bytes));
  return L;
}
// One bin of a walker in LDS, after the chain's layout.
struct __align__(16) PatchBin {
  double lg;
  uint32_t hist, known;
};
constexpr int kNearCells = 126;  // offsets within a halo of 2, and one for "none"

namespace {

template <int kCtrl, int kRows>
__device__ __attribute__((always_inline)) inline double dpp_or0_f64(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, int(lo_of(v)), kCtrl, kRows, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, int(hi_of(v)), kCtrl, kRows, 0xF, true);
  return join_f64(uint32_t(lo), uint32_t(hi));
}

// Inclusive prefix sum over the 64 lanes.
__device__ __attribute__((always_inline)) inline double wave_scan_f64(double v) {
  v += dpp_or0_f64<0x111, 0xF>(v);  // row_shr 1, 2, 4, 8
  v += dpp_or0_f64<0x112, 0xF>(v);
  v += dpp_or0_f64<0x114, 0xF>(v);
  v += dpp_or0_f64<0x118, 0xF>(v);
  v += dpp_or0_f64<0x142, 0xA>(v);  // the last lane of rows 0 and 2 into rows 1 and 3
  v += dpp_or0_f64<0x143, 0xC>(v);  // lane 31 into rows 2 and 3
  return v;
}

// n / d for n, d < 2^16 by one multiplication: inv = ceil(2^32 / d) is at most
// d / 2^32 too large, so the quotient is exact.
__device__ __attribute__((always_inline)) inline uint32_t div16(uint32_t n, uint32_t inv) { return __umulhi(n, inv); }

// Sum over the kG lanes of a group (4: a quad, 16: a row, 64: the wave);
// every lane of the group ends with it.
template <int kG>
__device__ __attribute__((always_inline)) inline double group_lanes_sum_f64(double v) {
  if constexpr (kG == 4) {
    v += dpp_f64<0xB1>(v);
    v += dpp_f64<0x4E>(v);
    return v;
  } else if constexpr (kG == 8) {
    return octet_sum_f64(v);
  } else if constexpr (kG == 16) {
    v += dpp_f64<0x128>(v);
    return octet_sum_f64(v);
  } else {
    return wave_sum_f64(v);
  }
}

}  // namespace

// A rejected move in the block's list of energy changes: a NaN that no
// accepted change can be (its comparison with the threshold fails).
constexpr long long kRejected = 0x7FF8DEAD00000000ll;

// kBM: basis functions, one less than the species (1, 2, 3).  kP: moves that
// a lane group evaluates per round.  kTrkLds: the tracker is held in LDS,
// else in HBM, where only its lookups per block and its commits touch it.
//
// kWL: Wang-Landau walkers with a histogram of their own and no adaptive
// windows (WangLandauSampler::step, wang_landau_sampler.cpp:232-317) on
// rounds of eight: ln g and the counts stay in LDS, and the round's energy
// changes are decided one after the other on them, up to the first move that
// an accepted one reaches.
struct PatchArgs {
  const ChainParams* params;
  ChainState* states;
  const ModelDev* models;
  int8_t* occ_pool;
  uint16_t* trk_pool;
  const int32_t* chain_order;
  const int64_t* n_moves;
  uint32_t* accept_log;
  int64_t log_words;
  int64_t time_limit;
  // walkers
  WLDev* walkers;
  double* logdos_pool;
  uint32_t* hist_pool;
  uint8_t* known_pool;
  int64_t n_checks, check_every;
  // constraints and bias
  HookDev* hooks;
  // per chain the energy changes of a block that its last launch did not end
  // (64, kRejected: none), valid as ChainState says
  double* tails;
};

// kHook: chains with constraints or a bias whose constraints depend on the
// proposal alone: sites that may hold any species or are fixed, fixed species
// of canonical chains, no pair constraint, no waste recycling.  Fixed sites
// keep their tracker slots, so which of a move's proposals is the first valid
// one is known before the block starts.  A bias on a flip's species count
// makes the round's moves depend on each other through the count: they are
// decided one after the other, with the bias at the counts a block can reach
// held across the lanes.  (16 binary SGC chains of 8^3 sites, a tenth of them
// fixed, biased: 15.3 -> 3.8 ms for 10240 moves each, against the one-move
// kernel.)
template <bool kCanonical, int kBM, int kG, int kR, int kW, int kP, bool kTrkLds, bool kWL = false, bool kHook = false>
__global__ __launch_bounds__(64 * kW) void patch_kernel(PatchArgs args) {
  const ChainParams* __restrict__ params = args.params;
  ChainState* __restrict__ states = args.states;
  const ModelDev* __restrict__ models = args.models;
  int8_t* __restrict__ occ_pool = args.occ_pool;
  uint16_t* __restrict__ trk_pool = args.trk_pool;
  const int32_t* __restrict__ chain_order = args.chain_order;
  uint32_t* __restrict__ accept_log = args.accept_log;
  const int64_t log_words = args.log_words, time_limit = args.time_limit;
  static_assert(kG == 4 || kG == 8 || kG == 16 || kG == 64, "lanes per move");
  static_assert(!(kWL || kHook) || (kW == 1 && kTrkLds), "walkers and chains with hooks are one wave");
  constexpr int kS = kBM + 1;
  constexpr int kQ = kBM == 1 ? 6 : (kBM == 2 ? 5 : 4);  // members per patch (patch_members)
  constexpr int kPer = 64 / kG;                           // moves a wave evaluates side by side
  constexpr int kK = kW * kP * kPer;                       // moves per round
  static_assert(kK == (kG == 64 || kG == 8 ? 8 : 16), "rounds of 16, or of 8 with eight lanes or a wave per move");
  constexpr bool kNear = kCanonical && kG != 64;  // member weights by offset in LDS
  constexpr int kSlots = kG * kR;
  constexpr int kThreads = 64 * kW;
  extern __shared__ __align__(16) unsigned char lds[];
  __shared__ double dphi_tab[kS * kS * kBM];  // [(old*S+new)*B + d]
  __shared__ double dsingle_tab[kS * kS];
  __shared__ double phi_tab[kBM * kS];
  // the round's moves, one copy per wave (no barrier between filling and
  // reading them)
  __shared__ uint4 slot_a[kW][kK];  // canonical: p_i, p_j, place of i seen from j, a | b << 8 | lane << 16
                                    // SGC: p, cell, image, species offset | lane << 16
  __shared__ uint4 slot_b[kW][kCanonical ? kK : 1];  // canonical: cell_i, cell_j, image_i, image_j
  __shared__ uint2 slot_s[kW][kCanonical ? kK : 1];  // canonical: site_i | site_j << 16, tracker slots alike
  __shared__ double2 slot_t[kW][kK];                 // accept below, reject above
  __shared__ double red[2][kK];                      // sums of the round's moves, by parity
  __shared__ uint64_t conf_l[2];                     // rounds of 16 on several waves: the pair bits
  __shared__ double de_l[64];                        // the block's accepted energy changes (kRejected: none)
  __shared__ uint32_t on_l[kCanonical ? 1 : 64];     // SGC: species change of each, old | new << 8
  __shared__ uint8_t axis_tab[3][256];               // pair test, see pair_hits
  __shared__ uint8_t mask_tab[608];
  __shared__ int stop_flag[2];
  const int chain = chain_order[blockIdx.x];
  const int tid = int(threadIdx.x);
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const ChainParams* __restrict__ pp = params + chain;
  const ModelDev& m = models[pp->model];
  const int N = pp->n_sites;

  SweepCtx c;
  c.S = kS;
  c.B = kBM;
  c.N = N;
  c.L1 = m.dims[0];
  c.L2 = m.dims[1];
  c.L3 = m.dims[2];
  c.L23 = c.L2 * c.L3;
  c.h = m.pad_h;
  c.P2 = m.pdims[1];
  c.P3 = m.pdims[2];
  c.mag23 = 0xFFFFFFFFu / uint32_t(c.L23);
  c.mag3 = 0xFFFFFFFFu / uint32_t(c.L3);
  c.DX = c.L1 * c.P2 * c.P3;
  c.DY = c.L2 * c.P3;
  c.DZ = c.L3;
  c.K = 0;
  c.trans = nullptr;
  c.trans_in_lds = false;
  c.trans_l = nullptr;
  const uint64_t im0 = m.imask[0], im1 = m.imask[1];
  const int occ_bytes = m.pdims[0] * c.P2 * c.P3;
  const PatchLayout L =
      patch_layout(occ_bytes, kCanonical && kTrkLds ? N : 0, m.ptab_size, kNear ? kNearCells * kSlots : 0);
  uint8_t* occ = reinterpret_cast<uint8_t*>(lds);
  double* tab = reinterpret_cast<double*>(lds + L.tab);
  [[maybe_unused]] uint8_t* near_w = lds + L.near;
  uint16_t* gtrk = trk_pool + pp->trk_off;
  uint16_t* trk = kTrkLds ? reinterpret_cast<uint16_t*>(lds + L.trk) : gtrk;

  // ---- stage the lattice, the tracker and the tables
  const uint8_t* gocc = reinterpret_cast<const uint8_t*>(occ_pool + pp->occ_off);
  {
    const uint32_t p23 = uint32_t(c.P2 * c.P3), mag_p23 = 0xFFFFFFFFu / p23, mag_p3 = 0xFFFFFFFFu / uint32_t(c.P3);
    for (int p = tid; p < occ_bytes; p += kThreads) {
      const uint32_t px = fast_div(uint32_t(p), p23, mag_p23);
      const uint32_t rem = uint32_t(p) - px * p23;
      const uint32_t py = fast_div(rem, uint32_t(c.P3), mag_p3);
      int x = int(px) - c.h, y = int(py) - c.h, z = int(rem - py * uint32_t(c.P3)) - c.h;
      x += x < 0 ? c.L1 : 0;
      x -= x >= c.L1 ? c.L1 : 0;
      y += y < 0 ? c.L2 : 0;
      y -= y >= c.L2 ? c.L2 : 0;
      z += z < 0 ? c.L3 : 0;
      z -= z >= c.L3 ? c.L3 : 0;
      occ[p] = gocc[(x * c.L2 + y) * c.L3 + z];
    }
  }
  if constexpr (kCanonical && kTrkLds)
    for (int i = tid; i < N; i += kThreads) trk[i] = gtrk[i];
  for (int i = tid; i < m.ptab_size; i += kThreads) tab[i] = m.ptab[i];
  for (int i = tid; i < kBM * kS; i += kThreads) phi_tab[i] = m.basis[i];
  for (int i = tid; i < kS * kS; i += kThreads) {
    const int o = i / kS, nw = i - o * kS;
    double ds = 0.0;
    for (int d = 0; d < kBM; ++d) {
      const double dp = m.basis[d * kS + nw] - m.basis[d * kS + o];
      dphi_tab[i * kBM + d] = dp;
      ds += pp->j1[d] * dp;
    }
    dsingle_tab[i] = ds;
  }
  // pair test: a change at cell a reaches a flip at cell b when a - b, wrapped,
  // is an offset of the model's interaction mask.  With cells packed a byte
  // per axis, a + L - b has the axes' differences in its bytes (L <= 127); each
  // axis' table gives its share of the mask index, or 200 outside the halo,
  // and the mask table ends in zeros.
  {
    const int w = 2 * c.h + 1;
    for (int i = tid; i < 3 * 256; i += kThreads) {
      const int ax = i >> 8, Ld = ax == 0 ? c.L1 : (ax == 1 ? c.L2 : c.L3);
      int e = (i & 255) - Ld + c.h;
      e += e < 0 ? Ld : 0;
      e -= e >= Ld ? Ld : 0;
      axis_tab[ax][i & 255] = uint8_t(e >= 0 && e < w ? e * (ax == 0 ? w * w : (ax == 1 ? w : 1)) : 200);
    }
    for (int i = tid; i < 608; i += kThreads)
      mask_tab[i] = i < 128 ? uint8_t(((i < 64 ? im0 : im1) >> (i & 63)) & 1u) : 0;
  }
  if constexpr (kNear)
    for (int i = tid; i < kNearCells * kSlots; i += kThreads) near_w[i] = 0;
  // slots that a round does not fill hold a move from before (its sites are
  // read, slot_swap takes its species as unchanged); at first the cell (0, 0, 0)
  if (lane < kK) {
    const uint32_t p0 = uint32_t((c.h * c.P2 + c.h) * c.P3 + c.h);
    slot_a[wave][lane] = kCanonical ? uint4{p0, p0, uint32_t(kNearCells - 1), 0} : uint4{p0, 0, p0, 0};
    if constexpr (kCanonical) {
      slot_b[wave][lane] = uint4{0, 0, p0, p0};
      slot_s[wave][lane] = uint2{0, 0};
    }
    slot_t[wave][lane] = double2{0.0, 0.0};
  }
  // this lane's patches (past the last: table 0, all zeros)
  int mo[kR][kQ], base[kR], wl[kR];
  {
    const int sub = lane & (kG - 1);
#pragma unroll
    for (int k = 0; k < kR; ++k) {
      const int it = sub + kG * k;
      const bool on = it < m.n_patch;
      const PatchRec* pr = m.patches + (on ? it : 0);
#pragma unroll
      for (int q = 0; q < kQ; ++q) mo[k][q] = on ? pr->m[q] : 0;
      base[k] = on ? int(pr->base) : 0;
      wl[k] = on ? int(pr->w_last) : 0;
    }
  }
  __syncthreads();
  if constexpr (kNear) {
    // a swap's second flip sees its first site changed: the index weight of
    // the member at each offset, per patch slot
    const int w = 2 * c.h + 1, shift = (c.h * c.P2 + c.h) * c.P3 + c.h;
    for (int i = tid; i < m.n_patch * kQ; i += kThreads) {
      const int it = i / kQ, q = i - it * kQ, off = m.patches[it].m[q];
      if (off == 0) continue;  // an unused place
      int weight = q == kQ - 1 ? int(m.patches[it].w_last) : 1;
      for (int t = 0; q != kQ - 1 && t < q; ++t) weight *= kS;
      const int lin = off + shift, x = lin / (c.P2 * c.P3), rem = lin - x * c.P2 * c.P3, y = rem / c.P3, z = rem - y * c.P3;
      near_w[((x * w + y) * w + z) * kSlots + it] = uint8_t(weight);
    }
    __syncthreads();
  }
  const double dphi01 = dphi_tab[kBM], dphi10 = dphi_tab[kS * kBM];  // two species: 0 -> 1 and 1 -> 0
  [[maybe_unused]] const double dsin01 = dsingle_tab[1], dsin10 = dsingle_tab[kS];

  double energy = states[chain].energy;
  const uint64_t t0 = states[chain].moves_done;
  const double e_ref = states[chain].e_ref;
  // ---- the walker: its bins follow the chain's layout in LDS, 16 bytes each,
  // so that a move reads one and writes one
  [[maybe_unused]] WLDev* __restrict__ wk = kWL ? args.walkers + chain : nullptr;
  const int nb = kWL ? wk->n_bins : 0;
  [[maybe_unused]] PatchBin* bins = reinterpret_cast<PatchBin*>(lds + L.total);
  [[maybe_unused]] double e_min = 0.0, span = 1.0, nbd = 1.0, wl_f = 0.0, bins_per_ev = 0.0;
  [[maybe_unused]] int cur = 0, first = 0;
  [[maybe_unused]] PatchBin at_cur{0.0, 0, 0};  // the current bin
  [[maybe_unused]] uint64_t n_out = 0, n_self = 0;
  if constexpr (kWL) {
    const int64_t boff = wk->bin_off;
    for (int i = lane; i < nb; i += 64) {
      bins[i] = PatchBin{args.logdos_pool[boff + i], args.hist_pool[boff + i], args.known_pool[boff + i]};
    }
    __syncthreads();
    e_min = wk->e_min;
    span = wk->e_max - e_min;
    nbd = double(nb);
    bins_per_ev = nbd / span;
    wl_f = wk->f;
    cur = wk->cur_bin;
    first = wk->is_first;
    at_cur = bins[cur];  // the host checks 0 <= cur < nb
  }
  if (!kWL && wave == 0) {
    // A launch that starts inside a block takes over the changes that earlier
    // launches made with the block's moves before it, and the energy at the
    // block's start.  (Where the state was changed meanwhile: no change, and
    // the energy as it is.)
    const int k0 = int(t0 & 63u);
    const ChainState& st = states[chain];
    const bool carried =
        k0 != 0 && st.blk_moves == t0 && __double_as_longlong(st.blk_end) == __double_as_longlong(energy);
    if (carried) energy = st.blk_energy;
    de_l[lane] = carried && lane < k0 ? args.tails[int64_t(chain) * 64 + lane] : __longlong_as_double(kRejected);
    if constexpr (!kCanonical) on_l[lane] = 0;
  }
  uint64_t n_acc = 0;
  double sum_de = 0.0, sum_de2 = 0.0;  // this lane's moves
  const double inv_n = 1.0 / double(N);
  double sing[kBM], sum_s[kBM], sum_s2[kBM], sum_se[kBM];
#pragma unroll
  for (int d = 0; d < kBM; ++d) sing[d] = sum_s[d] = sum_s2[d] = sum_se[d] = 0.0;
  if constexpr (!kCanonical && !kWL) {
    // every wave sums alike, so the singlets do not depend on kW
    double part[kBM];
#pragma unroll
    for (int d = 0; d < kBM; ++d) part[d] = 0.0;
    for (int i = lane; i < N; i += 64) {
      const int s = occ[ref_of<true>(c, i).p];
#pragma unroll
      for (int d = 0; d < kBM; ++d) part[d] += phi_tab[d * kS + s];
    }
#pragma unroll
    for (int d = 0; d < kBM; ++d) sing[d] = wave_sum_f64(part[d]) / double(N);
  }
  const double kT = pp->kT;
  const uint64_t seed = pp->seed, uid = pp->uid;
  const uint32_t np = uint32_t(pp->n_present);
  const uint32_t present_pk = pp->present_pk;
  const uint64_t cnt_lo = pp->count_pk[0], cnt_hi = pp->count_pk[1];
  const uint64_t seg_lo = pp->segoff_pk[0], seg_hi = pp->segoff_pk[1];
  uint32_t* acc_log = accept_log ? accept_log + int64_t(chain) * log_words : nullptr;
  const uint64_t t_begin = time_limit > 0 ? uint64_t(wall_clock64()) : 0u;

  // LDS written by this wave is read by it in program order; other waves are
  // ordered by barriers
  auto own_order = [] { __atomic_signal_fence(__ATOMIC_SEQ_CST); };

  // One flip over this lane's patches, in phases so that the loads of a
  // round go out together: member species, table indexes, entries, sum (two
  // species: plain, else the change for dphi).
  const int sub = lane & (kG - 1);
  typedef uint32_t Members[kR][kQ];
  typedef double Entries[kR][kBM];
  auto gather = [&](int p, Members& s) {
#pragma unroll
    for (int k = 0; k < kR; ++k)
#pragma unroll
      for (int q = 0; q < kQ; ++q) s[k][q] = occ[p + mo[k][q]];
  };
  auto index = [&](const Members& s, int (&idx)[kR]) {
#pragma unroll
    for (int k = 0; k < kR; ++k) {
      uint32_t v = s[k][kQ - 2];
#pragma unroll
      for (int q = kQ - 3; q >= 0; --q) v = v * uint32_t(kS) + s[k][q];
      idx[k] = int(v + __umul24(s[k][kQ - 1], uint32_t(wl[k])));
    }
  };
  // The member at padded offset `lin` holds a species `ds` higher than the
  // lattice says (lin 0: no member).
  auto index_shift = [&](int lin, int ds, int (&idx)[kR]) {
#pragma unroll
    for (int k = 0; k < kR; ++k) {
      int w = mo[k][kQ - 1] == lin ? wl[k] : 0, pw = 1;
#pragma unroll
      for (int q = 0; q < kQ - 1; ++q) {
        w = mo[k][q] == lin ? pw : w;
        pw *= kS;
      }
      idx[k] += lin != 0 ? w * ds : 0;
    }
  };
  auto entries = [&](const int (&idx)[kR], Entries& g) {
#pragma unroll
    for (int k = 0; k < kR; ++k) {
      const double* t = tab + (base[k] + kBM * idx[k]);
      if constexpr (kBM == 2) {
        const dbl2_t two = load_pair(t);
        g[k][0] = two.x;
        g[k][kBM - 1] = two.y;
      } else {
#pragma unroll
        for (int d = 0; d < kBM; ++d) g[k][d] = t[d];
      }
    }
  };
  auto total = [&](const Entries& g, const double (&dphi)[kBM]) {
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < kR; ++k) {
      if constexpr (kBM == 1) {
        v = k == 0 ? g[0][0] : v + g[k][0];
      } else {
#pragma unroll
        for (int d = 0; d < kBM; ++d) v = k == 0 && d == 0 ? dphi[0] * g[0][0] : fma(dphi[d], g[k][d], v);
      }
    }
    return v;
  };
  // keeps the scheduler from moving a phase's loads behind the waits of the
  // phase before
  auto phase = [] { __builtin_amdgcn_sched_barrier(0); };

  const uint32_t bias = uint32_t(c.L1) | (uint32_t(c.L2) << 8) | (uint32_t(c.L3) << 16);
  struct Axes {
    uint32_t x, y, z;
  };
  auto axes = [&](uint32_t cell_a, uint32_t cell_b) {
    const uint32_t d = cell_a + bias - cell_b;
    return Axes{axis_tab[0][d & 255u], axis_tab[1][(d >> 8) & 255u], axis_tab[2][d >> 16]};
  };
  // padded offset of a cell of the halo box
  auto offset_of = [&](uint32_t cell) {
    const uint32_t w = uint32_t(2 * c.h + 1), x = cell / (w * w), r = cell - x * w * w, y = r / w, z = r - y * w;
    return ((int(x) - c.h) * c.P2 + int(y) - c.h) * c.P3 + int(z) - c.h;
  };
  const uint32_t inv23 = 0xFFFFFFFFu / uint32_t(c.L23) + 1u, inv3 = 0xFFFFFFFFu / uint32_t(c.L3) + 1u;
  // image `im` of the site with image word w: an image that does not exist
  // repeats another one, so every lane may write
  const int im = lane & 7;
  const int step_x = (im & 1) ? c.DX : 0, step_y = (im & 2) ? c.DY : 0, step_z = (im & 4) ? c.DZ : 0;
  auto image = [&](uint32_t w) {
    const int ex = int(w << 10) >> 30, ey = int(w << 8) >> 30, ez = int(w << 6) >> 30;
    return int(w & 0xFFFFFu) + __mul24(ex, step_x) + __mul24(ey, step_y) + __mul24(ez, step_z);
  };
  uint4* const my_a = slot_a[wave];
  uint4* const my_b = slot_b[wave];
  uint2* const my_s = slot_s[wave];
  double2* const my_t = slot_t[wave];
  const int kd = lane & (kK - 1);  // the slot this lane decides
  // the first slot it commits (four waves: sites i and j of four moves a wave)
  const int ck = kK == 8 || kW == 1 ? lane >> 3 : (kW == 2 ? 8 * wave + (lane >> 3) : 4 * wave + (lane >> 4));
  // Pairs (a, b), a < b, of the round that a lane tests.  Rounds of 8: one
  // byte per b.  Rounds of 16: two words of four 16-bit rows; row r = 1..8
  // holds b = r (r pairs), then b = 16 - r (16 - r pairs).
  int pair_a[2], pair_b[2], conf_word = 0, conf_shift = 0;
  uint32_t conf_mask = (1u << kd) - 1u;
  if constexpr (kK == 8) {
    pair_a[0] = pair_a[1] = lane & 7;
    pair_b[0] = pair_b[1] = lane >> 3;
  } else {
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      const int r = 4 * (kW > 1 ? (wave & 1) : v) + (lane >> 4) + 1, j = lane & 15;
      pair_b[v] = j < r ? r : 16 - r;
      pair_a[v] = j < r ? j : j - r;
    }
    const int r = kd <= 8 ? (kd > 0 ? kd : 1) : 16 - kd;
    conf_word = (r - 1) >> 2;
    conf_shift = 16 * ((r - 1) & 3) + (kd <= 8 ? 0 : r);
  }
  // two packed tracker slots each: not zero when some slot is in both
  // (a zero half of v borrows into its own top bit of (v - 1) & ~v)
  auto shared_half = [](uint32_t s, uint32_t t) {
    const uint32_t x = s ^ t, y = s ^ __builtin_rotateright32(t, 16);
    return (((x - 0x00010001u) & ~x) | ((y - 0x00010001u) & ~y)) & 0x80008000u;
  };

  // ---- constraints and bias
  [[maybe_unused]] HookDev* hk = kHook ? args.hooks + chain : nullptr;
  [[maybe_unused]] const uint8_t* allowed = nullptr;
  [[maybe_unused]] const double* bias_tab = nullptr;
  [[maybe_unused]] uint32_t fixed = 0;
  [[maybe_unused]] int attempts = 1, bias_sp = -1, bias_cnt = 0, bias_at = 0;
  [[maybe_unused]] double bias_energy = 0.0, bias_lo = 0.0, bias_hi = 0.0, bias_top = 0.0;
  [[maybe_unused]] bool failed = false;
  if constexpr (kHook) {
    allowed = hk->allowed;
    fixed = hk->fixed_species;
    attempts = hk->max_attempts;
    bias_sp = hk->bias_species;
    bias_cnt = hk->bias_count;
    bias_tab = hk->bias_tab;
    bias_energy = hk->bias_energy;
  }

  uint32_t rnd = 0;
  // One block: moves t_blk .. t_blk + n_in - 1 of the stream, n_in <= 64, from
  // the launch's first move on; move t_blk has bit `log_at` of the chain's log
  // (below 0: -log_at moves come before the launch).  Returns n_in, or less:
  // the first move that has no valid proposal.
  auto make_block = [&](uint64_t t_blk, const int n_all, int64_t log_at) {
    int n_in = n_all;
    const int lo = log_at < 0 ? -int(log_at) : 0;
    // lane l decodes move t_blk + l
    Philox4 blk = philox4x64_10(t_blk + uint64_t(lane), 0, 0, 0, seed, uid);
    // canonical: species a and b of a block's move, its tracker slots
    auto swap_of = [&](const Philox4& w, uint32_t& a, uint32_t& b, int& ta, int& tb) {
      const uint32_t ia = bounded32(uint32_t(w.w0 >> 32), np);
      uint32_t ib = ia + 1u + bounded32(uint32_t(w.w0), np - 1u);
      ib -= ib >= np ? np : 0u;
      a = (present_pk >> (4u * ia)) & 15u;
      b = (present_pk >> (4u * ib)) & 15u;
      ta = unpack16(seg_lo, seg_hi, ia) + int(bounded64(w.w1, uint64_t(unpack16(cnt_lo, cnt_hi, ia))));
      tb = unpack16(seg_lo, seg_hi, ib) + int(bounded64(w.w2, uint64_t(unpack16(cnt_lo, cnt_hi, ib))));
    };
    if constexpr (kHook) {
      // proposal k of move t uses Philox counter (t, k, 0, 0); the first valid
      // one is made, and with `attempts` of them invalid the chain stops there
      // (montecarlo.py:970-991)
      if (!kCanonical && bias_sp >= 0) {
        bias_at = bias_cnt;
        auto at = [&](int n) { return bias_tab[n < 0 ? 0 : (n > N ? N : n)]; };
        bias_lo = at(bias_at - 64 + lane);
        bias_hi = at(bias_at + lane);
        bias_top = at(bias_at + 64);
      }
      bool ok = lane < lo || lane >= n_in;
      for (int k = 0;;) {
        if (!ok) {
          if constexpr (kCanonical) {
            uint32_t a, b;
            int ta, tb;
            swap_of(blk, a, b, ta, tb);
            ok = (((fixed >> a) | (fixed >> b)) & 1u) == 0u &&
                 (allowed == nullptr || (allowed[trk[ta]] != 0 && allowed[trk[tb]] != 0));
          } else {
            ok = allowed == nullptr || allowed[int(bounded64(blk.w1, uint64_t(N)))] != 0;
          }
        }
        if (__builtin_amdgcn_ballot_w64(!ok) == 0 || ++k >= attempts) break;
        if (!ok) blk = philox4x64_10(t_blk + uint64_t(lane), uint64_t(k), 0, 0, seed, uid);
      }
      const uint64_t bad = __builtin_amdgcn_ballot_w64(!ok);
      if (bad != 0) {
        failed = true;
        n_in = int(__builtin_ctzll(bad));
      }
    }
    // Metropolis test of the reference (montecarlo.py:950-956): accept when
    // dE < 0 or u <= exp(-dE / kT).  dE against -kT log u decides it outside a
    // margin far above the rounding of log and exp; inside, exp is evaluated.
    // (Walkers: log u itself.)
    const double log_u = log(unit_double(blk.w3));
    const double t_u = -kT * log_u, margin = 2e-12 * (kT + t_u);
    const double2 thr = kWL ? double2{log_u, 0.0} : double2{t_u - margin, t_u + margin};
    uint4 v_a{0, 0, 0, 0}, v_b{0, 0, 0, 0};
    uint2 v_s{0, 0};
    // padded index, packed cell and image word of a site
    auto place = [&](uint32_t site, uint32_t& p, uint32_t& cell, uint32_t& img) {
      const uint32_t x = div16(site, inv23), r = site - __umul24(x, uint32_t(c.L23));
      const uint32_t y = div16(r, inv3), z = r - __umul24(y, uint32_t(c.L3));
      p = __umul24(__umul24(x + c.h, uint32_t(c.P2)) + y + c.h, uint32_t(c.P3)) + z + c.h;
      cell = x | (y << 8) | (z << 16);
      Ref ref;
      ref.p = int(p);
      ref.x = int(x);
      ref.y = int(y);
      ref.z = int(z);
      img = image_word<true>(c, ref);
    };
    // canonical: the sites in the move's tracker slots
    auto set_sites = [&](uint32_t si, uint32_t sj) {
      place(si, v_a.x, v_b.x, v_b.z);
      place(sj, v_a.y, v_b.y, v_b.w);
      v_s.x = si | (sj << 16);
      const Axes at = axes(v_b.x, v_b.y);
      const uint32_t cell = at.x + at.y + at.z;  // of i in the halo box around j; 125 and more: outside
      v_a.z = kNear ? (cell < uint32_t(kNearCells - 1) ? cell : uint32_t(kNearCells - 1))
                    : (cell < uint32_t(kNearCells - 1) ? uint32_t(offset_of(cell)) : 0u);
    };
    if constexpr (kCanonical) {
      uint32_t a, b;
      int ta, tb;
      swap_of(blk, a, b, ta, tb);
      v_a.w = a | (b << 8) | (uint32_t(lane) << 16);
      v_s.y = uint32_t(ta) | (uint32_t(tb) << 16);
      set_sites(trk[ta], trk[tb]);
    } else {
      const Ref r = ref_of<true>(c, int(bounded64(blk.w1, uint64_t(N))));
      v_a = uint4{uint32_t(r.p), uint32_t(r.x) | (uint32_t(r.y) << 8) | (uint32_t(r.z) << 16), image_word<true>(c, r),
                  bounded32(uint32_t(blk.w0), uint32_t(kS - 1)) | (uint32_t(lane) << 16)};
    }
    auto first_to_last = [&] { return (n_in < 64 ? (uint64_t(1) << n_in) - 1u : ~uint64_t(0)) & (~uint64_t(0) << lo); };
    uint64_t open = first_to_last();  // moves not made yet
    while (open != 0) {
      // ---- the first kK open moves fill the slots
      const int rank = int(__builtin_amdgcn_mbcnt_hi(uint32_t(open >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(open), 0)));
      const bool in = ((open >> lane) & 1u) != 0 && rank < kK;
      const int n_open = int(__builtin_popcountll(open));
      const int n = n_open < kK ? n_open : kK;
      if (in) {
        my_a[rank] = v_a;
        my_t[rank] = thr;
        if constexpr (kCanonical) {
          my_b[rank] = v_b;
          my_s[rank] = v_s;
        }
      }
      // canonical: the tracker slots of the round's moves may have got other
      // sites since they were read
      uint32_t now_i = 0, now_j = 0;
      if constexpr (kCanonical) {
        now_i = trk[v_s.y & 0xFFFFu];
        now_j = trk[v_s.y >> 16];
      }
      own_order();
      // ---- the slots: what this lane evaluates, tests, commits and decides
      constexpr int kPairs = kK == 16 && kW == 1 ? 2 : 1;
      constexpr int kCom = kK == 16 && kW == 1 ? 2 : 1;
      uint4 ev[kP];
      uint2 pa[kPairs], pb[kPairs];  // cells (canonical: i, j)
      uint32_t sa[kPairs], sb[kPairs];
      uint4 ca[kCom];
      uint2 cimg[kCom], cs[kCom];
#pragma unroll
      for (int t = 0; t < kP; ++t) {
        const int slot = (wave * kP + t) * kPer + (kG == 64 ? 0 : lane / kG);
        ev[t] = my_a[slot];
        if constexpr (kCanonical) ev[t].w = slot_swap(ev[t].w, slot, n);
      }
#pragma unroll
      for (int v = 0; v < kPairs; ++v) {
        if constexpr (kCanonical) {
          pa[v] = *reinterpret_cast<const uint2*>(&my_b[pair_a[v]]);
          pb[v] = *reinterpret_cast<const uint2*>(&my_b[pair_b[v]]);
          sa[v] = my_s[pair_a[v]].y;
          sb[v] = my_s[pair_b[v]].y;
        } else {
          pa[v].x = my_a[pair_a[v]].y;
          pb[v].x = my_a[pair_b[v]].y;
        }
      }
#pragma unroll
      for (int v = 0; v < kCom; ++v) {
        ca[v] = my_a[ck + 8 * v];
        if constexpr (kCanonical) {
          cimg[v] = reinterpret_cast<const uint2*>(&my_b[ck + 8 * v])[1];
          cs[v] = my_s[ck + 8 * v];
        }
      }
      const uint4 da = my_a[kd];
      const double2 dt = my_t[kd];
      if constexpr (kCanonical) {
        const bool stale = in && (now_i | (now_j << 16)) != v_s.x;
        if (__builtin_amdgcn_ballot_w64(stale) != 0) {
          set_sites(now_i, now_j);
          continue;  // nothing was done yet: fill the slots again
        }
      }
      phase();
      // ---- members of this wave's moves; cell differences of the pairs
      double part[kP];
      // flips whose loads go out together: all of this wave's, or one after the
      // other where their members and entries would overflow the registers
      constexpr int kF = kCanonical ? 2 : 1;  // flips per move
      constexpr int kFlips = kP * kF;
      constexpr int kAtOnce = kFlips * kR * kQ <= 100 ? kFlips : 1;
      Axes ax[kPairs][kCanonical ? 4 : 1];
      uint32_t c_o[kCom], d_s = 0;
      auto other_loads = [&] {
#pragma unroll
        for (int v = 0; v < kPairs; ++v) {
          ax[v][0] = axes(pa[v].x, pb[v].x);
          if constexpr (kCanonical) {
            ax[v][1] = axes(pa[v].x, pb[v].y);
            ax[v][2] = axes(pa[v].y, pb[v].x);
            ax[v][3] = axes(pa[v].y, pb[v].y);
          }
        }
        if constexpr (!kCanonical) {
#pragma unroll
          for (int v = 0; v < kCom; ++v) c_o[v] = occ[ca[v].x];
          d_s = occ[da.x];
        }
      };
      uint32_t hit[kPairs];
      auto other_masks = [&] {
#pragma unroll
        for (int v = 0; v < kPairs; ++v) {
          hit[v] = 0;
#pragma unroll
          for (int u = 0; u < (kCanonical ? 4 : 1); ++u) hit[v] |= mask_tab[ax[v][u].x + ax[v][u].y + ax[v][u].z];
        }
      };
#pragma unroll
      for (int f0 = 0; f0 < kFlips; f0 += kAtOnce) {
        Members mem[kAtOnce];
        uint32_t near[kAtOnce][kNear ? kR : 1];
        uint32_t own[kAtOnce];
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
          const uint4 e = ev[(f0 + u) / kF];
          const bool second = kCanonical && (f0 + u) % 2 == 1;  // site j of a swap
          if constexpr (!kCanonical && kBM > 1) own[u] = occ[e.x];
          gather(int(second ? e.y : e.x), mem[u]);
          if (kNear && second)
#pragma unroll
            for (int k = 0; k < kR; ++k) near[u][kNear ? k : 0] = near_w[__umul24(e.z, uint32_t(kSlots)) + sub + kG * k];
        }
        if (f0 == 0) other_loads();
        phase();
        Entries g[kAtOnce];
        double dphi[kAtOnce][kBM];
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
          const uint4 e = ev[(f0 + u) / kF];
          const bool second = kCanonical && (f0 + u) % 2 == 1;
          int idx[kR];
          index(mem[u], idx);
          int o = int(e.w & 255u), nw = int((e.w >> 8) & 255u);
          if (second) {
            // the swap's second flip sees site i already changed (ce_updater.cpp:845-852)
            if constexpr (kNear) {
#pragma unroll
              for (int k = 0; k < kR; ++k) idx[k] += __mul24(int(near[u][k]), nw - o);
            } else if (e.z != 0u) {
              index_shift(int(e.z), nw - o, idx);
            }
          }
          entries(idx, g[u]);
          if constexpr (kBM > 1) {
            if constexpr (!kCanonical) {
              nw = int(own[u]) + 1 + o;
              o = int(own[u]);
              nw -= nw >= kS ? kS : 0;
            }
#pragma unroll
            for (int d = 0; d < kBM; ++d) dphi[u][d] = dphi_tab[(o * kS + nw) * kBM + d];
          } else {
            dphi[u][0] = 0.0;
          }
        }
        if (f0 == 0) other_masks();
        phase();
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
          const double v = total(g[u], dphi[u]);
          const int t = (f0 + u) / kF;
          if (kCanonical && (f0 + u) % 2 == 1)
            part[t] -= v;
          else
            part[t] = v;
        }
      }
      // ---- which earlier moves of the round reach which
      uint64_t conf[2] = {0, 0};
#pragma unroll
      for (int v = 0; v < kPairs; ++v) {
        if constexpr (kCanonical) hit[v] |= shared_half(sa[v], sb[v]);
        conf[v] = __builtin_amdgcn_ballot_w64(hit[v] != 0);
      }
      if constexpr (kK == 16 && kW > 1)
        if (wave < 2 && lane == 0) conf_l[wave] = conf[0];
      // the slot this lane decides
      uint32_t d_o = da.w & 255u, d_n = (da.w >> 8) & 255u;
      if constexpr (!kCanonical) {
        d_n = d_s + 1u + d_o;
        d_o = d_s;
        d_n -= d_n >= uint32_t(kS) ? uint32_t(kS) : 0u;
      }
      // ---- sums of the round's moves
      double* rs = red[rnd & 1u];
#pragma unroll
      for (int t = 0; t < kP; ++t) {
        const double s = group_lanes_sum_f64<kG>(part[t]);
        if ((lane & (kG - 1)) == 0) rs[(wave * kP + t) * kPer + (kG == 64 ? 0 : lane / kG)] = s;
      }
      if constexpr (kW > 1)
        __syncthreads();
      else
        own_order();
      // ---- decide: lane l slot l mod kK, so that a ballot repeats the round's verdicts
      const double tot = rs[kd];
      // earlier moves of the round that reach the slot's
      uint32_t conf_d;
      if constexpr (kK == 8) {
        conf_d = uint32_t(conf[0] >> (8 * kd)) & conf_mask;
      } else {
        const uint64_t word = kW > 1 ? conf_l[conf_word] : (conf_word ? conf[1] : conf[0]);
        conf_d = uint32_t(word >> conf_shift) & conf_mask;
      }
      double dE;
      if constexpr (kBM == 1) {
        const double d0 = d_o == 0 ? dphi01 : dphi10;
        dE = kCanonical ? __dmul_rn(d0, tot) : fma(d0, tot, d_o == 0 ? dsin01 : dsin10);
      } else {
        dE = kCanonical ? tot : tot + dsingle_tab[int(d_o) * kS + int(d_n)];
      }
      uint32_t com = 0, blocked = 0;
      if constexpr (kWL) {
        // ---- slot after slot; every lane holds the walker's state
        auto any = [](bool x) { return __builtin_amdgcn_ballot_w64(x) != 0; };  // of a value all lanes share
        int k = 0;
        for (; k < n; ++k) {
          if ((uint32_t(__builtin_amdgcn_readlane(int(conf_d), k)) & com) != 0) break;
          const double e_new = energy + readlane_f64(dE, k);
          // Truncated bin (histogram.cpp:66-69) from a product; its rounding is
          // below 1e-8 inside any histogram that fits here, so only near an
          // edge the quotient itself is formed.  Clamped before the
          // conversion: far outside stays outside, and NaN lies below.
          const double q = fmin(fmax((e_new - e_min) * bins_per_ev, -1e9), 1e9);
          int raw = int(q - 1e-8);
          if (any(raw != int(q + 1e-8)))
            raw = int(fmin(fmax(trunc((e_new - e_min) * nbd / span), -2147483648.0), 2147483647.0));
          const int bin = __builtin_amdgcn_readfirstlane(raw);
          if (uint32_t(bin) >= uint32_t(nb)) {
            // undone; a walker that has been in range counts its current bin
            // once more when the proposal lies above the top bin
            // (wang_landau_sampler.cpp:251-260)
            ++n_out;
            if (first || bin <= nb) continue;
          } else {
            n_self += bin == cur ? 1u : 0u;
            // accept if u < g(cur) / g(bin), or on the first in-range proposal
            // (histogram.cpp:130-135); log u decides outside a margin far
            // above the rounding of log and exp
            const PatchBin at_bin = bins[bin];
            const double diff = at_cur.lg - at_bin.lg;
            const double over = diff - readlane_f64(dt.x, k);
            bool take = any(over > 1e-12);
            if (!take && (first || !any(over < -1e-12))) {
              const int src = int(uint32_t(__builtin_amdgcn_readlane(int(da.w), k)) >> 16);
              take = first || any(diff > 0.0 || unit_double(readlane_u64(blk.w3, src)) < exp(diff));
            }
            if (take) {
              com |= 1u << k;
              energy = e_new;
              cur = bin;
              at_cur = at_bin;
              first = 0;
            }
          }
          // Histogram::update (histogram.cpp:71-90); LDS operations of one
          // wave complete in order, so the next slot reads it
          at_cur.lg += wl_f;
          at_cur.hist += 1u;
          at_cur.known = 1u;
          if (lane == 0) bins[cur] = at_cur;
        }
        blocked = ((1u << kK) - 1u) & ~((1u << k) - 1u);  // this slot and the later ones stay open
        n_acc += uint64_t(__builtin_popcount(com));
      } else if (kHook && !kCanonical && bias_sp >= 0) {
        // ---- slot after slot: the bias of the proposed state joins its
        // energy (montecarlo.py:926-930)
        auto any = [](bool x) { return __builtin_amdgcn_ballot_w64(x) != 0; };  // of a value all lanes share
        auto bias_of = [&](int n) {  // n within 64 of bias_at
          const int i = n - bias_at;
          return i < 0 ? readlane_f64(bias_lo, i + 64) : (i < 64 ? readlane_f64(bias_hi, i) : bias_top);
        };
        const int up = int(d_n == uint32_t(bias_sp)) - int(d_o == uint32_t(bias_sp));
        double now = bias_of(bias_cnt);
        int k = 0;
        for (; k < n; ++k) {
          if ((uint32_t(__builtin_amdgcn_readlane(int(conf_d), k)) & com) != 0) break;
          const int dc = __builtin_amdgcn_readlane(up, k);
          const double next = dc == 0 ? now : bias_of(bias_cnt + dc);
          const double de = readlane_f64(dE, k) + (next - now);
          bool take = any(de < readlane_f64(dt.x, k));
          if (!take && !any(de > readlane_f64(dt.y, k))) {
            const int src = int(uint32_t(__builtin_amdgcn_readlane(int(da.w), k)) >> 16);
            take = any(de < 0.0 || unit_double(readlane_u64(blk.w3, src)) <= exp(-de / kT));
          }
          if (take) {
            com |= 1u << k;
            dE = kd == k ? de : dE;
            bias_cnt += dc;
            bias_energy = next;
            now = next;
          }
        }
        blocked = ((1u << kK) - 1u) & ~((1u << k) - 1u);  // this slot and the later ones stay open
      } else {
        const bool valid = kd < n;
        bool yes = dE < dt.x;
        if (__builtin_amdgcn_ballot_w64(valid && !yes && !(dE > dt.y)) != 0) {
          const double u = unit_double(__shfl(blk.w3, int(da.w >> 16), 64));
          if (!yes && !(dE > dt.y)) yes = dE < 0.0 || u <= exp(-dE / kT);
        }
        const uint32_t acc = uint32_t(__builtin_amdgcn_ballot_w64(valid && yes)) & ((1u << kK) - 1u);
        // A move that an accepted, or a blocked, earlier one reaches is blocked:
        // it stays open.  The others are made; they do not read what a blocked
        // one may change, nor it what they change, so their order does not
        // matter.
        for (uint32_t next = acc; next != 0;) {
          const uint32_t b = uint32_t(__builtin_amdgcn_ballot_w64(valid && (conf_d & (acc | blocked)) != 0)) & ((1u << kK) - 1u);
          next = b & ~blocked;
          blocked = b;
        }
        com = acc & ~blocked;
      }
      if (com != 0) {
#pragma unroll
        for (int v = 0; v < kCom; ++v) {
          if (((com >> (ck + 8 * v)) & 1u) == 0) continue;
          if constexpr (kCanonical) {
            const uint8_t o = uint8_t(ca[v].w), nw = uint8_t(ca[v].w >> 8);
            if constexpr (kK == 16 && kW == 4) {
              occ[image((lane & 8) ? cimg[v].y : cimg[v].x)] = (lane & 8) ? o : nw;
            } else {
              occ[image(cimg[v].x)] = nw;
              occ[image(cimg[v].y)] = o;
            }
            const int first = kK == 16 && kW == 4 ? lane & 15 : im;
            if (first < 2) trk[first ? cs[v].y >> 16 : cs[v].y & 0xFFFFu] = uint16_t(first ? cs[v].x : cs[v].x >> 16);
          } else {
            uint32_t nw = c_o[v] + 1u + (ca[v].w & 255u);
            nw -= nw >= uint32_t(kS) ? uint32_t(kS) : 0u;
            occ[image(ca[v].z)] = uint8_t(nw);
          }
        }
        if ((kW == 1 || wave == 0) && lane < kK && ((com >> kd) & 1u)) {
          if constexpr (kWL) {
            const int64_t at = log_at + int64_t(da.w >> 16);
            if (acc_log != nullptr && at < 32 * log_words) atomicOr(acc_log + (at >> 5), 1u << (at & 31));
          } else {
            de_l[da.w >> 16] = dE;
            if constexpr (!kCanonical) on_l[da.w >> 16] = d_o | (d_n << 8);
          }
        }
      }
      open &= ~__builtin_amdgcn_ballot_w64(in && ((blocked >> (rank & 31)) & 1u) == 0);
      ++rnd;
      if constexpr (kW > 1)
        __syncthreads();  // the commits before the next round's reads
      else
        own_order();
    }
    // ---- the block's energies and samples: lane l after its own move
    if (!kWL && (kW == 1 || wave == 0)) {
      const double de = de_l[lane];
      const bool made = __double_as_longlong(de) != kRejected;
      const uint64_t acc_bits = __builtin_amdgcn_ballot_w64(made) & first_to_last();
      n_acc += uint64_t(__builtin_popcountll(acc_bits));
      if (acc_log != nullptr && lane < 3) {
        const int64_t at = log_at + lo;
        const int sh = int(at & 31);
        const uint64_t bits = acc_bits >> lo;
        const uint32_t part = lane == 0 ? uint32_t(bits << sh)
                                        : (lane == 1 ? uint32_t(bits >> (32 - sh)) : (sh ? uint32_t(bits >> (64 - sh)) : 0u));
        if (part != 0) atomicOr(acc_log + (at >> 5) + lane, part);
      }
      if (n_in < 64) {
        // left to a launch that goes on here
        args.tails[int64_t(chain) * 64 + lane] = de;
        if (lane == 0) states[chain].blk_energy = energy;
      }
      const double e_l = energy + wave_scan_f64(made ? de : 0.0);
      const bool here = lane >= lo && lane < n_in;
      const double d = here ? e_l - e_ref : 0.0;
      sum_de += d;
      sum_de2 = fma(d, d, sum_de2);
      energy = readlane_f64(e_l, 63);
      if constexpr (!kCanonical) {
        const int o = int(on_l[lane] & 255u), nw = int(on_l[lane] >> 8);
#pragma unroll
        for (int b = 0; b < kBM; ++b) {
          const double ds = o == nw ? 0.0 : __dmul_rn(dphi_tab[(o * kS + nw) * kBM + b], inv_n);
          const double s_l = sing[b] + wave_scan_f64(ds);
          const double s = here ? s_l : 0.0;
          sum_s[b] += s;
          sum_s2[b] = fma(s, s, sum_s2[b]);
          sum_se[b] = fma(s, d, sum_se[b]);
          sing[b] = readlane_f64(s_l, 63);
        }
      }
      de_l[lane] = __longlong_as_double(kRejected);
      if constexpr (!kCanonical) on_l[lane] = 0;
      own_order();
    }
    return n_in;
  };

  int64_t moves_made = 0;
  [[maybe_unused]] int converged = 0;
  [[maybe_unused]] uint64_t n_flat = 0;
  if constexpr (kWL) {
    const double flat_c = wk->flatness, f_min = wk->f_min;
    converged = wk->converged;
    int64_t steps = wk->steps, since_flat = wk->since_flat, prev_conv = wk->prev_conv;
    int inv_active = wk->inv_active;
    double inv_factor = wk->inv_factor, bin_change = wk->bin_change;
    const bool inverse_time = wk->inverse_time != 0;
    for (int64_t chk = 0; chk < args.n_checks && !converged && wk->status == 0; ++chk) {
      for (int64_t blk0 = 0; blk0 < args.check_every; blk0 += 64) {
        const int n_in = int(args.check_every - blk0 < 64 ? args.check_every - blk0 : 64);
        make_block(t0 + uint64_t(moves_made), n_in, moves_made);
        moves_made += n_in;
      }
      steps += args.check_every;
      since_flat += args.check_every;
      __syncthreads();
      // Histogram::is_flat over the known bins (histogram.cpp:102-128); the
      // sum is an unsigned 32-bit integer and the minimum starts at 100000000
      uint32_t sum = 0u, cnt = 0u, mn = 100000000u;
      for (int i = lane; i < nb; i += 64) {
        const PatchBin at = bins[i];
        if (at.known) {
          sum += at.hist;
          cnt += 1u;
          mn = min(mn, at.hist);
        }
      }
      sum = wave_add_u32(sum);
      cnt = wave_add_u32(cnt);
      mn = wave_min_u32(mn);
      const double mean = double(sum) / double(cnt);
      if (__builtin_amdgcn_readfirstlane(int(double(mn) > flat_c * mean)) != 0) {
        // wang_landau_sampler.cpp:337-394, convergence time in steps
        const double mc_time = double(steps) / nbd;
        if (inverse_time && prev_conv >= 0 && since_flat > prev_conv) {
          if (!inv_active) inv_factor = mc_time * wl_f;
          inv_active = 1;
        }
        prev_conv = since_flat;
        wl_f = inv_active ? inv_factor / mc_time : wl_f / 2.0;
        ++n_flat;
        for (int i = lane; i < nb; i += 64) bins[i].hist = 0u;
        at_cur.hist = 0u;
        __syncthreads();
        bin_change = 0.0;
        since_flat = 0;
      }
      if (wl_f < f_min) converged = 1;
      __syncthreads();
    }
    const int64_t boff = wk->bin_off;
    for (int i = lane; i < nb; i += 64) {
      const PatchBin at = bins[i];
      args.logdos_pool[boff + i] = at.lg;
      args.hist_pool[boff + i] = at.hist;
      args.known_pool[boff + i] = uint8_t(at.known);
    }
    if (lane == 0) {
      wk->cur_bin = cur;
      wk->is_first = first;
      wk->n_moves += uint64_t(moves_made);
      wk->n_accept += n_acc;
      wk->n_outside += n_out;
      wk->n_self += n_self;
      wk->f = wl_f;
      wk->converged = converged;
      wk->n_flat += n_flat;
      wk->inv_active = inv_active;
      wk->inv_factor = inv_factor;
      wk->bin_change = bin_change;
      wk->steps = steps;
      wk->since_flat = since_flat;
      wk->prev_conv = prev_conv;
    }
  } else {
    const int64_t nmov = args.n_moves[chain];
    moves_made = nmov;
    for (int64_t blk0 = -int64_t(t0 & 63u); blk0 < nmov; blk0 += 64) {
      if (time_limit > 0 && blk0 > 0) {
        int stop = int(uint64_t(wall_clock64()) - t_begin > uint64_t(time_limit));
        if constexpr (kW > 1) {
          int* f = &stop_flag[(blk0 >> 6) & 1];
          if (tid == 0) *f = stop;
          __syncthreads();
          stop = *f;
        }
        if (stop) {
          moves_made = blk0;
          break;
        }
      }
      const int made = make_block(t0 + uint64_t(blk0), int(nmov - blk0 < 64 ? nmov - blk0 : 64), blk0);
      if constexpr (kHook) {
        if (failed) {
          moves_made = blk0 + made;
          break;
        }
      }
    }
  }

  // ---- write back
  if constexpr (kW > 1) __syncthreads();
  uint8_t* wocc = reinterpret_cast<uint8_t*>(occ_pool + pp->occ_off);
  for (int i = tid; i < N; i += kThreads) wocc[i] = occ[ref_of<true>(c, i).p];
  if constexpr (kCanonical && kTrkLds)
    for (int i = tid; i < N; i += kThreads) gtrk[i] = trk[i];
  if (kHook && lane == 0) {
    hk->bias_count = bias_cnt;
    hk->bias_energy = bias_energy;
    if (failed) {
      hk->status = 1;
      hk->failed_move = t0 + uint64_t(moves_made);
    }
  }
  if (kWL && lane == 0) {
    ChainState* st = states + chain;
    st->energy = energy;
    st->moves_done = t0 + uint64_t(moves_made);
    st->n_accept += n_acc;
  }
  if (!kWL && wave == 0) {
    ChainState* st = states + chain;
    const double se = wave_sum_f64(sum_de), se2 = wave_sum_f64(sum_de2);
    if (lane == 0) {
      st->energy = energy;
      st->moves_done = t0 + uint64_t(moves_made);
      st->n_accept += n_acc;
      st->n_samples += uint64_t(moves_made);
      st->sum_de += se;
      st->sum_de2 += se2;
      st->blk_end = energy;
      st->blk_moves = t0 + uint64_t(moves_made);
    }
    if constexpr (!kCanonical) {
#pragma unroll
      for (int b = 0; b < kBM; ++b) {
        const double a = wave_sum_f64(sum_s[b]), a2 = wave_sum_f64(sum_s2[b]), ae = wave_sum_f64(sum_se[b]);
        if (lane == 0) {
          st->sum_s[b] += a;
          st->sum_s2[b] += a2;
          st->sum_se[b] += ae;
        }
      }
    }
  }
}

}  // namespace cemc
