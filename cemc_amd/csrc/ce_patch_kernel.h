// Patch kernel of the cluster-expansion Metropolis engine (gfx950): the sweep
// of one chain with the sub-clusters of a site regrouped into patches
// (ce_patches.h).  Instantiations: ce_patch_inst.hip.
//
// One workgroup of kW waves owns one chain on a closed-form periodic lattice
// with one translation group; the padded occupation box, the species tracker
// and the patch tables stay in LDS for the launch.  Moves are made in rounds
// of kK: all are evaluated against the same state, then committed in order
// up to the first one that reads what an accepted earlier one changed.
//
// Work split.  A flip needs 12 (two species, pairs to the 4th shell and
// triplets to the 2nd), 59 (three species, four-body clusters) or 426 (four
// species, four-body to the 3rd shell) patch entries where it needed 114, 494
// and 1746 sub-cluster entries.  kG lanes evaluate one move, kR patches each:
// a row of 16 lanes for up to 64 patches, so that a wave evaluates four moves
// at once and each sum takes four DPP levels inside a row; the whole wave for
// more.
//
// What bounds it: the dependent chain of a round (move fetch, gathers, table
// reads, sum, verdict, commit), not bandwidth.  So everything that does not
// depend on the verdict is done while the reads are in flight: which moves of
// the round affect which, where the commits would go; and everything that
// the next round does not need is put off to the end of the 64-move block,
// where lane l still holds move l: energies by one prefix sum over the lanes,
// sample sums in per-lane accumulators added up once per launch.
#pragma once

#include "ce_sweep.h"

namespace cemc {

// Dynamic LDS: padded occupation | tracker (canonical, when held in LDS) | patch tables.
struct PatchLayout {
  uint32_t trk, tab, total;
};
__host__ __device__ inline PatchLayout patch_layout(int occ_bytes, int trk_sites, int tab_doubles) {
  PatchLayout L;
  L.trk = align16(uint32_t(occ_bytes));
  L.tab = L.trk + align16(uint32_t(trk_sites) * 2u);
  L.total = L.tab + uint32_t(tab_doubles) * 8u;
  return L;
}

namespace {

constexpr int kNoPatch = 1 << 24;  // no lattice offset: the second site of a swap does not see the first

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

// Sum over the row of 16 lanes; every lane of the row ends with it.
__device__ __attribute__((always_inline)) inline double row_sum_f64(double v) {
  v += dpp_f64<0x128>(v);
  return octet_sum_f64(v);
}

// Padded-lattice offset of site i as seen from site j when it lies within
// the halo of j along every axis (then a member offset of j equals it exactly
// when the member is i), else kNoPatch.
__device__ __attribute__((always_inline)) inline int near_offset(const SweepCtx& c, const Ref& i, const Ref& j) {
  auto axis = [&](int d, int L) {
    d += d > c.h ? -L : 0;
    d += d < -c.h ? L : 0;
    return d;
  };
  const int dx = axis(i.x - j.x, c.L1), dy = axis(i.y - j.y, c.L2), dz = axis(i.z - j.z, c.L3);
  const bool in = dx >= -c.h && dx <= c.h && dy >= -c.h && dy <= c.h && dz >= -c.h && dz <= c.h;
  return in ? (dx * c.P2 + dy) * c.P3 + dz : kNoPatch;
}

}  // namespace

// kBM: basis functions, one less than the species (1, 2, 3).  kP: moves that
// a lane group evaluates per round.  kTrkLds: the tracker is held in LDS,
// else in HBM, where only its lookups per block and its commits touch it.
template <bool kCanonical, int kBM, int kG, int kR, int kW, int kP, bool kTrkLds>
__global__ __launch_bounds__(64 * kW) void patch_kernel(
    const ChainParams* __restrict__ params, ChainState* __restrict__ states, const ModelDev* __restrict__ models,
    int8_t* __restrict__ occ_pool, uint16_t* __restrict__ trk_pool, const int32_t* __restrict__ chain_order,
    const int64_t* __restrict__ n_moves, uint32_t* __restrict__ accept_log, int64_t log_words, int64_t time_limit) {
  static_assert(kG == 16 || kG == 64, "a row or the whole wave evaluates a move");
  constexpr int kS = kBM + 1;
  constexpr int kQ = kBM == 1 ? 6 : (kBM == 2 ? 5 : 4);  // members per patch (patch_members)
  constexpr int kPer = 64 / kG;                           // moves a wave evaluates side by side
  constexpr int kK = kW * kP * kPer;                       // moves per round
  static_assert(kK == 8 || (kK == 16 && kW == 4), "rounds of 8, or of 16 on four waves");
  constexpr int kThreads = 64 * kW;
  extern __shared__ __align__(16) unsigned char lds[];
  __shared__ double dphi_tab[kS * kS * kBM];  // [(old*S+new)*B + d]
  __shared__ double dsingle_tab[kS * kS];
  __shared__ double phi_tab[kBM * kS];
  __shared__ uint4 mv_a[64];  // canonical: p_i, p_j, offset of i seen from j, a | b << 8; SGC: p, cell, image, species offset
  __shared__ uint4 mv_b[kCanonical ? 64 : 1];  // canonical: cell_i, cell_j, image_i, image_j
  __shared__ uint2 mv_s[kCanonical ? 64 : 1];  // canonical: site_i | site_j << 16, slot_a | slot_b << 16
  __shared__ double red[2][kK];                // sums of the round's moves, by parity
  __shared__ uint16_t conf_l[kK];               // rounds of 16: earlier moves that affect each
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
  const uint64_t im0 = m.imask[0], im1 = m.imask[1];
  const int occ_bytes = m.pdims[0] * c.P2 * c.P3;
  const PatchLayout L = patch_layout(occ_bytes, kCanonical && kTrkLds ? N : 0, m.ptab_size);
  uint8_t* occ = reinterpret_cast<uint8_t*>(lds);
  double* tab = reinterpret_cast<double*>(lds + L.tab);
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
  const double dphi01 = dphi_tab[kBM], dphi10 = dphi_tab[kS * kBM];  // two species: 0 -> 1 and 1 -> 0

  double energy = states[chain].energy;
  const uint64_t t0 = states[chain].moves_done;
  const double e_ref = states[chain].e_ref;
  const int64_t nmov = n_moves[chain];
  uint64_t n_acc = 0;
  double sum_de = 0.0, sum_de2 = 0.0;  // this lane's moves
  const double inv_n = 1.0 / double(N);
  double sing[kBM], sum_s[kBM], sum_s2[kBM], sum_se[kBM];
#pragma unroll
  for (int d = 0; d < kBM; ++d) sing[d] = sum_s[d] = sum_s2[d] = sum_se[d] = 0.0;
  if constexpr (!kCanonical) {
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
  const double inv_kT = 1.0 / kT;
  const uint64_t seed = pp->seed, uid = pp->uid;
  const uint32_t np = uint32_t(pp->n_present);
  const uint32_t present_pk = pp->present_pk;
  const uint64_t cnt_lo = pp->count_pk[0], cnt_hi = pp->count_pk[1];
  const uint64_t seg_lo = pp->segoff_pk[0], seg_hi = pp->segoff_pk[1];
  uint32_t* acc_log = accept_log ? accept_log + int64_t(chain) * log_words : nullptr;
  const uint64_t t_begin = time_limit > 0 ? uint64_t(wall_clock64()) : 0u;
  int64_t moves_made = nmov;

  // LDS written by this wave is read by it in program order; other waves are
  // ordered by barriers
  auto own_order = [] { __atomic_signal_fence(__ATOMIC_SEQ_CST); };

  // one flip's table sum over this lane's patches around padded site p: the
  // slices' sums, or with dphi the change; `off`: this padded offset holds a
  // species `ds` higher than the lattice says
  auto flip = [&](int p, const double (&dphi)[kBM], bool patched, int off, int ds) {
    int idx[kR];
#pragma unroll
    for (int k = 0; k < kR; ++k) {
      uint32_t s[kQ];
#pragma unroll
      for (int q = 0; q < kQ; ++q) s[q] = occ[p + mo[k][q]];
      uint32_t v = s[kQ - 2];
#pragma unroll
      for (int q = kQ - 3; q >= 0; --q) v = v * uint32_t(kS) + s[q];
      idx[k] = int(v + __umul24(s[kQ - 1], uint32_t(wl[k])));
    }
    if (patched) {
#pragma unroll
      for (int k = 0; k < kR; ++k) {
        int w = mo[k][kQ - 1] == off ? wl[k] : 0, pw = 1;
#pragma unroll
        for (int q = 0; q < kQ - 1; ++q) {
          w = mo[k][q] == off ? pw : w;
          pw *= kS;
        }
        idx[k] += w * ds;
      }
    }
    double g[kR][kBM];
#pragma unroll
    for (int k = 0; k < kR; ++k) {
      const double* t = tab + (base[k] + kBM * idx[k]);
      if constexpr (kBM == 2) {
        const dbl2_t two = load_pair(t);
        g[k][0] = two.x;
        g[k][1] = two.y;
      } else {
#pragma unroll
        for (int d = 0; d < kBM; ++d) g[k][d] = t[d];
      }
    }
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

  uint32_t rnd = 0;
  for (int64_t blk0 = 0; blk0 < nmov; blk0 += 64) {
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
    // lane l decodes move blk0 + l
    const Philox4 blk = philox4x64_10(t0 + uint64_t(blk0) + uint64_t(lane), 0, 0, 0, seed, uid);
    const double log_u = log(unit_double(blk.w3));
    const int n_in = int(nmov - blk0 < 64 ? nmov - blk0 : 64);
    uint32_t v_old = 0, v_new = 0;  // canonical: species a and b
    int v_ta = 0, v_tb = 0;         // canonical: tracker slots
    int v_p = 0;                    // SGC: padded site
    uint32_t v_off = 0;             // SGC: offset of the new species
    // canonical: the sites now in the move's slots, to registers and LDS
    auto look_up = [&] {
      const int si = trk[v_ta], sj = trk[v_tb];
      const Ref ri = ref_of<true>(c, si), rj = ref_of<true>(c, sj);
      const uint32_t ci = uint32_t(ri.x) | (uint32_t(ri.y) << 8) | (uint32_t(ri.z) << 16);
      const uint32_t cj = uint32_t(rj.x) | (uint32_t(rj.y) << 8) | (uint32_t(rj.z) << 16);
      mv_a[lane] = uint4{uint32_t(ri.p), uint32_t(rj.p), uint32_t(near_offset(c, ri, rj)), v_old | (v_new << 8)};
      mv_b[lane] = uint4{ci, cj, image_word<true>(c, ri), image_word<true>(c, rj)};
      mv_s[lane] = uint2{uint32_t(si) | (uint32_t(sj) << 16), uint32_t(v_ta) | (uint32_t(v_tb) << 16)};
    };
    if constexpr (kCanonical) {
      const uint32_t ia = bounded32(uint32_t(blk.w0 >> 32), np);
      uint32_t ib = ia + 1u + bounded32(uint32_t(blk.w0), np - 1u);
      ib -= ib >= np ? np : 0u;
      v_old = (present_pk >> (4u * ia)) & 15u;
      v_new = (present_pk >> (4u * ib)) & 15u;
      v_ta = unpack16(seg_lo, seg_hi, ia) + int(bounded64(blk.w1, uint64_t(unpack16(cnt_lo, cnt_hi, ia))));
      v_tb = unpack16(seg_lo, seg_hi, ib) + int(bounded64(blk.w2, uint64_t(unpack16(cnt_lo, cnt_hi, ib))));
      look_up();
    } else {
      const Ref r = ref_of<true>(c, int(bounded64(blk.w1, uint64_t(N))));
      v_p = r.p;
      v_off = bounded32(uint32_t(blk.w0), uint32_t(kS - 1));
      mv_a[lane] = uint4{uint32_t(r.p), uint32_t(r.x) | (uint32_t(r.y) << 8) | (uint32_t(r.z) << 16),
                         image_word<true>(c, r), v_off};
    }
    // every wave writes the same values; the slowest wave may still be
    // reading the last block's, which it no longer uses (see the round's end)
    if constexpr (kW > 1)
      __syncthreads();
    else
      own_order();
    uint64_t acc_bits = 0;
    double de_made = 0.0;           // this lane's move: its energy change if accepted
    uint32_t o_made = 0, n_made = 0;  // SGC: its species change (equal: rejected)
    int l0 = 0;
    while (l0 < n_in) {
      const int n = n_in - l0 < kK ? n_in - l0 : kK;
      auto at = [&](int k) { return l0 + k < 63 ? l0 + k : 63; };
      // SGC: the species at this lane's own site
      uint32_t o_l = v_old, n_l = v_new;
      if constexpr (!kCanonical) {
        o_l = occ[v_p];
        n_l = o_l + 1u + v_off;
        n_l -= n_l >= uint32_t(kS) ? uint32_t(kS) : 0u;
      }
      // ---- this wave's moves
      double part[kP];
#pragma unroll
      for (int t = 0; t < kP; ++t) {
        const int k = (wave * kP + t) * kPer + (kG == 64 ? 0 : lane / kG);
        const uint4 a = mv_a[at(k)];
        double dphi[kBM];
        if constexpr (kCanonical) {
          const int o = int(a.w & 255u), nw = int(a.w >> 8);
#pragma unroll
          for (int d = 0; d < kBM; ++d) dphi[d] = kBM == 1 ? 0.0 : dphi_tab[(o * kS + nw) * kBM + d];
          const bool any = __builtin_amdgcn_ballot_w64(int(a.z) != kNoPatch) != 0;
          const double vi = flip(int(a.x), dphi, false, 0, 0);
          // the swap's second flip sees site i already changed (ce_updater.cpp:845-852)
          const double vj = flip(int(a.y), dphi, any, int(a.z), nw - o);
          part[t] = vi - vj;
        } else {
          if constexpr (kBM > 1) {
            const int o = occ[a.x];
            int nw = o + 1 + int(a.w);
            nw -= nw >= kS ? kS : 0;
#pragma unroll
            for (int d = 0; d < kBM; ++d) dphi[d] = dphi_tab[(o * kS + nw) * kBM + d];
          } else {
            dphi[0] = 0.0;
          }
          part[t] = flip(int(a.x), dphi, false, 0, 0);
        }
      }
      // ---- which earlier moves of the round affect which: lane (b, a)
      constexpr int kA = kK == 16 ? 16 : 8;
      const int pb = lane / kA + (kK == 16 ? 4 * wave : 0), pa = lane & (kA - 1);
      bool hit = false;
      int com_i = -1, com_j = -1;  // this lane's commit: padded images of sites i and j
      uint32_t com_o = 0, com_n = 0, com_sites = 0, com_slots = 0;
      const int ck = kK == 16 ? 4 * wave + (lane >> 4) : lane >> 3;  // the move it commits
      const int cim = lane & 7;
      if constexpr (kCanonical) {
        const uint4 vb = mv_b[at(pb)], va = mv_b[at(pa)];
        const uint32_t slb = mv_s[at(pb)].y, sla = mv_s[at(pa)].y;
        const uint32_t ta_a = sla & 0xFFFFu, tb_a = sla >> 16, ta_b = slb & 0xFFFFu, tb_b = slb >> 16;
        hit = cells_interact(va.x, vb.x, c, im0, im1) || cells_interact(va.x, vb.y, c, im0, im1) ||
              cells_interact(va.y, vb.x, c, im0, im1) || cells_interact(va.y, vb.y, c, im0, im1) || ta_a == ta_b ||
              ta_a == tb_b || tb_a == ta_b || tb_a == tb_b;
        const uint4 cb = mv_b[at(ck)];
        const uint2 cs = mv_s[at(ck)];
        const uint32_t on = mv_a[at(ck)].w;
        com_sites = cs.x;
        com_slots = cs.y;
        com_o = on & 255u;
        com_n = on >> 8;
        if constexpr (kK == 16) {
          com_i = image_of(c, (lane & 8) ? cb.w : cb.z, cim);
        } else {
          com_i = image_of(c, cb.z, cim);
          com_j = image_of(c, cb.w, cim);
        }
      } else {
        hit = cells_interact(mv_a[at(pa)].y, mv_a[at(pb)].y, c, im0, im1);
        const uint4 ca = mv_a[at(ck)];
        com_i = image_of(c, ca.z, cim);
        if (kK == 16 && (lane & 8)) com_i = -1;
        com_n = occ[ca.x] + 1u + ca.w;
        com_n -= com_n >= uint32_t(kS) ? uint32_t(kS) : 0u;
      }
      const uint64_t conf = __builtin_amdgcn_ballot_w64(hit && pa < pb);
      // ---- sums of the round's moves
      double* rs = red[rnd & 1u];
#pragma unroll
      for (int t = 0; t < kP; ++t) {
        const double s = kG == 16 ? row_sum_f64(part[t]) : wave_sum_f64(part[t]);
        if ((lane & (kG - 1)) == 0) rs[(wave * kP + t) * kPer + (kG == 64 ? 0 : lane / kG)] = s;
      }
      if constexpr (kK == 16) {
        if (lane < 4) conf_l[4 * wave + lane] = uint16_t(conf >> (16 * lane));
      }
      if constexpr (kW > 1)
        __syncthreads();
      else
        own_order();
      // ---- every lane decides the move it decoded
      const int r = lane - l0;
      const bool valid = r >= 0 && r < n;
      const double tot = rs[valid ? r : 0];
      uint32_t conf_r = 0;
      if constexpr (kK == 16) conf_r = conf_l[valid ? r : 0];
      double dE;
      if constexpr (kBM == 1) {
        const double d0 = o_l == 0 ? dphi01 : dphi10;
        dE = kCanonical ? __dmul_rn(d0, tot) : fma(d0, tot, dsingle_tab[o_l == 0 ? 1 : kS]);
      } else {
        dE = kCanonical ? tot : tot + dsingle_tab[int(o_l) * kS + int(n_l)];
      }
      // the Metropolis test of the sweep kernel (ce_sweep.h)
      const double x = -dE * inv_kT;
      const double margin = 1e-12 * (1.0 + fabs(x));
      int verdict = (dE < 0.0 || log_u < x - margin) ? 1 : (log_u > x + margin ? 0 : 2);
      if (valid && verdict == 2) verdict = int(unit_double(blk.w3) <= exp(-dE / kT));
      const uint64_t acc = __builtin_amdgcn_ballot_w64(valid && verdict == 1) >> l0;  // bit k: move k of the round
      int stop = n;
      if constexpr (kK == 16) {
        const uint64_t hits = __builtin_amdgcn_ballot_w64(valid && (conf_r & uint32_t(acc)) != 0) >> l0;
        if (hits != 0) stop = int(__builtin_ctzll(hits));
      } else {
        uint32_t dup = uint32_t(acc) & 0xFFu;
        dup |= dup << 8;
        dup |= dup << 16;
        const uint64_t hits = conf & ((uint64_t(dup) << 32) | dup);  // byte b: accepted moves that affect move b
        if (hits != 0) {
          const int first = int(__builtin_ctzll(hits)) >> 3;
          stop = first < stop ? first : stop;
        }
      }
      const uint32_t com = uint32_t(acc) & ((1u << stop) - 1u);
      if (com != 0) {
        if ((com >> ck) & 1u) {
          if constexpr (kCanonical) {
            if constexpr (kK == 16) {
              if (com_i >= 0) occ[com_i] = uint8_t((lane & 8) ? com_o : com_n);
            } else {
              if (com_i >= 0) occ[com_i] = uint8_t(com_n);
              if (com_j >= 0) occ[com_j] = uint8_t(com_o);
            }
            const int first = kK == 16 ? (lane & 15) : cim;
            if (first == 0) trk[com_slots & 0xFFFFu] = uint16_t(com_sites >> 16);
            if (first == 1) trk[com_slots >> 16] = uint16_t(com_sites & 0xFFFFu);
          } else {
            if (com_i >= 0) occ[com_i] = uint8_t(com_n);
          }
        }
        const bool mine = valid && ((com >> (r & 31)) & 1u);
        de_made = mine ? dE : de_made;
        if constexpr (!kCanonical) {
          o_made = mine ? o_l : o_made;
          n_made = mine ? n_l : n_made;
        }
        acc_bits |= uint64_t(com) << l0;
      }
      l0 += stop;
      ++rnd;
      if constexpr (kW > 1)
        __syncthreads();  // the commits before the next round's reads
      else
        own_order();
      if constexpr (kCanonical) {
        // later moves of the block whose slots got other sites
        if (com != 0 && l0 < n_in) {
          bool stale = false;
          uint32_t rest = com;
          while (rest != 0) {
            const int k = l0 - stop + int(__builtin_ctz(rest));
            rest &= rest - 1u;
            const int ta = __builtin_amdgcn_readlane(v_ta, k), tb = __builtin_amdgcn_readlane(v_tb, k);
            stale = stale || v_ta == ta || v_ta == tb || v_tb == ta || v_tb == tb;
          }
          if (__builtin_amdgcn_ballot_w64(stale && lane >= l0) != 0) {
            look_up();
            if constexpr (kW > 1)
              __syncthreads();
            else
              own_order();
          }
        }
      }
    }
    n_acc += uint64_t(__builtin_popcountll(acc_bits));
    if (acc_log != nullptr && tid < 2) {
      const int64_t w = blk0 >> 5;
      if (lane == 0) acc_log[w] = uint32_t(acc_bits);
      if (lane == 1 && n_in > 32) acc_log[w + 1] = uint32_t(acc_bits >> 32);
    }
    // ---- the block's energies and samples: lane l after its own move
    if (kW == 1 || wave == 0) {
      const double e_l = energy + wave_scan_f64(de_made);
      const double d = lane < n_in ? e_l - e_ref : 0.0;
      sum_de += d;
      sum_de2 = fma(d, d, sum_de2);
      energy = readlane_f64(e_l, 63);
      if constexpr (!kCanonical) {
#pragma unroll
        for (int b = 0; b < kBM; ++b) {
          const double ds = o_made == n_made ? 0.0 : __dmul_rn(dphi_tab[(int(o_made) * kS + int(n_made)) * kBM + b], inv_n);
          const double s_l = sing[b] + wave_scan_f64(ds);
          const double s = lane < n_in ? s_l : 0.0;
          sum_s[b] += s;
          sum_s2[b] = fma(s, s, sum_s2[b]);
          sum_se[b] = fma(s, d, sum_se[b]);
          sing[b] = readlane_f64(s_l, 63);
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
  if (wave == 0) {
    ChainState* st = states + chain;
    const double se = wave_sum_f64(sum_de), se2 = wave_sum_f64(sum_de2);
    if (lane == 0) {
      st->energy = energy;
      st->moves_done = t0 + uint64_t(moves_made);
      st->n_accept += n_acc;
      st->n_samples += uint64_t(moves_made);
      st->sum_de += se;
      st->sum_de2 += se2;
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
