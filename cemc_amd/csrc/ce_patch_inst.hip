// Instantiations of the patch kernel for one number of waves per chain,
// CEMC_PATCH_WAVES (1, 2, 4, 8), one object each; exposes
// patch_fn_w<W>(canonical, kbm, kg, kr, trk_lds, hooks), the kernel's address or
// nullptr for a variant that is not built.  One wave: a quad per move, up to 60
// patches; two or four waves: a row of 16 lanes per move, up to 64 patches;
// two, four or eight waves: a wave per move, up to 448 patches.  kg 8: the
// Wang-Landau kernel, or (hooks) chains with constraints or a bias.
#include "ce_patch_kernel.h"

#ifndef CEMC_PATCH_WAVES
#error "CEMC_PATCH_WAVES must be defined"
#endif

namespace cemc {

namespace {

constexpr int W = CEMC_PATCH_WAVES;

template <bool C, int KBM>
const void* row_fn(int kr) {
  if constexpr (W == 1) {
    if (kr == 3) return reinterpret_cast<const void*>(&patch_kernel<C, KBM, 4, 3, 1, 1, true>);
    if (kr == 6) return reinterpret_cast<const void*>(&patch_kernel<C, KBM, 4, 6, 1, 1, true>);
    if (kr == 9) return reinterpret_cast<const void*>(&patch_kernel<C, KBM, 4, 9, 1, 1, true>);
    if (kr == 15) return reinterpret_cast<const void*>(&patch_kernel<C, KBM, 4, 15, 1, 1, true>);
  } else if constexpr (W <= 4) {
    constexpr int kP = 4 / W;
    if (kr == 1) return reinterpret_cast<const void*>(&patch_kernel<C, KBM, 16, 1, W, kP, true>);
    if (kr == 2) return reinterpret_cast<const void*>(&patch_kernel<C, KBM, 16, 2, W, kP, true>);
    if (kr == 4) return reinterpret_cast<const void*>(&patch_kernel<C, KBM, 16, 4, W, kP, true>);
  }
  return nullptr;
}

// Wang-Landau walkers, or chains with hooks (H): eight lanes per move, up to 64 patches
template <bool C, int KBM, bool H>
const void* octet_fn(int kr) {
  if constexpr (W == 1) {
    if (kr == 2) return reinterpret_cast<const void*>(&patch_kernel<C, KBM, 8, 2, 1, 1, true, !H, H>);
    if (kr == 4) return reinterpret_cast<const void*>(&patch_kernel<C, KBM, 8, 4, 1, 1, true, !H, H>);
    if (kr == 8) return reinterpret_cast<const void*>(&patch_kernel<C, KBM, 8, 8, 1, 1, true, !H, H>);
  }
  return nullptr;
}

template <bool C, int KBM, bool T>
const void* wave_fn(int kr) {
  if constexpr (W >= 2) {
    constexpr int kP = 8 / W;
    if (kr == 2) return reinterpret_cast<const void*>(&patch_kernel<C, KBM, 64, 2, W, kP, T>);
    if (kr == 4) return reinterpret_cast<const void*>(&patch_kernel<C, KBM, 64, 4, W, kP, T>);
    if (kr == 7) return reinterpret_cast<const void*>(&patch_kernel<C, KBM, 64, 7, W, kP, T>);
  }
  return nullptr;
}

template <bool C, bool H>
const void* pick_octet(int kbm, int kr) {
  return kbm == 1 ? octet_fn<C, 1, H>(kr) : (kbm == 2 ? octet_fn<C, 2, H>(kr) : (kbm == 3 ? octet_fn<C, 3, H>(kr) : nullptr));
}

template <bool C>
const void* pick(int kbm, int kg, int kr, bool trk_lds, bool hooks) {
  if (kg == 8) return hooks ? pick_octet<C, true>(kbm, kr) : pick_octet<C, false>(kbm, kr);
  if (hooks) return nullptr;
  if (kg == (W == 1 ? 4 : 16)) {
    if (!trk_lds) return nullptr;
    return kbm == 1 ? row_fn<C, 1>(kr) : (kbm == 2 ? row_fn<C, 2>(kr) : (kbm == 3 ? row_fn<C, 3>(kr) : nullptr));
  }
  if (kg != 64) return nullptr;
  if (!C || trk_lds)
    return kbm == 1 ? wave_fn<C, 1, true>(kr)
                    : (kbm == 2 ? wave_fn<C, 2, true>(kr) : (kbm == 3 ? wave_fn<C, 3, true>(kr) : nullptr));
  return kbm == 3 ? wave_fn<C, 3, false>(kr) : nullptr;
}

}  // namespace

#define CEMC_PATCH_FN_NAME2(W_) patch_fn_w##W_
#define CEMC_PATCH_FN_NAME(W_) CEMC_PATCH_FN_NAME2(W_)

const void* CEMC_PATCH_FN_NAME(CEMC_PATCH_WAVES)(bool canonical, int kbm, int kg, int kr, bool trk_lds, bool hooks) {
  return canonical ? pick<true>(kbm, kg, kr, trk_lds, hooks) : pick<false>(kbm, kg, kr, trk_lds, hooks);
}

}  // namespace cemc
