// gemm_wide_inst.hip -- the wide GEMM's instances for one (weight type, x type,
// fused norm), chosen by GW_WT / GW_XT / GW_NM; the build compiles this file
// once per combination.  GW_PICK names the picker gemm_wide.hip calls.
#include "gemm_wide_core.h"

typedef void (*wide_fn)(ThvmGemvArgs);
wide_fn GW_PICK(int MT, int NT) {
  switch (MT * 8 + NT) {
    case 2 * 8 + 1: return k_gemm_wide<GW_WT, GW_XT, 2, 1, GW_NM>;
    case 2 * 8 + 2: return k_gemm_wide<GW_WT, GW_XT, 2, 2, GW_NM>;
    case 2 * 8 + 4: return k_gemm_wide<GW_WT, GW_XT, 2, 4, GW_NM>;
    case 4 * 8 + 1: return k_gemm_wide<GW_WT, GW_XT, 4, 1, GW_NM>;
    case 4 * 8 + 2: return k_gemm_wide<GW_WT, GW_XT, 4, 2, GW_NM>;
    case 4 * 8 + 4: return k_gemm_wide<GW_WT, GW_XT, 4, 4, GW_NM>;
    default: return nullptr;
  }
}
