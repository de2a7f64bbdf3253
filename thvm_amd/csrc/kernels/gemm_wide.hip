// gemm_wide.hip -- launcher of the wide MFMA GEMM (gemm_wide_core.h): checks,
// tile and split choice, launch.
#include "gemm_wide_core.h"
#include "launch.h"
#include <stdio.h>

typedef void (*wide_fn)(ThvmGemvArgs);
// one picker per (weight type, x type, fused norm), each in its own unit
#define WIDE_PICKERS(X) X(2, 0, 0) X(2, 0, 1) X(2, 1, 0) X(1, 0, 0) X(1, 0, 1) X(0, 1, 0)
#define WIDE_DECL(w, x, n) wide_fn wide_pick_##w##_##x##_##n(int MT, int NT);
WIDE_PICKERS(WIDE_DECL)
#undef WIDE_DECL

// Where this kernel takes over from k_gemm (16 < M <= 64; above it is the only
// one).  k_gemm's x reads grow with M K N / (16 NT), this one pays a longer
// chain per block (a barrier per 128 k, the split hand-off).  Measured on
// gfx950, cold tiled fp8 weights in a graph, k_gemm / this kernel, us:
//                  M 8          M 16         M 17         M 60
//   28672 x 4096   22.0 / 21.2  23.0 / 21.3  28.5 / 21.4  40.5 / 26.1   wide N
//   14336 x 2048    9.3 /  7.5   9.8 /  7.8  10.1 /  7.8  16.1 / 11.1
//   32000 x 1024   10.9 /  8.7  11.9 /  8.9  13.3 /  8.9  20.0 / 11.7
//    4096 x 14336  13.6 / 13.6  15.5 / 13.9  17.1 / 13.9  33.1 / 18.7   long K
//    1600 x 6400    7.6 /  8.4   8.4 /  8.5   9.4 /  8.5  16.3 / 11.2
//    2048 x 8192    8.0 /  9.2   9.0 /  9.3  10.2 /  9.3  18.4 / 11.8
//    6144 x 4096    7.6 /  8.4   8.1 /  8.8   9.2 /  8.8  14.1 / 12.4   middling: by M
//    4096 x 4096    6.2 /  8.0   6.6 /  8.1   7.4 /  8.1  11.8 / 10.4
//    2048 x 4096    5.6 /  7.2   6.0 /  7.3   7.0 /  7.3  11.4 /  9.6
//    6400 x 1600    5.3 /  6.8   5.6 /  6.9   6.3 /  6.9   9.2 /  9.4   small: k_gemm
//    1600 x 1600    4.2 /  6.3   4.3 /  6.5   5.0 /  6.5   7.1 /  8.9
// and this kernel's time over k_gemm's on the far side of the lines: 4096 x 2048
// (and 6400, 8192 x 1600) M 33 1.06..1.21, M 48 1.02..1.15, M 64 0.99..1.08; 16-bit
// 4096, 8192 x 6144 M 17 1.04..1.07 (M 24 1.00).
// At 16 rows and fewer the widest N gain 4..25% too, and a long K 10% at 16;
// the line stays at 16 because k_gemm also takes a norm ahead of the product
// there, and a decoder of 5 to 16 rows holds no workspace.
extern "C" int thvm_k_gemm_wide_use(const ThvmGemvArgs *a) {
  if (a->seq) return 1;
  if (a->M <= 16) return 0;
  if (a->M > 64 || a->N >= 10240) return 1;
  if (a->K >= 6144) return a->M >= 24 || a->wdt == THVM_DT_FP8E4M3 || a->K >= 8192;
  return a->M > 32 && a->K >= 2048 && (uint64_t)a->N * a->K >= (a->K >= 4096 ? 8u << 20 : 12u << 20);
}

// Tile and splits.  One block of 8 waves is resident per CU (more than 128
// VGPRs), so the grid is planned in rounds of 256 blocks.
//   * one tile of x rows (M <= 64; bound by the weight stream): 64 weight rows
//     per block while that makes at most 256 blocks, else 128, and 256 for the
//     widest N (an LM head runs many rounds anyway: 128256 x 4096 at M = 60,
//     113 us with 128 rows, 102 with 256).  Behind a fused norm over more than 32
//     rows every block norms x again, which fp8 weights do not hide: 128 rows
//     from 129 such tiles on (16384 x 14336, M = 33: 69 us with 64 rows, 51 with
//     128, k_gemm 61; 10240 x 4096 23 and 18; 14336 x 2048 14.4 and 14.7);
//   * several (prompt chunks; bound by the MFMA and LDS pipes): the cheapest of
//     64, 128, 256 rows by rounds x chunks x the measured time of a chunk
//     (0.40, 0.56 and 1.04 us), e.g. at M = 299: 6144 x 4096 128 rows 22.4 us
//     against 256 26.5, 4096 x 14336 256 rows in 3 splits 47.5 against 58;
//   * splits fill the last round only (blocks * splits <= 256): a split costs
//     its hand-off (~4 chunks) and a read of its tile (~1 chunk), and a block
//     runs its chunks in fours.
// (asked for by the builtin's argument checks too, before the launcher's: in 64
// bits, and with no rows or columns one empty block)
static uint64_t tiles_of(uint32_t n, uint32_t t) { return ((uint64_t)n + t - 1) / t; }
static void wide_plan(const ThvmGemvArgs *a, int *MT, int *NT, uint32_t *SP) {
  *MT = a->M <= 32 ? 2 : 4;
  const uint64_t mt = tiles_of(a->M, 16u * *MT), g64 = tiles_of(a->N, 64);
  const uint32_t CH = (a->K / 64 + GW_KG - 1) / GW_KG;
  static const float chunk[3] = {0.40f, 0.56f, 1.04f};
  const bool xbound = a->norm && a->wdt == THVM_DT_FP8E4M3 && a->M > 32 && a->K >= 4096;
  const int one = g64 <= (xbound ? 128 : 256) ? 1 : g64 <= 512 ? 2 : 4;
  float best = 0.f;
  *NT = 1;
  *SP = 1;
  for (int i = 0; i < 3; i++) {
    const int nt = 1 << i;
    if (a->tune_r ? (int)a->tune_r != nt : mt == 1 && nt != one) continue;
    const uint64_t blocks = (g64 + nt - 1) / nt * mt;
    const uint32_t smax = a->tune_blocks ? a->tune_blocks
                        : blocks == 0 || blocks >= 256 ? 1 : 256 / blocks < 8 ? (uint32_t)(256 / blocks) : 8;
    for (uint32_t sp = a->tune_blocks ? smax : 1; sp <= smax && (sp == 1 || 4ull * sp <= CH); sp++) {
      const uint64_t per = ((CH + sp - 1) / sp + 3) / 4 * 4, rounds = (blocks * sp + 255) / 256;
      const float t = chunk[i] * (float)(rounds * per) + (sp > 1 ? 0.40f * (float)(4 + sp) : 0.f);
      if (best == 0.f || t < best) { best = t; *NT = nt; *SP = sp; }
    }
  }
}

// bytes the splits of this call need
extern "C" uint64_t thvm_k_gemm_wide_ws(const ThvmGemvArgs *a) {
  int MT, NT;
  uint32_t SP;
  if (!thvm_k_gemm_wide_use(a)) return 0;
  wide_plan(a, &MT, &NT, &SP);
  if (SP <= 1) return 0;
  const uint64_t tiles = tiles_of(a->N, 64u * NT) * tiles_of(a->M, 16u * MT);
  return GW_CTR_BYTES + tiles * SP * (GW_NWAVES * NT * MT * 1024ull + 16ull * MT * 4);
}

// splits are planned within 256 blocks, of at most 256 x 64 tiles
extern "C" uint64_t thvm_k_gemm_wide_ws_max(void) {
  return GW_CTR_BYTES + 256ull * (GW_NWAVES * 4 * 4 * 1024ull + 64 * 4);
}

extern "C" int thvm_k_gemm_wide(const ThvmGemvArgs *a, hipStream_t s, char *err, int errlen) {
  if (a->norm && (a->norm != 1 || a->xdt != THVM_DT_BF16 || a->norm_w == nullptr)) {
    snprintf(err, errlen, "gemm_wide: fuses RMSNorm with a gain over bf16 x only");
    return -1;
  }
  if (a->tune_r && a->tune_r != 1 && a->tune_r != 2 && a->tune_r != 4) {
    snprintf(err, errlen, "gemm_wide: r (64-row weight tiles per block) must be 1, 2 or 4");
    return -1;
  }
  if (a->K % 64 || ((uint64_t)a->ldx * 2) % 16 || ((uintptr_t)a->x & 15) || ((uintptr_t)a->w & 15)) {
    snprintf(err, errlen, "gemm_wide: K a multiple of 64, x rows and W 16-byte aligned");
    return -1;
  }
  if (64ull * a->ldx * 2 >= (1ull << 31) || 64ull * a->K * (a->wdt == THVM_DT_FP8E4M3 ? 1 : 2) >= (1ull << 30)) {
    snprintf(err, errlen, "gemm_wide: 64 rows of x or W exceed 1 GiB");
    return -1;
  }
  int MT, NT;
  uint32_t SP;
  wide_plan(a, &MT, &NT, &SP);
  ThvmGemvArgs k = *a;
  k.splits = SP;
  if (SP > 1 && tiles_of(a->N, 64u * NT) * tiles_of(a->M, 16u * MT) > GW_CTR_BYTES / 4) {
    snprintf(err, errlen, "gemm_wide: %u splits of more than %u tiles", SP, GW_CTR_BYTES / 4);
    return -1;
  }
  if (SP > 1 && (a->ws == nullptr || a->ws_bytes < thvm_k_gemm_wide_ws(a))) {
    snprintf(err, errlen, "gemm_wide: %u splits need %llu bytes of workspace", SP,
             (unsigned long long)thvm_k_gemm_wide_ws(a));
    return -1;
  }
  const int xbf = a->xdt == THVM_DT_BF16, xf16 = a->xdt == THVM_DT_FP16;
  wide_fn f = nullptr;
  const int w = a->wdt == THVM_DT_FP8E4M3 ? GW_FP8 : a->wdt == THVM_DT_BF16 ? GW_BF16 : a->wdt == THVM_DT_FP16 ? GW_F16 : -1;
  const int x = xbf ? GX_BF16 : xf16 ? GX_F16 : -1, nm = a->norm ? 1 : 0;
  static_assert(GW_F16 == 0 && GW_BF16 == 1 && GW_FP8 == 2 && GX_BF16 == 0 && GX_F16 == 1, "picker numbering");
#define WIDE_CASE(W, X, Q) if (w == W && x == X && nm == Q) f = wide_pick_##W##_##X##_##Q(MT, NT);
  WIDE_PICKERS(WIDE_CASE)
#undef WIDE_CASE
  if (!f) { snprintf(err, errlen, "gemm_wide: no kernel for w=%u x=%u NT=%d", a->wdt, a->xdt, NT); return -1; }
  // four rows per lane at a time where every row and buffer is aligned for it
  const uintptr_t al = a->ydt == THVM_DT_FP32 ? 15 : 7;
  const bool qkv = a->epi == THVM_EPI_QKV || a->epi == THVM_EPI_QKV_ROPE;
  k.vec4 = a->N % 4 == 0 && a->ldy % 4 == 0 && !((uintptr_t)a->y & al) && !((uintptr_t)a->res & al) &&
           !((uintptr_t)a->bias & al) && !((uintptr_t)a->scale & 15) &&
           (!qkv || (a->head_dim % 4 == 0 && !((uintptr_t)a->kcache & al) && !((uintptr_t)a->vcache & al) &&
                     !((uintptr_t)a->rope_cos & 7) && !((uintptr_t)a->rope_sin & 7)));
  if (a->seq && !k.vec4) {
    snprintf(err, errlen, "gemm_wide: seq needs aligned rows of four (the scalar epilogue has one position per row)");
    return -1;
  }
  const uint64_t total = tiles_of(a->M, 16u * MT) * tiles_of(a->N, 64u * NT) * SP, grid = (total + 7) / 8 * 8;
  if (grid > 0x7fffffffull) { snprintf(err, errlen, "gemm_wide: grid too large"); return -1; }
  const uint32_t xlds = 2u * 16u * MT * GW_XROW, elds = (uint32_t)GW_NWAVES * NT * MT * 1024u;
  const uint32_t lds = xlds > elds ? xlds : elds;
  thvm_launch(true, true, f, dim3((uint32_t)grid), dim3(GW_THREADS), lds, s, k);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { snprintf(err, errlen, "gemm_wide launch: %s", hipGetErrorString(e)); return -1; }
  return 0;
}
