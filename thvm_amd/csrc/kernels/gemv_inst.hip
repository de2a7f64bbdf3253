// gemv_inst.hip -- the standalone GEMV kernel instances for one (weight type,
// x type) pair, chosen at compile time by GEMV_WT / GEMV_XD; the build
// compiles this file once per pair (twelve translation units in parallel
// instead of one unit holding every instance).  GEMV_PICK names the pair's
// picker, which gemv.hip's launcher calls.
#include "gemv_core.h"

#if !defined(GEMV_WT) || !defined(GEMV_XD) || !defined(GEMV_PICK)
#error "gemv_inst.hip is compiled with -DGEMV_WT=<0..3> -DGEMV_XD=<0..3> -DGEMV_PICK=<name>"
#endif

// The standalone kernel: waves own row groups blockIdx*nw + wave, grid-stride.
// blockIdx.y selects a chunk of M batch rows (x, y and res advance by M rows
// per chunk): batches above 4 rows whose operands the MFMA GEMM does not take
// run as chunks of 4, each output row computed exactly as at M <= 4.
// More than one x row: blocks of at most 8 waves, two per CU (128 VGPRs).  The
// fused norm is a template argument there: one instance for all of them spilled
// with four chunks in flight, and two chunks took up to 1.6 times as long over
// long rows (M = 3, 256 x 14336 fp8 13.3 us against 9.2) and 1.1 times at wide N
// (M = 4, 128256 x 4096 123 against 113).  us in one block of 1024 threads at
// most / now, fp8: 28672 x 4096 with a fused RMSNorm M = 2 28.9 / 24.2, M = 3
// 36.7 / 27.1, M = 4 43.3 / 32.9; 4096 x 4096 fp16 with a LayerNorm 11.6 / 9.8,
// 13.1 / 11.0, 15.2 / 14.7.
template <int WT, int XD, int M, int R, int U, int NK = -1>
__global__ __launch_bounds__(M == 1 ? 1024 : 512, 4) void k_gemv(ThvmGemvArgs a) {
  extern __shared__ __align__(16) unsigned char xs_raw[];
  // a fused norm's partial sums, after the rows (the launcher adds the room)
  constexpr uint32_t XB = WT == WT_F32 || XD == XD_F32 ? 4 : 2;
  float *const red = (float *)(xs_raw + (size_t)M * a.K * XB);
  const int nw = blockDim.x >> 6;
  const uint32_t g = blockIdx.x * nw + (threadIdx.x >> 6);
  if (blockIdx.y) {
    const uint64_t m0 = (uint64_t)blockIdx.y * M, ys = a.ydt == THVM_DT_FP32 ? 4 : 2;
    a.x = (const char *)a.x + m0 * a.ldx * XDr<XD>::B;
    a.y = (char *)a.y + m0 * a.ldy * ys;
    if (a.res) a.res = (const char *)a.res + m0 * a.ldy * ys;
  }
  // a fused norm reduces over the first 512 threads whatever the block size,
  // so its summation order (and the rounded row it stages) is the same at 8
  // and 16 waves per block, and the same as the persistent step's
  const uint32_t nthr = blockDim.x < 512 ? blockDim.x : 512;
  gemv_core<WT, XD, M, R, U, false, NK>(
      a, xs_raw, red, g, gridDim.x * nw, nthr, (int)(nthr >> 6), [] { return true; },
      [&](int m) { return (const void *)((const char *)a.x + (uint64_t)m * a.ldx * XDr<XD>::B); },
      [](uint32_t, const float (&)[R][M]) {}, (uint32_t)blockDim.x);
  pclk_end(a.clk, a.clk_cap);
}

// -------------------------------------------------------------------------
typedef void (*gemv_fn)(ThvmGemvArgs);

// U chunks per lane and row in flight.  A lane's chunk order is the same at any
// U, so the sums are the same bits; the tuning key u only chooses between 4 and 8
// at one row.
template <int WT, int XD, int M, int R, int U>
static gemv_fn pick_n(uint32_t norm) {
  return norm == 0 ? k_gemv<WT, XD, M, R, U, 0> : norm == 1 ? k_gemv<WT, XD, M, R, U, 1> : k_gemv<WT, XD, M, R, U, 2>;
}
template <int WT, int XD, int R, int U>
static gemv_fn pick_m(uint32_t M, uint32_t norm) {
  if constexpr (XD == XD_SUM4) {
    return M == 1 ? k_gemv<WT, XD, 1, R, U> : nullptr;   // one row only
  } else {
    switch (M) {
      case 1: return k_gemv<WT, XD, 1, R, U>;
      case 2: return pick_n<WT, XD, 2, R, 4>(norm);
      case 3: return pick_n<WT, XD, 3, R, 4>(norm);
      case 4: return pick_n<WT, XD, 4, R, 4>(norm);
      default: return nullptr;
    }
  }
}
template <int WT, int XD>
static gemv_fn pick_ru(uint32_t M, int R, int U, uint32_t norm) {
  if (R == 1) return U == 8 ? pick_m<WT, XD, 1, 8>(M, norm) : pick_m<WT, XD, 1, 4>(M, norm);
  return U == 8 ? pick_m<WT, XD, 2, 8>(M, norm) : pick_m<WT, XD, 2, 4>(M, norm);
}
gemv_fn GEMV_PICK(uint32_t M, int R, int U, uint32_t norm) { return pick_ru<GEMV_WT, GEMV_XD>(M, R, U, norm); }
