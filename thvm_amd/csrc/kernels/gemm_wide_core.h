// gemm_wide_core.h -- the projections of many x rows: y[m,n] = sum_k x[m,k] W[n,k]
// on gfx950 MFMA for batches above 16 rows and for prompt chunks of hundreds of
// rows.  W is [N, K] in fp16 / bf16 / fp8-e4m3 (+ per-row f32 scale), row-major
// or in the tile layout of thvm_k_tile_w, x [M, K] bf16 or fp16, f32
// accumulation; the outputs are the GEMV's (store / residual / GELU / SwiGLU /
// q,k RoPE + KV append, with the same rounding points as epilogue.h).
//
// What bounds it: k_gemm (gemm.hip) gives each wave of a block its own K slice
// and so its own x, and every block reads all of x for the 16..64 weight rows
// it owns: at 64 rows the x reads from L2 are 8 times the weight bytes of the
// 14336-wide down projection (470 MB against 59).  Here the 8 waves of a block
// share one x tile in LDS, 4 along the weight rows by 2 along k, and K is split
// over blocks where the weight rows alone would not fill the chip, so a block
// reads only its K slice of x for 64 NT weight rows.
//   * tile: BM = 16 MT x rows by BN = 64 NT weight rows, waves w and w + 4 the
//     16-row groups w NT .. w NT + NT - 1 of the block, one on the even and one
//     on the odd 64-k steps; per step a wave reads 2 MT x operands from LDS for
//     2 NT MT MFMAs, and at the end the two halves of k meet through LDS;
//   * x chunks of 128 k (a step for each wave of a pair), two LDS buffers: the
//     next chunk is stored while this one is consumed (one barrier per chunk);
//     x and weights are both requested U = 4 chunks ahead (2 where the widest
//     tile's registers leave no more: x 8 MT, weights 4 NT x WB of them a chunk);
//   * sums in two levels: an MFMA chain runs over 4 chunks (16-bit weights: 1) and
//     is then added to the tile's sums.  Error against float64 of the f32 sums
//     (2-norm over the result's, 1e-7; K = 1024 .. 14336, K unsplit, the worst):
//                          fp8 W          bf16 W         fp16 W
//       one chain          0.74 .. 2.99   1.28 .. 5.31   1.48 .. 5.42
//       two levels         0.64 .. 1.16   0.76 .. 2.00   0.85 .. 2.03
//       k_gemm (8 slices)  0.68 .. 1.40   0.83 .. 2.59   0.95 .. 2.76
//       the GEMV           0.59 .. 0.83   0.67 .. 1.16   0.86 .. 2.03
//     It costs up to 4% (28672 x 4096 fp8, M = 512, tiled: 141 -> 147 us; M = 60
//     26.0 -> 26.1);
//   * rows padded by 16 bytes: the 16 rows of one operand read fall in
//     different banks;
//   * splits > 1: each block stores its f32 tile with system-scope stores and
//     counts itself on the tile's counter; the last one sums the tiles in split
//     order (whatever the arrival order: the result is the same bits every
//     run) and runs the epilogue;
//   * block order: blocks go to the 8 XCDs round-robin, so tile t of XCD c is
//     number c * per + t of the (n tile, m tile) list with the m tiles of one n
//     tile next to each other: they read the same weights through one L2.
//   * RMSNorm on x fused (NM, bf16 x) as in gemm.hip: rnd(x g[k]) is staged, the
//     sums of x^2 scale the finished rows.
#pragma once
#include "dev_common.h"
#include "../kern_api.h"
#include "epilogue.h"
#include "mfma_ops.h"
#include "coh.h"

#define GW_NWAVES 4                     /* waves along the weight rows   */
#define GW_KG 2                         /* waves along k: one 64-k step of a chunk each */
#define GW_THREADS (64 * GW_NWAVES * GW_KG)
#define GW_KC (64 * GW_KG)              /* k per x chunk                 */
#define GW_CTR_BYTES 8192u              /* 2048 tile counters            */
#define GW_XROW (GW_KC * 2 + 16)        /* bytes of an x row in LDS      */

// four 16-bit / f32 values of the activation type <-> floats
template <uint32_t DT>
__device__ __forceinline__ void act4_dec(const uint4 &q, float o[4]) {
  if (DT == THVM_DT_FP32) {
    o[0] = __uint_as_float(q.x); o[1] = __uint_as_float(q.y); o[2] = __uint_as_float(q.z); o[3] = __uint_as_float(q.w);
  } else if (DT == THVM_DT_BF16) {
    o[0] = __uint_as_float(q.x << 16); o[1] = __uint_as_float(q.x & 0xffff0000u);
    o[2] = __uint_as_float(q.y << 16); o[3] = __uint_as_float(q.y & 0xffff0000u);
  } else {
    o[0] = h2f((f16_t)(q.x & 0xffffu)); o[1] = h2f((f16_t)(q.x >> 16));
    o[2] = h2f((f16_t)(q.y & 0xffffu)); o[3] = h2f((f16_t)(q.y >> 16));
  }
}
template <uint32_t DT>
__device__ __forceinline__ float act_rnd(float v) {
  return DT == THVM_DT_BF16 ? rbf(v) : DT == THVM_DT_FP16 ? rh(v) : v;
}
template <uint32_t DT>
__device__ __forceinline__ uint32_t act_pk(float a, float b) {   // 16-bit types
  return DT == THVM_DT_BF16 ? (uint32_t)f2bf(a) | ((uint32_t)f2bf(b) << 16)
                            : (uint32_t)f2h(a) | ((uint32_t)f2h(b) << 16);
}
template <uint32_t DT>
__device__ __forceinline__ void act4_st(void *p, uint64_t i, const float v[4]) {
  if (DT == THVM_DT_FP32) *(float4 *)((float *)p + i) = make_float4(v[0], v[1], v[2], v[3]);
  else *(uint2 *)((uint16_t *)p + i) = make_uint2(act_pk<DT>(v[0], v[1]), act_pk<DT>(v[2], v[3]));
}
template <uint32_t DT>
__device__ __forceinline__ uint4 act4_ld(const void *p, uint64_t i) {
  if (DT == THVM_DT_FP32) return *(const uint4 *)((const float *)p + i);
  const uint2 q = *(const uint2 *)((const uint16_t *)p + i);
  return make_uint4(q.x, q.y, 0u, 0u);
}

// The epilogue of a wave's NT x MT tiles, four consecutive weight rows of one
// x row per lane and tile: 8-byte (f32: 16-byte) residual loads, all requested
// before the first is used, and stores.  The host sends only shapes here whose
// rows and strides are multiples of four and whose buffers are aligned for it;
// others take the scalar epilogue.
template <int MT, int NT, uint32_t DT>
__device__ __forceinline__ void wide_epilogue(const ThvmGemvArgs &a, const uint32_t nw, const uint32_t m0,
                                              const f32x4_t (&acc)[NT][MT], const int li, const int lg) {
  const uint32_t N = a.N, M = a.M;
  float v[NT][MT][4];
#pragma unroll
  for (int t = 0; t < NT; t++) {
    const uint32_t n = nw + 16u * t + 4u * lg;
    const uint32_t nc = n < N ? n : 0u;               // rows past N are never stored
    float4 s = make_float4(1.f, 1.f, 1.f, 1.f);
    if (a.scale) s = *(const float4 *)(a.scale + nc);
    float b[4] = {0.f, 0.f, 0.f, 0.f};
    if (a.bias) act4_dec<DT>(act4_ld<DT>(a.bias, nc), b);
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
      v[t][mt][0] = acc[t][mt][0] * s.x + b[0];
      v[t][mt][1] = acc[t][mt][1] * s.y + b[1];
      v[t][mt][2] = acc[t][mt][2] * s.z + b[2];
      v[t][mt][3] = acc[t][mt][3] * s.w + b[3];
    }
  }
#define WIDE_EACH(...)                                                    \
  _Pragma("unroll") for (int t = 0; t < NT; t++)                          \
  _Pragma("unroll") for (int mt = 0; mt < MT; mt++) {                     \
    const uint32_t n = nw + 16u * t + 4u * lg, m = m0 + 16u * mt + li;    \
    const bool ok = n < N && m < M;                                       \
    __VA_ARGS__                                                                 \
  }
  switch (a.epi) {
    case THVM_EPI_STORE:
      WIDE_EACH(if (ok) act4_st<DT>(a.y, (uint64_t)m * a.ldy + n, v[t][mt]);)
      break;
    case THVM_EPI_RESID: {
      uint4 rq[NT][MT];
      WIDE_EACH(rq[t][mt] = act4_ld<DT>(a.res, ok ? (uint64_t)m * a.ldy + n : 0u);)
      WIDE_EACH(
        float r[4]; act4_dec<DT>(rq[t][mt], r);
        float o[4] = {r[0] + act_rnd<DT>(v[t][mt][0]), r[1] + act_rnd<DT>(v[t][mt][1]),
                      r[2] + act_rnd<DT>(v[t][mt][2]), r[3] + act_rnd<DT>(v[t][mt][3])};
        if (ok) act4_st<DT>(a.y, (uint64_t)m * a.ldy + n, o);)
    } break;
    case THVM_EPI_GELU:
      WIDE_EACH(
        float o[4];
        _Pragma("unroll") for (int i = 0; i < 4; i++) o[i] = gelu_tanh_f(act_rnd<DT>(v[t][mt][i]));
        if (ok) act4_st<DT>(a.y, (uint64_t)m * a.ldy + n, o);)
      break;
    case THVM_EPI_SWIGLU:
      WIDE_EACH(
        const float h0 = silu_f(act_rnd<DT>(v[t][mt][0])) * act_rnd<DT>(v[t][mt][1]);
        const float h1 = silu_f(act_rnd<DT>(v[t][mt][2])) * act_rnd<DT>(v[t][mt][3]);
        const uint64_t i = (uint64_t)m * a.ldy + n / 2;
        if (ok) {
          if (DT == THVM_DT_FP32) *(float2 *)((float *)a.y + i) = make_float2(h0, h1);
          else *(uint32_t *)((uint16_t *)a.y + i) = act_pk<DT>(h0, h1);
        })
      break;
    case THVM_EPI_QKV_ROPE:
    case THVM_EPI_QKV: {
      const uint32_t hd = a.head_dim, Hq = a.n_heads * hd, Hk = a.n_kv_heads * hd;
      const int32_t pos = a.len[0] - 1;
      if (pos < 0 || (uint32_t)pos >= a.max_seq) break;
      const bool rope = a.epi == THVM_EPI_QKV_ROPE;
      float2 cs[NT][MT], sn[NT][MT];
      // row m is position pos + m % T of sequence m / T (T rows a sequence; a
      // speculative verify's rows are all one sequence's)
      const uint32_t T = a.spec ? M : a.seq ? a.seq : 1u;
      WIDE_EACH(
        const uint32_t pm = (uint32_t)pos + m % T;
        const bool rot = rope && ok && n < Hq + Hk && pm < a.max_seq;
        const uint64_t ti = rot ? (uint64_t)pm * (hd / 2) + (n % hd) / 2 : 0u;
        cs[t][mt] = make_float2(1.f, 1.f);
        sn[t][mt] = make_float2(0.f, 0.f);
        if (rope) {
          const float2 c = *(const float2 *)(a.rope_cos + ti); const float2 s = *(const float2 *)(a.rope_sin + ti);
          if (rot) { cs[t][mt] = c; sn[t][mt] = s; }
        })
      WIDE_EACH(
        const uint32_t pm = (uint32_t)pos + m % T; const uint32_t d = n % hd;
        const bool rot = rope && n < Hq + Hk;
        float x[4]; float o[4];
        _Pragma("unroll") for (int i = 0; i < 4; i++) { x[i] = act_rnd<DT>(v[t][mt][i]); o[i] = x[i]; }
        if (rot) {
          o[0] = x[0] * cs[t][mt].x - x[1] * sn[t][mt].x;
          o[1] = x[1] * cs[t][mt].x + x[0] * sn[t][mt].x;
          o[2] = x[2] * cs[t][mt].y - x[3] * sn[t][mt].y;
          o[3] = x[3] * cs[t][mt].y + x[2] * sn[t][mt].y;
        }
        if (ok && pm < a.max_seq) {
          if (n < Hq) {
            act4_st<DT>(a.y, (uint64_t)m * a.ldy + n, o);
          } else {
            const bool isk = n < Hq + Hk;
            const uint32_t off = isk ? n - Hq : n - Hq - Hk;
            const uint64_t ci = (((uint64_t)(m / T) * a.n_kv_heads + off / hd) * a.max_seq + pm) * hd + d;
            act4_st<DT>(isk ? a.kcache : a.vcache, ci, o);
          }
        })
    } break;
    default: break;
  }
#undef WIDE_EACH
}

template <int WT, int XT, int MT, int NT, int NM>
__global__ __launch_bounds__(GW_THREADS, 2) void k_gemm_wide(ThvmGemvArgs a) {
  extern __shared__ __align__(16) unsigned char xs[];      // [2][BM][GW_XROW]
  __shared__ float ssum[NM ? 16 * MT : 1];
  __shared__ uint32_t last;
  static_assert(!NM || XT == GX_BF16, "the fused norm stages bf16 x");
  // U chunks in flight (two where the tile's registers leave no more), F chunks a
  // chain, T chunks a turn of the loop
  constexpr int BM = 16 * MT, WB = WT == GW_FP8 ? 1 : 2, U = NT == 4 && MT == 4 ? 2 : 4;
  constexpr int F = WT == GW_FP8 ? 4 : 1, T = 4;
  constexpr int NI = BM * 16 / GW_THREADS;                 // 16-byte x pieces per thread and chunk
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane((tid >> 6) % GW_NWAVES), kg = __builtin_amdgcn_readfirstlane(tid >> 6) / GW_NWAVES;
  const uint32_t N = a.N, K = a.K, M = a.M, SP = a.splits, S = K / 64;
  const uint32_t CH = (S + GW_KG - 1) / GW_KG;             // chunks of K
  // this block's tile and split
  const uint32_t mtiles = (M + BM - 1) / BM, ntiles = (N + 64u * NT - 1) / (64u * NT), total = ntiles * mtiles * SP;
  const uint32_t per = (total + 7) / 8, id = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (blockIdx.x / 8 >= per || id >= total) return;        // block-uniform
  const uint32_t m0 = (id % mtiles) * BM, r1 = id / mtiles, sp = r1 % SP, n0 = (r1 / SP) * (64u * NT);
  const uint32_t tile = (r1 / SP) * mtiles + id % mtiles;
  const uint32_t c0 = CH * sp / SP, c1 = CH * (sp + 1) / SP, s0 = c0 * GW_KG, s1 = min(c1 * GW_KG, S);
  const uint32_t nw = n0 + wv * (16u * NT);                // this wave's first weight row

  const uint64_t wrow_b = (uint64_t)K * (WT == GW_FP8 ? 1 : 2);
  const bool tl = a.wtiled != 0;
  const uint32_t nend = tl ? ((N + 15u) & ~15u) : N;
  const uint32_t nrow = nw < nend ? min(nend - nw, 16u * NT) : 0u;
  const buf_t wrs = buf_rsrc((const char *)a.w + (nw < nend ? (uint64_t)nw * wrow_b : 0u), (uint32_t)(nrow * wrow_b));
  const uint32_t sstep = tl ? 1024u * WB : 64u * WB, jstep = tl ? 1024u : 16u;
  uint32_t wo[NT];
#pragma unroll
  for (int t = 0; t < NT; t++)
    wo[t] = tl ? (uint32_t)(t * S * WB * 1024u) + lane * 16u
               : (uint32_t)((16u * t + li) * wrow_b) + lg * 16 * WB;
  // x rows m0 .. of the tile; rows at or past M read zero
  const uint32_t xrows = min(M - m0, (uint32_t)BM);
  const buf_t xrs = buf_rsrc((const char *)a.x + (uint64_t)m0 * a.ldx * 2,
                             (uint32_t)(((uint64_t)(xrows - 1) * a.ldx + K) * 2));
  const buf_t grs = buf_rsrc(NM ? (const void *)a.norm_w : (const void *)a.x, NM ? K * 4u : 0u);

  // chained through the accumulator alone, a row's sum takes a rounding per 32 k
  // of its slice; so a chain starts anew every F chunks and is added to the sums
  // of the ones before.  F is where the error is least of what the registers
  // allow: 16-bit weights, whose products round more in a chain, fold every chunk,
  // which needs no second set of accumulators either (with it the widest tile
  // spilled: 4096 x 14336 bf16, M = 512, 172 -> 207 us)
  f32x4_t acc[NT][MT], ch[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int mt = 0; mt < MT; mt++) acc[t][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  uint4 wr[U][NT][WB];
  auto wload = [&](int u, uint32_t s) {
    const uint32_t so = s < s1 ? s * sstep : BUF_OOB;
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int j = 0; j < WB; j++) wr[u][t][j] = buf_ld_stream16(wrs, wo[t] + so + j * jstep);
  };
  // x piece i of a thread: row i*XRP + tid/16, 8 k at 8 (tid % 16) of the chunk
  constexpr int XRP = GW_THREADS / 16;
  const uint32_t xr = tid >> 4, xk = (tid & 15) * 8;
  const uint32_t kend = s1 * 64;
  struct XChunk { uint4 x[NI], g[2]; };
  XChunk xv[U];                                            // chunk c in xv[c % U]
  float ss[NI];
#pragma unroll
  for (int i = 0; i < NI; i++) ss[i] = 0.f;
  auto xload = [&](XChunk &xv, uint32_t k0) {
    const uint32_t k = k0 + xk;
    const bool live = k < kend;
#pragma unroll
    for (int i = 0; i < NI; i++)
      xv.x[i] = buf_ld16(xrs, live ? ((xr + XRP * i) * a.ldx + k) * 2u : BUF_OOB);
    if (NM) {
      xv.g[0] = buf_ld16(grs, live ? k * 4u : BUF_OOB);
      xv.g[1] = buf_ld16(grs, live ? k * 4u + 16u : BUF_OOB);
    }
  };
  auto xstore = [&](XChunk &xv, int buf) {
    if (NM) {
      const uint32_t gw[8] = {xv.g[0].x, xv.g[0].y, xv.g[0].z, xv.g[0].w, xv.g[1].x, xv.g[1].y, xv.g[1].z, xv.g[1].w};
#pragma unroll
      for (int i = 0; i < NI; i++) {
        const uint32_t q[4] = {xv.x[i].x, xv.x[i].y, xv.x[i].z, xv.x[i].w};
        uint32_t o[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const float lo = __uint_as_float(q[j] << 16), hi = __uint_as_float(q[j] & 0xffff0000u);
          ss[i] = fmaf(lo, lo, ss[i]);
          ss[i] = fmaf(hi, hi, ss[i]);
          o[j] = pk_bf16(lo * __uint_as_float(gw[2 * j]), hi * __uint_as_float(gw[2 * j + 1]));
        }
        xv.x[i] = make_uint4(o[0], o[1], o[2], o[3]);
      }
    }
#pragma unroll
    for (int i = 0; i < NI; i++)
      *(uint4 *)(xs + (size_t)buf * (BM * GW_XROW) + (xr + XRP * i) * GW_XROW + xk * 2) = xv.x[i];
  };
  auto compute = [&](int buf, int so, int u, bool first) {
    const unsigned char *xb = xs + (size_t)buf * (BM * GW_XROW) + li * GW_XROW + so * 128 + lg * 32;
    uint4 B[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int j = 0; j < 2; j++) B[mt][j] = *(const uint4 *)(xb + mt * (16 * GW_XROW) + j * 16);
#pragma unroll
    for (int t = 0; t < NT; t++) {
      uint4 A0, A1;
      if (WT == GW_FP8) {
        const uint4 q = wr[u][t][0];
        fp8x4_op<XT>(q.x, A0.x, A0.y);
        fp8x4_op<XT>(q.y, A0.z, A0.w);
        fp8x4_op<XT>(q.z, A1.x, A1.y);
        fp8x4_op<XT>(q.w, A1.z, A1.w);
      } else {
        A0 = wr[u][t][0];
        A1 = wr[u][t][WB - 1];
      }
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        if constexpr (F == 1) {
          const f32x4_t c = mfma16<XT>(A0, B[mt][0], f32x4_t{0.f, 0.f, 0.f, 0.f});
          acc[t][mt] += mfma16<XT>(A1, B[mt][1], c);
        } else {
          ch[t][mt] = mfma16<XT>(A0, B[mt][0], first ? f32x4_t{0.f, 0.f, 0.f, 0.f} : ch[t][mt]);
          ch[t][mt] = mfma16<XT>(A1, B[mt][1], ch[t][mt]);
        }
      }
    }
  };
  // the LDS writes of every wave, and only they, before the next reads
  auto meet = [&] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };
  auto fold = [&] {
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int mt = 0; mt < MT; mt++) acc[t][mt] += ch[t][mt];
  };
  static_assert(T % U == 0 && T % 2 == 0 && (F == 1 || F == T), "a turn is whole turns of the register sets and LDS buffers, and one chain");
  const uint32_t nch = (c1 - c0 + T - 1) / T * T;     // run T at a time (zeros past the slice)
  // x and weights are both requested U chunks ahead: a wave's loads return in
  // issue order, so the wait for an x chunk is a wait for every weight load
  // issued before it, and a late x load would drain the weights' window
  {
    XChunk x0;
    xload(x0, s0 * 64);
#pragma unroll
    for (int u = 0; u < U; u++) {
      xload(xv[(u + 1) % U], s0 * 64 + (u + 1) * GW_KC);
      wload(u, s0 + u * GW_KG + kg);
      __builtin_amdgcn_sched_barrier(0);
    }
    xstore(x0, 0);
  }
  for (uint32_t c = 0; c < nch; c += T) {
#pragma unroll
    for (int f = 0; f < T; f++) {
      const int u = f % U;
      const uint32_t s = s0 + (c + f) * GW_KG;        // the chunk's first step
      meet();
      xstore(xv[(u + 1) % U], (u + 1) & 1);           // the next chunk
      xload(xv[(u + 1) % U], s * 64 + (U + 1) * GW_KC);
      __builtin_amdgcn_sched_barrier(0);
      compute(u & 1, kg, u, f == 0);
      wload(u, s + kg + U * GW_KG);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (F > 1) fold();
  }
  if (NM) {
#pragma unroll
    for (int i = 0; i < NI; i++) {                    // a row's 16 lanes are one DPP row
      const float s = row16_sum(ss[i]);
      if ((tid & 15) == 0) ssum[xr + XRP * i] = s;
    }
    __syncthreads();
  }

  // the two k halves meet: each wave keeps MH x tiles (kg MH .. of the block's
  // MT) and hands the others to its partner through LDS
  constexpr int MH = MT / GW_KG;
  static_assert(GW_KG == 2 && MT % 2 == 0, "tiles are exchanged in halves");
  f32x4_t own[NT][MH];
  {
    __syncthreads();
    float4 *const ex = (float4 *)xs;                       // [KG][NWAVES][NT][MH][64]
    auto slot = [&](int g, int t, int q) { return ((((g * GW_NWAVES + wv) * NT + t) * MH + q) * 64) + lane; };
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int q = 0; q < MH; q++) {
        const f32x4_t give = kg ? acc[t][q] : acc[t][MH + q];
        own[t][q] = kg ? acc[t][MH + q] : acc[t][q];
        ex[slot(kg, t, q)] = make_float4(give[0], give[1], give[2], give[3]);
      }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int q = 0; q < MH; q++) {
        const float4 o = ex[slot(kg ^ 1, t, q)];
        const f32x4_t p = f32x4_t{o.x, o.y, o.z, o.w};
        own[t][q] = kg ? p + own[t][q] : own[t][q] + p;    // k order: step 0 of a chunk first
      }
  }
  const uint32_t mo = (uint32_t)kg * (16u * MH);           // first owned x row in the tile

  if (SP > 1) {
    // the workspace: one counter per tile at its head (the same place for every
    // shape: calls of other shapes share the workspace and must not write
    // there), the partial tiles [tile][split][wave][tiles][lane] float4, then
    // the rows' sums of x^2 [tile][split][BM]
    constexpr uint32_t TB = GW_NWAVES * NT * MT * 1024u;
    const uint64_t ssoff = GW_CTR_BYTES + (uint64_t)ntiles * mtiles * SP * TB;
    char *const tb = (char *)a.ws + GW_CTR_BYTES + (uint64_t)tile * SP * TB;
    char *const sb = (char *)a.ws + ssoff + (uint64_t)tile * SP * BM * 4;
    const uint32_t lo = (uint32_t)(kg * GW_NWAVES + wv) * (NT * MH * 1024u) + lane * 16u;
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int mt = 0; mt < MH; mt++) {
        const f32x4_t v = own[t][mt];
        coh_st16(tb, sp * TB + lo + (t * MH + mt) * 1024u,
                 make_uint4(__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])));
      }
    if (NM && tid < BM) coh_stf(sb, (sp * BM + tid) * 4u, ssum[tid]);
    vm_drain();
    __syncthreads();
    if (tid == 0) {
      uint32_t *ctr = (uint32_t *)a.ws + tile;
      const uint32_t old = __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last = old == SP - 1 ? 1u : 0u;
      if (last) __hip_atomic_exchange(ctr, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!last) return;                                // block-uniform
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int mt = 0; mt < MH; mt++) own[t][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (uint32_t q = 0; q < SP; q++) {
      uint4 pv[NT][MH];
#pragma unroll
      for (int t = 0; t < NT; t++)
#pragma unroll
        for (int mt = 0; mt < MH; mt++) pv[t][mt] = coh_ld16(tb, q * TB + lo + (t * MH + mt) * 1024u);
#pragma unroll
      for (int t = 0; t < NT; t++)
#pragma unroll
        for (int mt = 0; mt < MH; mt++) {
          own[t][mt][0] += __uint_as_float(pv[t][mt].x);
          own[t][mt][1] += __uint_as_float(pv[t][mt].y);
          own[t][mt][2] += __uint_as_float(pv[t][mt].z);
          own[t][mt][3] += __uint_as_float(pv[t][mt].w);
        }
    }
    if (NM) {
      if (tid < BM) {
        float s = 0.f;
        for (uint32_t q = 0; q < SP; q++) s += coh_ldf(sb, (q * BM + tid) * 4u);
        ssum[tid] = s;
      }
      __syncthreads();
    }
  }
  if (NM) {
#pragma unroll
    for (int mt = 0; mt < MH; mt++) {
      const float inv = 1.0f / sqrtf(ssum[mo + 16 * mt + li] * (1.0f / (float)K) + a.norm_eps);
#pragma unroll
      for (int t = 0; t < NT; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) own[t][mt][i] *= inv;
    }
  }
  if (a.vec4) {
    if (a.ydt == THVM_DT_BF16) wide_epilogue<MH, NT, THVM_DT_BF16>(a, nw, m0 + mo, own, li, lg);
    else if (a.ydt == THVM_DT_FP16) wide_epilogue<MH, NT, THVM_DT_FP16>(a, nw, m0 + mo, own, li, lg);
    else wide_epilogue<MH, NT, THVM_DT_FP32>(a, nw, m0 + mo, own, li, lg);
    return;
  }
  for (int t = 0; t < NT; t++)
    for (int mt = 0; mt < MH; mt++) {
      const uint32_t n = nw + 16u * t + 4u * lg, m = m0 + mo + 16u * mt + li;
      if (m >= M) continue;
      f32x4_t v = own[0][0];
#pragma unroll
      for (int q = 0; q < NT * MH; q++)
        if (q == t * MH + mt) v = own[q / MH][q % MH];
      const float p0[2][1] = {{v[0]}, {v[1]}}, p1[2][1] = {{v[2]}, {v[3]}};
      gemv_epilogue<2, 1>(a, n, p0, m);
      gemv_epilogue<2, 1>(a, n + 2, p1, m);
    }
}
