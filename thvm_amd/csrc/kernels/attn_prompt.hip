// attn_prompt.hip -- causal attention of a prompt chunk over the KV cache: T
// consecutive positions of each of B sequences, position L-1+t of a sequence
// attending to its cache rows [0, L+t) (the chunk's own rows are in the cache
// already).  16-bit caches of head dim 64 or 128; the decode split
// (k_attn_mf, attn.hip) runs one position per block and would read the cache
// once per position.
//
// Here the 16 columns of the MFMA tiles are 16 positions of one head, where the
// decode split has the query heads there; operand layouts and the log2-domain
// online softmax are those of k_attn_mf.  p keeps the 24 bits it has in the
// one-launch decode form (f32 there), as a sum of 16-bit terms, each the
// rounding of what the ones before leave: three in bf16 (8 bits each), two in
// fp16 (11 each, p scaled by 2^14 so that the second stays out of fp16's
// subnormals; the scale cancels in acc / l):
//   * a block is 16 positions x GH heads of one kv head (GH = 2 where G is
//     even: each K / V tile loaded serves both), 4 waves, the cache's 16-row
//     tiles round-robin over the waves with the next one in flight;
//   * a column's causal limit is its lane's own (column l % 16), so the mask is
//     one compare per score; the block stops at its last position's row;
//   * the waves meet once through LDS and the block writes the finished rows:
//     no partials, no second launch.
// Bound by latency at a few hundred positions (C4's 32 heads, 299 positions:
// 304 blocks); grid (position tiles, kv heads x G / GH, B), longest tiles first.
#include "attn_core.h"
#include "mfma_ops.h"
#include "launch.h"
#include <stdio.h>

#define AP_WAVES 4
#define AP_THREADS (AP_WAVES * 64)

template <int HD, int AT, int GH>
__global__ __launch_bounds__(AP_THREADS, 2) void k_attn_prompt(ThvmAttnArgs a) {
  static_assert(AT == AT_BF16 || AT == AT_F16, "16-bit caches");
  constexpr int XT = AT == AT_BF16 ? GX_BF16 : GX_F16;
  constexpr int KS = HD / 32, NC = HD / 8, PT = AT == AT_BF16 ? 3 : 2;   // PT: 16-bit terms of p
  constexpr float PS = AT == AT_BF16 ? 1.0f : 16384.0f;
  constexpr uint32_t EXP = AT == AT_BF16 ? 0x7f80u : 0x7c00u;              // all ones: infinite or NaN
  extern __shared__ __align__(16) float apl[];
  float(*const wacc)[GH * 16][HD + 4] = (float(*)[GH * 16][HD + 4])apl;      // [wave][head, position][d]
  __shared__ float wm[AP_WAVES][GH * 16], wl[AP_WAVES][GH * 16];
  const uint32_t T = a.T, G = a.H / a.Hkv, GP = G / GH;
  const uint32_t t0 = (gridDim.x - 1 - blockIdx.x) * 16u;
  const uint32_t kvh = blockIdx.y / GP, h0 = kvh * G + (blockIdx.y % GP) * GH, b = blockIdx.z;
  const int32_t pos = a.len[0] - 1;                       // the chunk's first position
  if (pos < 0) return;
  const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lc = lane & 15,
            lg = lane >> 4;
  // cache rows this block reads: those up to its last position's, inside the cache
  const int32_t r1 = min(pos + (int32_t)min(t0 + 16u, T), (int32_t)a.max_seq);
  const int32_t lim = pos + (int32_t)t0 + lc + 1;         // this column's rows
  const int nt = (r1 + 15) / 16;
  const uint64_t cbase = ((uint64_t)b * a.Hkv + kvh) * a.max_seq * HD * 2;
  const buf_t krs = buf_rsrc((const char *)a.kcache + cbase, a.max_seq * HD * 2);
  const buf_t vrs = buf_rsrc((const char *)a.vcache + cbase, a.max_seq * HD * 2);
  // q^T operands: column lc is position t0 + lc (past T: zeros)
  const buf_t qrs = buf_rsrc((const char *)a.q + (uint64_t)b * T * a.H * HD * 2, T * a.H * HD * 2);
  uint4 qb[GH][KS];
#pragma unroll
  for (int g = 0; g < GH; g++)
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
      qb[g][ks] = buf_ld16(qrs, t0 + lc < T ? (((t0 + lc) * a.H + h0 + g) * HD + 8 * lg + 32 * ks) * 2u : BUF_OOB);
  uint4 kb[2][KS], vb[2][4];
  auto issue = [&](int buf, int t) {
    const int32_t rk = 16 * t + lc, rv = 16 * t + 4 * lg;
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
      kb[buf][ks] = buf_ld16(krs, rk < r1 ? (uint32_t)(rk * HD + 8 * lg + 32 * ks) * 2 : BUF_OOB);
#pragma unroll
    for (int j = 0; j < 4; j++)
      vb[buf][j] = buf_ld16(vrs, rv + j < r1 && lc < NC ? (uint32_t)((rv + j) * HD + 8 * lc) * 2 : BUF_OOB);
  };
  const float qs = a.scale * LOG2E;
  float m[GH], l[GH];
  f32x4_t acc[GH][8];
#pragma unroll
  for (int g = 0; g < GH; g++) {
    m[g] = -INFINITY;
    l[g] = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; e++) acc[g][e] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  int tbad = -1;                                          // see tile: a masked tile with V that is not finite
  float pbad[GH][4] = {};
  auto tile = [&](int buf, int t) {
    const int32_t rb = 16 * t + 4 * lg;
    uint32_t pt[GH][PT][2];
    float p[GH][4];
#pragma unroll
    for (int g = 0; g < GH; g++) {
      f32x4_t sc = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ks++) sc = mfma16<XT>(kb[buf][ks], qb[g][ks], sc);
      float sv[4];
#pragma unroll
      for (int i = 0; i < 4; i++) sv[i] = rb + i < lim && rb + i < r1 ? sc[i] * qs : -INFINITY;
      float mx = fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3]));
      mx = fmaxf(mx, xor16_f(mx));
      mx = fmaxf(mx, xor32_f(mx));
      const float mn = fmaxf(m[g], mx);
      const float f = m[g] == -INFINITY ? 0.0f : fexp2(m[g] - mn);
#pragma unroll
      for (int i = 0; i < 4; i++) p[g][i] = sv[i] == -INFINITY ? 0.0f : fexp2(sv[i] - mn) * PS;
      l[g] = l[g] * f + ((p[g][0] + p[g][1]) + (p[g][2] + p[g][3]));
      m[g] = mn;
      if (__builtin_amdgcn_ballot_w64(f != 1.0f)) {
#pragma unroll
        for (int e = 0; e < 8; e++)
#pragma unroll
          for (int i = 0; i < 4; i++) acc[g][e][i] *= f;
      }
      // P^T operands: term k = rnd(p - the terms before), each difference exact
#pragma unroll
      for (int h = 0; h < 2; h++) {
        float x0 = p[g][2 * h], x1 = p[g][2 * h + 1];
#pragma unroll
        for (int k = 0; k < PT; k++) {
          pt[g][k][h] = AT == AT_BF16 ? pk_bf16(x0, x1) : pk_f16(x0, x1);
          x0 -= AT == AT_BF16 ? __uint_as_float(pt[g][k][h] << 16) : h2f((f16_t)(pt[g][k][h] & 0xffffu));
          x1 -= AT == AT_BF16 ? __uint_as_float(pt[g][k][h] & 0xffff0000u) : h2f((f16_t)(pt[g][k][h] >> 16));
        }
      }
    }
    uint32_t w[4][4] = {{vb[buf][0].x, vb[buf][0].y, vb[buf][0].z, vb[buf][0].w},
                        {vb[buf][1].x, vb[buf][1].y, vb[buf][1].z, vb[buf][1].w},
                        {vb[buf][2].x, vb[buf][2].y, vb[buf][2].z, vb[buf][2].w},
                        {vb[buf][3].x, vb[buf][3].y, vb[buf][3].z, vb[buf][3].w}};
    // A masked score is a zero p, but zero times a V that is not finite (an
    // overflow in a later position) is NaN: in the tiles that some column of the
    // block masks such values leave the products, and after the last tile the
    // columns that do see their rows add them one by one.  Those tiles are the
    // block's last two at most, so a wave's is its last: its p are the final ones.
    if (16 * t + 15 > pos + (int32_t)t0) {                // wave-uniform
      uint32_t bad = 0;
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const uint32_t lo = (w[j][k] & EXP) == EXP ? 0xffffu : 0u, hi = (w[j][k] >> 16 & EXP) == EXP ? 0xffff0000u : 0u;
          bad |= lo | hi;
          w[j][k] &= ~(lo | hi);
        }
      if (__builtin_amdgcn_ballot_w64(bad != 0)) {
        tbad = t;                                         // (the wave's last tile)
#pragma unroll
        for (int g = 0; g < GH; g++)
#pragma unroll
          for (int i = 0; i < 4; i++) pbad[g][i] = p[g][i];
      }
    }
#pragma unroll
    for (int e = 0; e < 8; e++) {
      // column 8 lc + e of rows 0..3: the low (e even) or high half of dword e/2
      const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;
      const uint32_t a01 = __builtin_amdgcn_perm(w[1][e >> 1], w[0][e >> 1], sel);
      const uint32_t a23 = __builtin_amdgcn_perm(w[3][e >> 1], w[2][e >> 1], sel);
#pragma unroll
      for (int g = 0; g < GH; g++) {
#pragma unroll
        for (int k = 0; k < PT; k++) acc[g][e] = mfma16x16<XT>(a01, a23, pt[g][k][0], pt[g][k][1], acc[g][e]);
      }
    }
  };
  // two register sets in flight; the loads past the block's rows read zeros
  __builtin_amdgcn_sched_barrier(0);
  issue(0, wv);
  __builtin_amdgcn_sched_barrier(0);
  issue(1, wv + AP_WAVES);
  __builtin_amdgcn_sched_barrier(0);
  for (int t = wv; t < nt; t += 2 * AP_WAVES) {
    tile(0, t);
    __builtin_amdgcn_sched_barrier(0);
    issue(0, t + 2 * AP_WAVES);
    __builtin_amdgcn_sched_barrier(0);
    if (t + AP_WAVES < nt) tile(1, t + AP_WAVES);         // wave-uniform
    __builtin_amdgcn_sched_barrier(0);
    issue(1, t + 3 * AP_WAVES);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (tbad >= 0) {                                        // wave-uniform
#pragma unroll 1
    for (int jj = 0; jj < 4; jj++)                        // rows 16 tbad + 4 jj + i: their p are in lane group jj
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int32_t r = 16 * tbad + 4 * jj + i;
        float pr[GH];
#pragma unroll
        for (int g = 0; g < GH; g++) pr[g] = __shfl(pbad[g][i], lc + 16 * jj);
#pragma unroll
        for (int q = 0; q < 4; q++) {                     // this lane's d = 8 (4 lg + q) + e
          const int mm = 4 * lg + q;
          const uint4 v = buf_ld16(vrs, r < r1 && r < lim && mm < NC ? (uint32_t)(r * HD + 8 * mm) * 2 : BUF_OOB);
          const uint32_t vw[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
          for (int e = 0; e < 8; e++) {
            const uint32_t h = e & 1 ? vw[e >> 1] >> 16 : vw[e >> 1] & 0xffffu;
            if ((h & EXP) != EXP) continue;
            const float x = AT == AT_BF16 ? __uint_as_float(h << 16) : h2f((f16_t)h);
#pragma unroll
            for (int g = 0; g < GH; g++) acc[g][e][q] += pr[g] * x;
          }
        }
      }
  }
#pragma unroll
  for (int g = 0; g < GH; g++) {
    l[g] += xor16_f(l[g]);
    l[g] += xor32_f(l[g]);
    if (lg == 0) { wm[wv][g * 16 + lc] = m[g]; wl[wv][g * 16 + lc] = l[g]; }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int mm = 4 * lg + i;                          // d = 8 mm + e
      if (mm < NC) {
        *(float4 *)&wacc[wv][g * 16 + lc][8 * mm] = make_float4(acc[g][0][i], acc[g][1][i], acc[g][2][i], acc[g][3][i]);
        *(float4 *)&wacc[wv][g * 16 + lc][8 * mm + 4] = make_float4(acc[g][4][i], acc[g][5][i], acc[g][6][i], acc[g][7][i]);
      }
    }
  }
  __syncthreads();
  for (int o = tid; o < GH * 16 * HD / 2; o += AP_THREADS) {
    const int r = o / (HD / 2), d = 2 * (o % (HD / 2)), g = r / 16;
    const uint32_t t = t0 + r % 16;
    if (t >= T) continue;
    float M = wm[0][r];
#pragma unroll
    for (int w = 1; w < AP_WAVES; w++) M = fmaxf(M, wm[w][r]);
    float s0 = 0.0f, s1 = 0.0f, lt = 0.0f;
#pragma unroll
    for (int w = 0; w < AP_WAVES; w++) {
      const float mw = wm[w][r], f = mw == -INFINITY ? 0.0f : fexp2(mw - M);
      const float2 v = *(const float2 *)&wacc[w][r][d];
      s0 += v.x * f;
      s1 += v.y * f;
      lt += f * wl[w][r];
    }
    const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
    const uint32_t pk = (uint32_t)act_bits<AT>(s0 * inv) | ((uint32_t)act_bits<AT>(s1 * inv) << 16);
    *(uint32_t *)((uint16_t *)a.out + (((uint64_t)b * T + t) * a.H + h0 + g) * HD + d) = pk;
  }
}

typedef void (*ap_fn)(ThvmAttnArgs);

extern "C" int thvm_k_attn_prompt(const ThvmAttnArgs *a, hipStream_t s, char *err, int errlen) {
  const int bf = a->cdt == THVM_DT_BF16;
  if (a->H == 0 || a->Hkv == 0 || a->H % a->Hkv || a->B == 0 || a->B > 65535 || a->T == 0 || a->max_seq == 0 ||
      (a->hd != 64 && a->hd != 128) || (!bf && a->cdt != THVM_DT_FP16) || a->qdt != a->cdt || a->odt != a->cdt) {
    snprintf(err, errlen, "attn_prompt: 16-bit caches, q and out of one type, hd 64 or 128 (H=%u Hkv=%u hd=%u T=%u)",
             a->H, a->Hkv, a->hd, a->T);
    return -1;
  }
  if ((uint64_t)a->T * a->H * a->hd * 2 >= (1ull << 31) || (uint64_t)a->max_seq * a->hd * 2 >= (1ull << 31)) {
    snprintf(err, errlen, "attn_prompt: a sequence's q rows or one head's cache rows of 2 GiB or more");
    return -1;
  }
  const uint32_t G = a->H / a->Hkv, GH = G % 2 ? 1 : 2;
  ap_fn f = a->hd == 128 ? (GH == 2 ? (bf ? k_attn_prompt<128, AT_BF16, 2> : k_attn_prompt<128, AT_F16, 2>)
                                    : (bf ? k_attn_prompt<128, AT_BF16, 1> : k_attn_prompt<128, AT_F16, 1>))
                         : (GH == 2 ? (bf ? k_attn_prompt<64, AT_BF16, 2> : k_attn_prompt<64, AT_F16, 2>)
                                    : (bf ? k_attn_prompt<64, AT_BF16, 1> : k_attn_prompt<64, AT_F16, 1>));
  const uint32_t lds = AP_WAVES * GH * 16 * (a->hd + 4) * 4, hy = a->H / GH;
  if (hy > 65535) { snprintf(err, errlen, "attn_prompt: %u heads", a->H); return -1; }
  if (lds > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void *)f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) { snprintf(err, errlen, "attn_prompt: hipFuncSetAttribute: %s", hipGetErrorString(e)); return -1; }
  }
  thvm_launch(true, true, f, dim3((a->T + 15) / 16, hy, a->B), dim3(AP_THREADS), lds, s, *a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { snprintf(err, errlen, "attn_prompt launch: %s", hipGetErrorString(e)); return -1; }
  return 0;
}
