// linear_skinny_kernel for rows of any length from 16 bytes on, at any address.
//
// The last chunk of a row is its LAST 16 bytes, so that no load leaves a tensor; the bytes the chunk before has counted
// already meet zeros in the weight operand.  The loads are the same in number, unaligned: a row length costs next to
// nothing, where the tiled kernel gathered byte by byte.  A kernel of its own: as one template with the aligned form, that
// one ran 4 % slower (1024 -> 4096, 64 rows: 6.06 / 6.31 us).
// Measured, whole calls, tiled kernel -> this: 1 row 1003 -> 1000 62.6 -> 4.5 us; 64 rows 1000 -> 1000 64.6 -> 5.4; 200 rows
// 2056 -> 2048 132 -> 10.6; 64 rows 4001 -> 3001 275 -> 29; 256 rows 3999 -> 4001 423 -> 102; 256 rows 72 -> 40 9.7 -> 4.4.
#pragma once
#include "linear_skinny.h"

template <int MODE>
__global__ __launch_bounds__(256) void linear_skinny_any_kernel(SkinnyGeom g, EpiArgs e)
{
  __shared__ v4i part[4][4][64];  // [wave][s][lane]: partial accumulators of the K parts
  __shared__ int wpart[4][64];    // partial weight-row sums
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, lgrp = lane >> 4;
  const int n0 = blockIdx.x * 16;  // this workgroup's 16 neurons
  const int KT = (g.K + 63) / 64;
  // block of 64 rows (blockIdx.y counts the row blocks that other workgroups of the same neurons take), part of K
  const int rb = blockIdx.y * (4 / g.kparts) + wave / g.kparts, kp = wave % g.kparts;
  const int mb = rb * 64;
  const int kt0 = KT * kp / g.kparts, kt1 = KT * (kp + 1) / g.kparts;
  const bool active = mb < g.M;

  // weight rows past N and K chunks past K are read from a valid address and zeroed
  const bool nok = n0 + l16 < g.N;
  const int8_t *wrow = g.w + (long long)min(n0 + l16, g.N - 1) * g.K;
  const uint8_t *arow[4];
#pragma unroll
  for (int s = 0; s < 4; s++) arow[s] = g.in + (long long)min(mb + 16 * s + l16, g.M - 1) * g.K;

  // the bytes of a row's last chunk that the chunk before does not hold
  v4i tail;
  const int skip = (16 - g.K % 16) % 16;
#pragma unroll
  for (int d = 0; d < 4; d++) tail[d] = skip <= 4 * d ? -1 : skip >= 4 * d + 4 ? 0 : (int)(0xffffffffu << (8 * (skip - 4 * d)));

  int wsum = 0;  // this lane's share of sum_k w[n0 + l16][k] over this wave's part of K
  v4i acc[4];
#pragma unroll
  for (int s = 0; s < 4; s++) acc[s] = (v4i){0, 0, 0, 0};
  if (active) {
    for (int kb = kt0; kb < kt1; kb += 4) {
      // four slices: all loads first
      v4i wf[4], af[4][4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int kt = min(kb + u, kt1 - 1);
        const int p = 64 * kt + 16 * lgrp;
        const int ko = p >= g.K ? 0 : min(p, g.K - 16);
        wf[u] = *(const v4i_u *)(wrow + ko);
#pragma unroll
        for (int s = 0; s < 4; s++) af[u][s] = *(const v4i_u *)(arow[s] + ko);
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int kt = kb + u;
        const bool ok = kt < kt1 && nok && 64 * kt + 16 * lgrp < g.K;
        if (!ok) wf[u] = (v4i){0, 0, 0, 0};
        if (64 * kt + 16 * lgrp + 16 > g.K) wf[u] &= tail;
        wsum = __builtin_amdgcn_sdot4(wf[u].x, 0x01010101, wsum, false);
        wsum = __builtin_amdgcn_sdot4(wf[u].y, 0x01010101, wsum, false);
        wsum = __builtin_amdgcn_sdot4(wf[u].z, 0x01010101, wsum, false);
        wsum = __builtin_amdgcn_sdot4(wf[u].w, 0x01010101, wsum, false);
#pragma unroll
        for (int s = 0; s < 4; s++)
          acc[s] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[u], af[u][s] ^ (int)0x80808080, acc[s], 0, 0, 0);
      }
    }
  }
  // ---- the K parts of a block of rows meet in LDS ---------------------------------------
  if (g.kparts > 1) {
#pragma unroll
    for (int s = 0; s < 4; s++) part[wave][s][lane] = acc[s];
    wpart[wave][lane] = wsum;
    __syncthreads();
    if (kp == 0) {
      for (int q = 1; q < g.kparts; q++) {
#pragma unroll
        for (int s = 0; s < 4; s++) acc[s] += part[wave + q][s][lane];
        wsum += wpart[wave + q][lane];
      }
    }
  }
  if (kp != 0 || !active) return;

  // ---- epilogue ---------------------------------------------------------------------------
  // acc[s][r] = neuron n0 + 4*lgrp + r of row mb + 16*s + l16
  int ws = wsum;
  ws += __shfl_xor(ws, 16);
  ws += __shfl_xor(ws, 32);  // every lane: sum of weight row n0 + l16
  int corr[4];
  bn_t kk[4], ll[4];
  bool ks = true;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int n = n0 + 4 * lgrp + r;
    corr[r] = 128 * __shfl(ws, 4 * lgrp + r);
    kk[r] = 0;
    ll[r] = 0;
    if (n < g.N) {
      if (g.bias) corr[r] += (MODE == EPI_OUT32) ? ((const int *)g.bias)[n] : (int)g.bias[n];
      if (MODE == EPI_BN) {
        kk[r] = e.k[n];
        ll[r] = e.lambda[n];
      }
    }
    ks = ks && bn_k_small(kk[r]);
  }
  const bool k_small = __all(ks);
  const bool acc24 = g.K <= 256;
  const bool vec4 = (g.N & 3) == 0 && ((uintptr_t)g.out & 3) == 0;
  constexpr int QM = MODE == EPI_OUT32 ? EPI_RAW : MODE;
#pragma unroll
  for (int s = 0; s < 4; s++) {
    const int m = mb + 16 * s + l16;
    if (m >= g.M) continue;
    const int a0 = acc[s][0] + corr[0], a1 = acc[s][1] + corr[1], a2 = acc[s][2] + corr[2], a3 = acc[s][3] + corr[3];
    const int nb = n0 + 4 * lgrp;
    if constexpr (MODE == EPI_OUT32) {
      int *o = (int *)g.out + (long long)m * g.N + nb;
      const int v[4] = {a0, a1, a2, a3};
#pragma unroll
      for (int r = 0; r < 4; r++)
        if (nb + r < g.N) o[r] = v[r];
    } else {
      const unsigned p = acc24 ? requant4<QM, true>(a0, a1, a2, a3, kk, ll, k_small, e.mult, e.shift)
                               : requant4<QM, false>(a0, a1, a2, a3, kk, ll, k_small, e.mult, e.shift);
      uint8_t *o = (uint8_t *)g.out + (long long)m * g.N + nb;
      if (vec4 && nb + 4 <= g.N) {
        *(unsigned *)o = p;
      } else {
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (nb + r < g.N) o[r] = (uint8_t)(p >> (8 * r));
      }
    }
  }
}
