// Convolution of any channel count, filter and stride from a band of the input staged once in LDS.
//
// A workgroup computes a run of output pixels of one image (whole rows where they fit, else part of a row; a pointwise
// layer is one long row) times up to 64 * TN channels.  The input rows behind them are brought into LDS once, pixel by
// pixel, at a pitch of an odd number of 16-byte chunks, and every filter tap reads them from there: K is cut into
// 16-byte chunks (tap, 16 channels), four to an MFMA step, and the activation fragment of a step is one ds_read_b128 per
// lane at pixel + tap.  A pixel outside the image is 0x80 (a = 0 as a - 128): no masks, no bounds checks, no gather in
// the main loop, whatever the geometry.
//
// Channel counts that are no multiples of 16: the last chunk of a pixel holds its LAST 16 bytes, of which those that the
// chunk before already has are zero in LDS (they multiply whatever the weight fragment has there); the weight fragment
// is fetched the same way, so no load ever leaves the tensors.  With fewer than 16 channels the chunk of the very first
// pixel (and weight row) would start in front of its tensor: that one is shifted into place.
//
// The waves of a workgroup split the channels (WN of them; the others split the pixels), so a weight byte is fetched by
// one wave only: straight from global memory in MFMA operand layout, PF steps at a time, the next PF steps requested
// before the current ones are multiplied.  128 * sum(w) comes from one more MFMA per weight fragment against ones.
//
// Bound: layers of up to a few MB, by the latency of load -> LDS -> multiply -> store (57x43 24 -> 40: 15 MFMAs and 718 vector
// instructions a wave, which waits half of its time; constants are waited for before the input is asked for); larger ones by
// too few waves and the vector instructions around each MFMA (24x27 168 -> 176 5x5: 1.7 waves per SIMD, 6.6 vector instructions
// per MFMA, matrix cores 20 % and LDS 10 % busy).  Measured, whole calls, against the 128 x 64 tile with a byte gather that these
// shapes took: 57x43 24 -> 40 stride 2 batch 32 19.3 -> 9.4 us; 15x31 168 -> 16 batch 19 236 -> 11; 24x27 168 -> 176 5x5 stride 2 batch
// 72 409 -> 46; 21x36 56 -> 32 stride 2 batch 25 82 -> 7.5; 14x14 24 -> 48 batch 31 19 -> 6.6 (the call's host time).
#pragma once
#include <type_traits>

#include "conv_band_geom.h"
#include "igemm.h"

// the 16 bytes of v moved up by n bytes (0 < n < 16), zeros below
__device__ __forceinline__ v4i bytes_up(v4i v, int n)
{
  unsigned __int128 t = ((unsigned __int128)((unsigned long long)(unsigned)v.z | ((unsigned long long)(unsigned)v.w << 32)) << 64) |
                        ((unsigned long long)(unsigned)v.x | ((unsigned long long)(unsigned)v.y << 32));
  t <<= 8 * n;
  return (v4i){(int)(unsigned)t, (int)(unsigned)(t >> 32), (int)(unsigned)(t >> 64), (int)(unsigned)(t >> 96)};
}

// TN: 16-channel groups per wave; TM: 16-pixel groups per wave
template <int TN, int TM>
__global__ __launch_bounds__(256) void conv_band_kernel(BandGeom g, EpiArgs e)
{
  constexpr int PF = TN == 4 ? 2 : TN == 2 ? 4 : 8;  // K steps whose weights are in flight
  extern __shared__ __attribute__((aligned(16))) unsigned char band_lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lgrp = lane >> 4;
  const int wave_n = wave & (g.WN - 1), wave_m = wave / g.WN;

  const unsigned id = (unsigned)xcd_remap(blockIdx.x, g.total);
  const unsigned t1 = fastdiv(id, g.d_nb), t2 = fastdiv(t1, g.d_xt), b = fastdiv(t2, g.d_band);
  const int nch = 16 * TN * g.WN;                                    // channels of the workgroup
  const int n0 = (int)(id - t1 * g.nblocks) * nch;
  const int ox0 = (int)(t1 - t2 * g.xtiles) * g.PC, oy0 = (int)(t2 - b * g.bands) * g.R;
  const int pc = min(g.PC, g.Wo - ox0), rows = min(g.R, g.Ho - oy0);
  const int px = rows * pc;

  // ---- weight fragments: row i of fragment t is channel wn0 + (i/4)*4*TN + 4*t + i%4 -----------------------------
  const int wn0 = n0 + wave_n * 16 * TN;
  const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc((void *)g.w, 0, (unsigned)g.N * (unsigned)g.K, 0x00020000);
  const int nslots = g.kx * g.ky * g.CG;
  const int wrow = wn0 + (l16 >> 2) * (4 * TN) + (l16 & 3);
  v4i wf[2][PF][TN];
  auto load_w = [&](v4i (&wb)[PF][TN], int kk0) {
    typedef unsigned v4u __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int p = 0; p < PF; p++) {
      const int q = 4 * (kk0 + p) + lgrp;
      const int tap = (int)fastdiv((unsigned)q, g.d_cg), c16 = q - tap * g.CG;
      const int ko = tap * g.Ci + min(16 * c16, g.Ci - 16);
#pragma unroll
      for (int t = 0; t < TN; t++) {
        const int n = wrow + 4 * t, off = n * g.K + ko;
        const v4u v = __builtin_amdgcn_raw_buffer_load_b128(rsrc_w, (q < nslots && n < g.N) ? (unsigned)max(off, 0) : 0xffffffffu, 0, 0);
        wb[p][t] = (v4i){(int)v.x, (int)v.y, (int)v.z, (int)v.w};
        if (g.Ci < 16 && __any(off < 0))
          if (off < 0) wb[p][t] = bytes_up(wb[p][t], -off);
      }
    }
  };
  load_w(wf[0], 0);

  // ---- per-channel constants and the tap table -> LDS ---------------------------------------------------------------
  int *c_bias = (int *)(band_lds + g.c_off);
  bn_t *c_k = (bn_t *)(c_bias + nch), *c_l = c_k + nch;
  if (tid < nch) {
    const int n = n0 + tid;
    const bool ok = n < g.N;
    c_bias[tid] = (g.bias && ok) ? (int)g.bias[n] : 0;
    // (only read for batch-norm; written in every mode, which is the shorter code: 57x43 24 -> 40 9.38 us, 9.46 with a branch)
    c_k[tid] = g.mode == EPI_BN ? (ok ? e.k[n] : (bn_t)0) : g.mode == EPI_MULT ? (bn_t)e.mult : (bn_t)1;
    c_l[tid] = (g.mode == EPI_BN && ok) ? e.lambda[n] : (bn_t)0;
  }
  int *tab = (int *)(band_lds + g.tab_off);
  for (int q = tid; q < 4 * g.NK; q += 256) {
    const int tap = (int)fastdiv((unsigned)q, g.d_cg), c16 = q - tap * g.CG;
    const int fy = (int)fastdiv((unsigned)tap, g.d_kx), fx = tap - fy * g.kx;
    tab[q] = q < nslots ? (fy * g.IW + fx) * g.CP + 16 * c16 : 0;  // (slots past the filter: zero weights)
  }

  // ---- stage the input ------------------------------------------------------------------------------------------------
  {
    const int iy0 = oy0 * g.sy - g.pt, ix0 = ox0 * g.sx - g.pl;
    const int iw = (pc - 1) * g.sx + g.kx, nr = (rows - 1) * g.sy + g.ky;
    const int chunks = nr * g.IW * g.CG;
    const long long ibase = (long long)b * g.H * g.W * g.Ci;
    const int dup = 16 * g.CG - g.Ci;  // bytes of a pixel's last chunk that the one before it has too
    constexpr int UN = 4;
    for (int t0 = tid; t0 < chunks; t0 += 256 * UN) {
      v4i v[UN];
      int dst[UN], under[UN];
      unsigned ok[UN];
      bool last[UN];
#pragma unroll
      for (int u = 0; u < UN; u++) {
        const int t = min(t0 + 256 * u, chunks - 1);
        const int p = (int)fastdiv((unsigned)t, g.d_cg), c16 = t - p * g.CG;
        const int row = (int)fastdiv((unsigned)p, g.d_iw), col = p - row * g.IW;
        const int iy = iy0 + row, ix = ix0 + col;
        const bool in = (unsigned)iy < (unsigned)g.H && (unsigned)ix < (unsigned)g.W && col < iw;
        const long long off = in ? ibase + ((long long)iy * g.W + ix) * g.Ci + min(16 * c16, g.Ci - 16) : 0;
        v[u] = *(const v4i_u *)(g.in + max(off, 0ll));
        under[u] = off < 0 ? (int)-off : 0;
        ok[u] = in ? 0xffffffffu : 0u;
        last[u] = c16 == g.CG - 1;
        dst[u] = p * g.CP + 16 * c16;
      }
#pragma unroll
      for (int u = 0; u < UN; u++) {
        if (g.Ci < 16 && __any(under[u]))
          if (under[u]) v[u] = bytes_up(v[u], under[u]);
        v4i w;
#pragma unroll
        for (int d = 0; d < 4; d++) w[d] = (int)(((unsigned)v[u][d] & ok[u]) ^ 0x80808080u);
        if (dup) {
#pragma unroll
          for (int d = 0; d < 4; d++) w[d] &= last[u] ? (int)~low_bytes(dup - 4 * d) : -1;
        }
        if (t0 + 256 * u < chunks) *(v4i *)(band_lds + dst[u]) = w;
      }
    }
  }
  __syncthreads();

  // ---- multiply -----------------------------------------------------------------------------------------------------------
  v4i acc[TN][TM], wacc[TN];
  int base[TM];
#pragma unroll
  for (int t = 0; t < TN; t++) {
    wacc[t] = (v4i){0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < TM; s++) acc[t][s] = (v4i){0, 0, 0, 0};
  }
#pragma unroll
  for (int s = 0; s < TM; s++) {
    const int p = min((wave_m * TM + s) * 16 + l16, px - 1);
    const int y = (int)fastdiv((unsigned)p, g.d_pc), x = p - y * pc;
    base[s] = (y * g.sy * g.IW + x * g.sx) * g.CP;
  }
  // ones where a chunk holds a byte that counts: all of it, or the end of a pixel's last chunk
  const int dup = 16 * g.CG - g.Ci;
  v4i ones_last;
#pragma unroll
  for (int d = 0; d < 4; d++) ones_last[d] = (int)(0x01010101u & ~low_bytes(dup - 4 * d));
  const v4i ones_all = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
  auto steps = [&](v4i (&wb)[PF][TN], int kk0) {
#pragma unroll
    for (int p = 0; p < PF; p++) {
      if (kk0 + p < g.NK) {
        const int q = 4 * (kk0 + p) + lgrp;
        const int toff = tab[q];
        v4i ones = ones_all;
        if (dup) {
          const int c16 = q - (int)fastdiv((unsigned)q, g.d_cg) * g.CG;
          if (c16 == g.CG - 1) ones = ones_last;
        }
        v4i af[TM];
#pragma unroll
        for (int s = 0; s < TM; s++) af[s] = *(const v4i *)(band_lds + base[s] + toff);
#pragma unroll
        for (int t = 0; t < TN; t++) wacc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wb[p][t], ones, wacc[t], 0, 0, 0);
#pragma unroll
        for (int s = 0; s < TM; s++)
#pragma unroll
          for (int t = 0; t < TN; t++) acc[t][s] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wb[p][t], af[s], acc[t][s], 0, 0, 0);
      }
    }
  };
  for (int kk = 0; kk < g.NK; kk += 2 * PF) {
    if (kk + PF < g.NK) load_w(wf[1], kk + PF);
    steps(wf[0], kk);
    if (kk + 2 * PF < g.NK) load_w(wf[0], kk + 2 * PF);
    if (kk + PF < g.NK) steps(wf[1], kk + PF);
  }

  // ---- epilogue: acc[t][s][r] = channel cb + 4*t + r of pixel 16*s + l16 -----------------------------------------------
  const int cl = wave_n * 16 * TN + lgrp * 4 * TN, cb = n0 + cl;
  const bool acc24 = g.K <= 256;  // |acc| <= K * 255 * 128 + 128 < 2^23
  unsigned packed[TM][TN];
  auto requantise = [&](auto md) {
    constexpr int MODE = decltype(md)::value;
#pragma unroll
    for (int t = 0; t < TN; t++) {
      int corr[4];
      bn_t kk[4], ll[4];
      bool ks = true;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        kk[r] = MODE == EPI_BN ? c_k[cl + 4 * t + r] : (bn_t)0;
        ll[r] = MODE == EPI_BN ? c_l[cl + 4 * t + r] : (bn_t)0;
        ks = ks && bn_k_small(kk[r]);
        corr[r] = c_bias[cl + 4 * t + r] + 128 * wacc[t][r];
      }
      const bool k_small = __all(ks);
#pragma unroll
      for (int s = 0; s < TM; s++) {
        const int a0 = acc[t][s][0] + corr[0], a1 = acc[t][s][1] + corr[1];
        const int a2 = acc[t][s][2] + corr[2], a3 = acc[t][s][3] + corr[3];
        packed[s][t] = acc24 ? requant4<MODE, true>(a0, a1, a2, a3, kk, ll, k_small, e.mult, e.shift)
                             : requant4<MODE, false>(a0, a1, a2, a3, kk, ll, k_small, e.mult, e.shift);
      }
    }
  };
  if (g.mode == EPI_BN) requantise(std::integral_constant<int, EPI_BN>{});
  else if (g.mode == EPI_MULT) requantise(std::integral_constant<int, EPI_MULT>{});
  else requantise(std::integral_constant<int, EPI_RAW>{});
  uint8_t *ob = g.out + (((long long)b * g.Ho + oy0) * g.Wo + ox0) * g.N + cb;  // (R > 1: whole rows, one run of pixels)
#pragma unroll
  for (int s = 0; s < TM; s++) {
    const int p = (wave_m * TM + s) * 16 + l16;
    if (p >= px) continue;
    uint8_t *o = ob + (long long)p * g.N;
    if (cb + 4 * TN <= g.N) {
      if constexpr (TN == 4) *(v4i_u *)o = (v4i){(int)packed[s][0], (int)packed[s][1 % TN], (int)packed[s][2 % TN], (int)packed[s][3 % TN]};
      else if constexpr (TN == 2) *(v2i_u *)o = (v2i){(int)packed[s][0], (int)packed[s][1 % TN]};
      else *(i32_u *)o = (int)packed[s][0];
    } else {
#pragma unroll
      for (int c = 0; c < 4 * TN; c++)
        if (cb + c < g.N) o[c] = (uint8_t)(packed[s][c >> 2] >> (8 * (c & 3)));
    }
  }
}
