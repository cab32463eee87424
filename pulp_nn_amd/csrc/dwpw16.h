// Depthwise 3x3 at stride 2 + pointwise 1x1 in one kernel for few planes 16 pixels wide with 128 channels or more: the vector ALU takes
// the depthwise stage straight from memory.
//
// At stride 2 a tile's input is four times its output, so dwpw_kernel, which has it in LDS before it multiplies, is bound by getting it
// there: 16 x 16 pixels of 256 channels are five loads a thread, one round trip to memory after the other, and with 448 channels or more they come in slabs
// with barriers between.  Here a wave keeps its five input rows in registers, 64 channels of two output rows, and all channels of a tile are in
// flight at once: two items for each 64 channels, eight waves, tiles of 32 pixels, as many workgroups to a tile as give every compute unit one.
//
// The depthwise stage is the register-resident scheme of dw3x3_rows_kernel (depthwise.h): a lane quad loads a dword, its four channels, of four
// neighbouring pixels each and transposes it into four pixels per channel, v_dot4 on byte windows, requantised bytes transposed back.  The pointwise stage
// takes blocks of 32 pixels x 64 channels, weights straight from memory in operand layout, the first ones requested before the depthwise stage.
// Call by call, dwpw_kernel / here: 16x16x128 -> 256 batch 1 6.2 / 5.9 us, 16x16x256 -> 512 batch 1 8.0 / 7.2, batch 16 8.7 / 8.2, 16x16x512 batch 1
// 12.9 / 10.4, batch 64 17.1 / 15.2, 16x16x1024 batch 32 49.2 / 24.7; which calls come here, and both sides of the lines: dwpw_small16().
#pragma once
#include "depthwise.h"
#include "dwpw.h"

#define DWPW16_WAVES 8

struct DwPw16Geom {
  const uint8_t *in;      // HWC [B][H][16][C]
  uint8_t *out;           // HWC [B][Ho][8][Co]
  int M, C, H, Ho, Co;    // M: output pixels
  int nsplit;             // workgroups that share a tile, each computing a part of the output channels
  FastDiv d_ho;
  DwPwBlock blk;
};

// KP: 64-byte slices of K whose weights a wave holds at once
template <int KP>
__global__ __launch_bounds__(64 * DWPW16_WAVES) void dwpw16_kernel(DwPw16Geom g)
{
  constexpr int BP = DWPW16_PX, R = 2, NIN = 5, RD = 4, WO = 8;  // rows of an item, its input rows, dwords of a channel's row
  extern __shared__ __attribute__((aligned(16))) unsigned char dwpw_lds[];  // activation operand [C / 64][32 pixels][64 bytes], then bias, k, lambda
  typedef unsigned v4u __attribute__((ext_vector_type(4)));
  const DwPwBlock &P = g.blk;
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, lgrp = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tile = blockIdx.x / g.nsplit, part = blockIdx.x - tile * g.nsplit, m0 = tile * BP;
  const int KT = g.C / 64, NBT = (g.Co + 63) / 64, nb_per = (NBT + g.nsplit - 1) / g.nsplit;
  const int nb_lo = part * nb_per, nblk = max(min(NBT, nb_lo + nb_per) - nb_lo, 0), nch = 64 * nblk;
  int *c_bias = (int *)(dwpw_lds + BP * g.C);
  bn_t *c_k = (bn_t *)(c_bias + nch), *c_l = c_k + nch;
  const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};

  // weight fragment t of channel block nb: row i of it is channel 64 * nb + (i / 4) * 16 + 4 * t + i % 4, so that a lane ends up with 16
  // consecutive channels
  v4i wf[KP][4];
  auto load_w = [&](int nb, int kt0) {
    const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc((void *)P.pw_w, 0, (unsigned)g.Co * (unsigned)g.C, 0x00020000);
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int kk = 0; kk < KP; kk++) {
        const int n = 64 * nb + (l16 >> 2) * 16 + 4 * t + (l16 & 3), kb = 64 * (kt0 + kk) + 16 * lgrp;
        const v4u v = __builtin_amdgcn_raw_buffer_load_b128(rsrc_w, n < g.Co && kt0 + kk < KT ? (unsigned)(n * g.C + kb) : 0xffffffffu, 0, 0);
        wf[kk][t] = (v4i){(int)v.x, (int)v.y, (int)v.z, (int)v.w};
      }
  };
  int dw_w[3], dw_b;  // the nine filter bytes, bias
  bn_t dw_k, dw_l;
  auto load_dw = [&](int ch) {
    const int8_t *p = P.dw_wt + ch * 9;
    dw_w[0] = *(const i32_u *)p;
    dw_w[1] = *(const i32_u *)(p + 4);
    dw_w[2] = (int)p[8];
    dw_b = P.dw_bias ? (int)P.dw_bias[ch] : 0;
    dw_k = dw_l = 0;
    if (P.mode_dw == EPI_BN) {
      dw_k = P.e_dw.k[ch];
      dw_l = P.e_dw.lambda[ch];
    }
  };
  // ---- requests: the first item's filter, the constants of the channels out, the first weights (loads complete in this order) -----------
  load_dw((wave % KT) * 64 + lane);
  constexpr int NCI = 2;  // at most 1024 output channels
  int cb[NCI];
  bn_t ck[NCI], cl[NCI];
#pragma unroll
  for (int q = 0; q < NCI; q++) {
    const int c = tid + q * 64 * DWPW16_WAVES, n = 64 * nb_lo + c;
    const bool ok = c < nch && n < g.Co;
    cb[q] = P.pw_bias && ok ? (int)P.pw_bias[n] : 0;
    ck[q] = P.mode_pw == EPI_BN && ok ? P.e_pw.k[n] : (bn_t)0;
    cl[q] = P.mode_pw == EPI_BN && ok ? P.e_pw.lambda[n] : (bn_t)0;
  }
  if (wave < nblk) load_w(nb_lo + wave, 0);
#pragma unroll
  for (int q = 0; q < NCI; q++) {
    const int c = tid + q * 64 * DWPW16_WAVES;
    if (c < nch) {
      c_bias[c] = cb[q];
      c_k[c] = ck[q];
      c_l[c] = cl[q];
    }
  }

  // ---- depthwise stage: an item is 64 channels of two output rows -------------------------------------------------------------------------
  const unsigned sel1 = quad_sel1(lane), sel2 = quad_sel2(lane);
  for (int it = wave; it < 2 * KT; it += DWPW16_WAVES) {
    const int seg = it / KT, ch = (it - seg * KT) * 64 + lane, mi = m0 + seg * (R * WO);  // (both rows in one image)
    if (mi >= g.M) break;
    const int orow = mi / WO, b = (int)fastdiv((unsigned)orow, g.d_ho), oy0 = orow - b * g.Ho;
    unsigned row[NIN][RD];
    const uint8_t *src = g.in + (long long)b * g.H * 16 * g.C + (lane & 3) * g.C + (ch & ~3);
#pragma unroll
    for (int r = 0; r < NIN; r++) {
      const int iy = oy0 * 2 - 1 + r;
      const bool ok = (unsigned)iy < (unsigned)g.H;
      const uint8_t *rp = src + (long long)min(max(iy, 0), g.H - 1) * 16 * g.C;
#pragma unroll
      for (int d = 0; d < RD; d++) {
        const unsigned v = *(const unsigned *)(rp + (long long)(4 * d) * g.C);
        row[r][d] = ok ? v : 0u;
      }
    }
#pragma unroll
    for (int r = 0; r < NIN; r++)
#pragma unroll
      for (int d = 0; d < RD; d++) row[r][d] = quad_transpose4x4_perm(row[r][d], sel1, sel2) ^ 0x80808080u;
    if (it != wave) load_dw(ch);
    const unsigned w0 = (unsigned)dw_w[0], w1 = (unsigned)dw_w[1], w2 = (unsigned)dw_w[2];
    const unsigned wA[3] = {w0 & 0xffffffu, __builtin_amdgcn_alignbyte(w1, w0, 3) & 0xffffffu, (w1 >> 16) | ((w2 & 255u) << 16)};
    const unsigned wB[3] = {wA[0] << 8, wA[1] << 8, wA[2] << 8};
    const int wsum = __builtin_amdgcn_sdot4((int)w0, 0x01010101, __builtin_amdgcn_sdot4((int)w1, 0x01010101, dw_w[2], false), false);
    const int corr = 128 * wsum + dw_b, mult = P.e_dw.mult, shift = P.e_dw.shift;
    const bn_t kk = dw_k, ll = dw_l;
    const bool fastq = P.mode_dw == EPI_BN ? __all(bn_k_small(kk)) : shift >= 16;
    // (after the transpose back this lane holds channels ch & ~3 .. + 3 of column 4 * xg + lane % 4)
    const int c4 = ch & ~3, pl0 = seg * (R * WO) + (lane & 3);
    auto body = [&](auto md, auto fq) {
#pragma unroll
      for (int ro = 0; ro < R; ro++) {
#pragma unroll
        for (int xg = 0; xg < WO / 4; xg++) {
          constexpr int NS = 4;  // dwords of a window of four outputs
          int acc[4] = {corr, corr, corr, corr};
#pragma unroll
          for (int i = 0; i < 3; i++) {
            unsigned span[NS];
#pragma unroll
            for (int d = 0; d < NS; d++) {
              const int col = xg * 2 - 1 + d;  // dword column
              span[d] = col >= 0 && col < RD ? row[ro * 2 + i][col < 0 ? 0 : col >= RD ? RD - 1 : col] : 0x80808080u;
            }
            dw_tap<3, NS>(span, wA[i], wB[i], acc[0]);
            dw_tap<5, NS>(span, wA[i], wB[i], acc[1]);
            dw_tap<7, NS>(span, wA[i], wB[i], acc[2]);
            dw_tap<9, NS>(span, wA[i], wB[i], acc[3]);
          }
          const unsigned packed = requant4_same<decltype(md)::value, decltype(fq)::value>(acc[0], acc[1], acc[2], acc[3], kk, ll, mult, shift);
          const int pl = pl0 + ro * WO + 4 * xg;
          *(unsigned *)(dwpw_lds + (c4 >> 6) * (64 * BP) + pl * 64 + ((((c4 >> 4) & 3) ^ ((pl >> 1) & 3)) << 4) + (c4 & 15)) =
              quad_transpose4x4_perm(packed, sel1, sel2) ^ 0x80808080u;
        }
      }
    };
    if (P.mode_dw == EPI_BN) {
      if (fastq) body(std::integral_constant<int, EPI_BN>{}, std::true_type{});
      else body(std::integral_constant<int, EPI_BN>{}, std::false_type{});
    } else if (P.mode_dw == EPI_MULT) {
      if (fastq) body(std::integral_constant<int, EPI_MULT>{}, std::true_type{});
      else body(std::integral_constant<int, EPI_MULT>{}, std::false_type{});
    } else {
      body(std::integral_constant<int, EPI_RAW>{}, std::false_type{});
    }
  }
  __syncthreads();

  // ---- pointwise stage -------------------------------------------------------------------------------------------------------------------------
  for (int blk = wave; blk < nblk; blk += DWPW16_WAVES) {
    v4i acc[4][2], wacc[4];
#pragma unroll
    for (int t = 0; t < 4; t++) wacc[t] = acc[t][0] = acc[t][1] = (v4i){0, 0, 0, 0};
    for (int kt0 = 0; kt0 < KT; kt0 += KP) {
      if (kt0 || blk != wave) load_w(nb_lo + blk, kt0);
#pragma unroll
      for (int kk = 0; kk < KP; kk++) {
        if (kt0 + kk < KT) {
          const unsigned char *a = dwpw_lds + (kt0 + kk) * (64 * BP) + l16 * 64 + ((lgrp ^ ((l16 >> 1) & 3)) << 4);
          const v4i af[2] = {*(const v4i *)a, *(const v4i *)(a + 1024)};
#pragma unroll
          for (int t = 0; t < 4; t++) {
#pragma unroll
            for (int s = 0; s < 2; s++) acc[t][s] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[kk][t], af[s], acc[t][s], 0, 0, 0);
            wacc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[kk][t], ones, wacc[t], 0, 0, 0);
          }
        }
      }
    }
    // acc[t][s][r] = channel 64 * blk + 16 * lgrp + 4 * t + r of the workgroup's, pixel 16 * s + l16; wacc[t][r] = the sum of that channel's weights
    const int c0 = 64 * blk + 16 * lgrp, mult = P.e_pw.mult, shift = P.e_pw.shift;
    unsigned packed[2][4];
    auto requantise = [&](auto md) {
      constexpr int MODE = decltype(md)::value;
#pragma unroll
      for (int t = 0; t < 4; t++) {
        int corr[4];
        bn_t kk[4], ll[4];
        bool ks = true;
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int c = c0 + 4 * t + r;  // (constants of channels past the last one are zero)
          kk[r] = c_k[c];
          ll[r] = c_l[c];
          ks = ks && bn_k_small(kk[r]);
          corr[r] = c_bias[c] + 128 * wacc[t][r];
        }
        const bool k_small = __all(ks);
#pragma unroll
        for (int s = 0; s < 2; s++) {
          const int a0 = acc[t][s][0] + corr[0], a1 = acc[t][s][1] + corr[1], a2 = acc[t][s][2] + corr[2], a3 = acc[t][s][3] + corr[3];
          packed[s][t] = g.C <= 256 ? requant4<MODE, true>(a0, a1, a2, a3, kk, ll, k_small, mult, shift)   // |acc| <= K * 255 * 128 + 128 < 2^23
                                    : requant4<MODE, false>(a0, a1, a2, a3, kk, ll, k_small, mult, shift);
        }
      }
    };
    if (P.mode_pw == EPI_BN) requantise(std::integral_constant<int, EPI_BN>{});
    else if (P.mode_pw == EPI_MULT) requantise(std::integral_constant<int, EPI_MULT>{});
    else requantise(std::integral_constant<int, EPI_RAW>{});
#pragma unroll
    for (int s = 0; s < 2; s++) {
      const int m = m0 + 16 * s + l16, n = 64 * nb_lo + c0;
      if (m < g.M && n < g.Co) *(v4i *)(g.out + (long long)m * g.Co + n) = (v4i){(int)packed[s][0], (int)packed[s][1], (int)packed[s][2], (int)packed[s][3]};
    }
  }
}
