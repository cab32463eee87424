// Pointwise convolution with any number of input channels up to 512 and any number of output channels from 16 up: the
// scheme of pw_stream.h (weights resident in LDS in MFMA fragment order, pixels from memory straight into registers in
// the MFMA column-operand layout, two steps ahead, every wave a contiguous run of pixels) where rows are not made of
// whole 16-byte chunks or the channel count is none of pw_stream_kernel's.
//
// K tail: the last chunk of a pixel is its LAST 16 bytes, fetched with an unaligned load; the bytes the chunk before
// already has meet zero weights.  No load leaves the tensor (fewer than 16 channels: the chunk of the first pixels is
// shifted into place).  Channels: blocks of up to 256, zero weights past the last one; a step's bytes are gathered in a
// per-wave LDS tile and written in 16-byte pieces, the last piece of a pixel being its last 16 bytes.
//
// Bound: not HBM alone.  The three layers below move their bytes (K + N per pixel) at 2.4, 3.7 and 2.7 TB/s where a copy reaches
// 6.2; LDS is busy half of the time (weight fragments, the output tile; a fifth of that bank conflicts) and waves wait 38 to
// 52 % of theirs.  Measured, whole calls, against the tiled kernel whose operands were gathered byte
// by byte: 19x28 120 -> 424 batch 234 267 -> 26 us (68 MB); 56x23 304 -> 100 batch 234 100 -> 35 (122 MB); 63x26 9 -> 256
// batch 92 55 -> 14; 24x28 367 -> 176 batch 14 30 -> 13; 25x11 64 -> 136 batch 152 21 -> 7.0.
#pragma once
#include <type_traits>

#include "conv_band.h"
#include "pw_any_geom.h"

template <int KS, int NP, int MODE, int NW>
__global__ __launch_bounds__(64 * NW) void pw_any_kernel(PwAnyGeom g, EpiArgs e)
{
  constexpr int NC = 64 * NP;             // channels of a block, padded
  constexpr int OROW = PW_ANY_OROW(NP);   // (17 dwords more than a multiple of 64 banks: rows start in different banks)
  extern __shared__ __attribute__((aligned(16))) unsigned char pwa_lds[];
  int8_t *Wl = (int8_t *)pwa_lds;
  bn_t *kl = (bn_t *)(pwa_lds + NC * KS * 64);
  bn_t *ll = kl + NC;
  int *corr_l = (int *)(ll + NC);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lgrp = lane >> 4;
  unsigned char *ob = (unsigned char *)(corr_l + NC) + wave * (16 * OROW);

  // blocks of channels of the same pixels on the same XCD: they share the input through its L2
  const int blk = g.nblk > 1 ? ((int)blockIdx.x >> 3) % g.nblk : 0;
  const int wg = g.nblk > 1 ? ((int)blockIdx.x >> 3) / g.nblk * 8 + ((int)blockIdx.x & 7) : (int)blockIdx.x;
  const int n0 = blk * g.NB, nb = min(g.NB, g.N - n0);

  int px, px_end;
  pw_any_run(g, wg, wave, NW, &px, &px_end);
  int koff[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ks++) {
    const int k = ks * 64 + lgrp * 16;
    koff[ks] = k < g.K ? min(k, g.K - 16) : g.K < 16 ? g.K - 16 : 0;  // (chunks past K: zero weights)
  }
  // unconditional loads from clamped addresses
  auto load_a = [&](v4i (&a)[KS], int p0) {
    const long long m = max(min(p0 + l16, px_end - 1), 0);
    const long long row = m * g.K;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) a[ks] = *(const v4i_u *)(g.in + (KS == 1 ? max(row + koff[ks], 0ll) : row + koff[ks]));
  };
  v4i b0[KS], b1[KS], b2[KS];
  load_a(b0, px);
  load_a(b1, px + 16);

  // ---- weights and per-channel constants -> LDS ---------------------------------------------------------------------
  {
    constexpr int CHUNKS = NC * KS * 4, SB = 64 * NW, CH = (CHUNKS + SB - 1) / SB;
    constexpr int UN = CH < 8 ? CH : 8;
    for (int u0 = 0; u0 < CH; u0 += UN) {
      v4i wv[UN];
#pragma unroll
      for (int u = 0; u < UN; u++) {
        // LDS row R = ((p*KS + ks)*4 + t)*16 + i holds channel p*64 + (i/4)*16 + 4*t + i%4
        const int q = min(tid + SB * (u0 + u), CHUNKS - 1), R = q >> 2, c = q & 3;
        const int i = R & 15, t = (R >> 4) & 3, ks = (R / 64) % KS, p = R / (64 * KS);
        const int n = p * 64 + (i >> 2) * 16 + 4 * t + (i & 3), k = ks * 64 + 16 * c;
        const bool ok = n < nb && k < g.K;
        const long long off = ok ? (long long)(n0 + n) * g.K + min(k, g.K - 16) : 0;
        v4i v = *(const v4i_u *)(g.w + max(off, 0ll));
        if (KS == 1 && __any(off < 0))
          if (off < 0) v = bytes_up(v, (int)-off);
        const int dup = k - (g.K - 16);  // > 0: the first bytes of the chunk are the chunk before's
#pragma unroll
        for (int d = 0; d < 4; d++) v[d] &= ok ? (int)~low_bytes(dup - 4 * d) : 0;
        wv[u] = v;
      }
#pragma unroll
      for (int u = 0; u < UN; u++) {
        const int q = tid + SB * (u0 + u);
        if (q < CHUNKS) *(v4i *)&Wl[lds_off(q >> 2, q & 3)] = wv[u];
      }
    }
  }
  bool small = true;
  for (int n = tid; n < NC; n += 64 * NW) {
    const bool ok = n < nb;
    corr_l[n] = (g.bias && ok) ? (int)g.bias[n0 + n] : 0;
    if constexpr (MODE == EPI_BN) {
      kl[n] = ok ? e.k[n0 + n] : (bn_t)0;
      ll[n] = ok ? e.lambda[n0 + n] : (bn_t)0;
      small = small && bn_k_small(kl[n]);
    }
  }
  const bool k_small = __syncthreads_and(small);
  // corr = bias + 128 * sum_k w
  for (int tile = wave; tile < NP * 4; tile += NW) {
    const int p = tile / 4, t = tile % 4;
    v4i acc = {0, 0, 0, 0};
    const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      const v4i wf = *(const v4i *)&Wl[lds_off(((p * KS + ks) * 4 + t) * 16 + l16, lgrp)];
      acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf, ones, acc, 0, 0, 0);
    }
    if (l16 == 0) {
      v4i *c4 = (v4i *)&corr_l[p * 64 + lgrp * 16 + 4 * t];
      *c4 = *c4 + acc * 128;
    }
  }
  __syncthreads();

  // ---- stream pixels ----------------------------------------------------------------------------------------------------
  const int cpr = (nb + 15) / 16;
  const FastDiv d_cpr = blk + 1 == g.nblk ? g.d_cpr_last : g.d_cpr;
  auto process = [&](v4i (&a)[KS], int p0, auto nt) {
    constexpr bool NT = decltype(nt)::value;
    if constexpr (KS == 1) {
      if (g.K < 16) {  // the first pixels' chunk starts in front of the tensor
        const long long off = (long long)max(min(p0 + l16, px_end - 1), 0) * g.K + g.K - 16;
        if (__any(off < 0))
          if (off < 0) a[0] = bytes_up(a[0], (int)-off);
      }
    }
#pragma unroll
    for (int ks = 0; ks < KS; ks++) a[ks] ^= (int)0x80808080;
#pragma unroll 1
    for (int p = 0; p < NP; p++) {
      const int cb = p * 64 + lgrp * 16;
      // (an offset the compiler cannot see through: with one group it would read all weights before the pixel loop and
      // keep them in registers it does not have)
      int wofs = 0;
      if constexpr (NP == 1) asm volatile("" : "+s"(wofs));
      v4i acc[4];
#pragma unroll
      for (int ks = 0; ks < KS; ks++)
#pragma unroll
        for (int t = 0; t < 4; t++) {
          const v4i wf = *(const v4i *)&Wl[wofs + lds_off(((p * KS + ks) * 4 + t) * 16 + l16, lgrp)];
          acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf, a[ks], ks == 0 ? *(const v4i *)&corr_l[cb + 4 * t] : acc[t], 0, 0, 0);
        }
      unsigned packed[4];
#pragma unroll
      for (int t = 0; t < 4; t++) {
        bn_t kk[4], lam[4];
        if constexpr (MODE == EPI_BN) {
#pragma unroll
          for (int c = 0; c < 4; c++) {
            kk[c] = kl[cb + 4 * t + c];
            lam[c] = ll[cb + 4 * t + c];
          }
        }
        if (MODE == EPI_MULT && e.shift >= 16)
          packed[t] = requant4<MODE, KS <= 4, true>(acc[t][0], acc[t][1], acc[t][2], acc[t][3], kk, lam, k_small, e.mult, e.shift);
        else
          packed[t] = requant4<MODE, KS <= 4>(acc[t][0], acc[t][1], acc[t][2], acc[t][3], kk, lam, k_small, e.mult, e.shift);
      }
      int *o = (int *)(ob + l16 * OROW + cb);
#pragma unroll
      for (int t = 0; t < 4; t++) o[t] = (int)packed[t];
    }
    // piece idx of the step: 16 bytes of pixel idx / cpr; rows past the end of the run and pieces past the last are
    // redirected (same bytes to the same address): no branch, fixed store count
    const int last = px_end - 1 - p0;
    v4i v[NP];
    uint8_t *dst[NP];
#pragma unroll
    for (int r = 0; r < NP; r++) {
      const int idx = min(r * 64 + lane, 16 * cpr - 1);
      const int row0 = (int)fastdiv((unsigned)idx, d_cpr), row = min(row0, last);
      const int col = min(16 * (idx - row0 * cpr), nb - 16);
      const int *src = (const int *)(ob + row * OROW + (col & ~3));
      v[r] = (v4i){src[0], src[1], src[2], src[3]};
      if (g.NB & 3) {  // (one block of an odd number of channels: the last piece is not dword aligned)
        const int x = src[4], sh = col & 3;
        v[r] = (v4i){(int)__builtin_amdgcn_alignbyte((unsigned)v[r].y, (unsigned)v[r].x, sh), (int)__builtin_amdgcn_alignbyte((unsigned)v[r].z, (unsigned)v[r].y, sh),
                     (int)__builtin_amdgcn_alignbyte((unsigned)v[r].w, (unsigned)v[r].z, sh), (int)__builtin_amdgcn_alignbyte((unsigned)x, (unsigned)v[r].w, sh)};
      }
      dst[r] = g.out + (long long)(p0 + row) * g.N + n0 + col;
    }
#pragma unroll
    for (int r = 0; r < NP; r++) {
      if constexpr (NT) __builtin_nontemporal_store(v[r], (v4i_u *)dst[r]);
      else *(v4i_u *)dst[r] = v[r];
    }
  };
  auto stream = [&](auto nt) {
    for (; px < px_end; px += 16) {
      load_a(b2, px + 32);
      process(b0, px, nt);
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        b0[ks] = b1[ks];
        b1[ks] = b2[ks];
      }
    }
  };
  if (g.nt) stream(std::true_type{});
  else stream(std::false_type{});
}
