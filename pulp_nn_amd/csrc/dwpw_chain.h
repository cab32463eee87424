// A run of depthwise + pointwise blocks whose stages give every one of sixteen waves at most one item: 16 channels of a strip, 64 pixels x
// 16 channels (tiles of up to 64 pixels and of 128, 192 or 256 channels, of up to 128 pixels and 128 channels).  The arithmetic and the tile of dwpw_kernel; what differs is that
// a block is straight-line code with the next block's loads in flight: the next depthwise layer's parameters are asked for behind the
// barrier in the middle of a block, the weights behind the multiply, the next pointwise layer's parameters behind the barrier at its end,
// all of them to LDS, and each is waited for half a block later.
//
// Bound: one workgroup per image and compute unit, four waves per SIMD.  Of the 8000 cycles a block of 64 pixels x 256 channels takes, the
// set-up of operands and constants is 900, the depthwise rows 1500, the multiply 1300, requantisation 900, requests for the next
// block 700, the rest waiting at the two barriers for the waves that share a SIMD with three others: instructions issued, some 450 a
// wave.  Five blocks of 8x8x256: 32.8 -> 19.9 us at batch 256, 31.9 -> 17.6 at batch 1 (with the depthwise stage on the vector ALU 6000 cycles of
// 14000, weights in operand layout and constants per wave 2500 to 4500 of requests).
#pragma once
#include "dwpw.h"

// LDS of the launch: the tile's, the pointwise layer's parameters, and a row that pixels past the last one are written to.
PULPNN_HD int dwpw_chain_spare(int tile_lds, int C) { return tile_lds + dwpw_par(C, (int)sizeof(bn_t), false).bytes; }
PULPNN_HD int dwpw_chain_lds(int tile_lds, int C) { return dwpw_chain_spare(tile_lds, C) + 1024; }

#define DWPW_CHAIN_KP 4  // slices of K whose weights are in LDS: all of them
template <int W>
__global__ __launch_bounds__(1024) void dwpw_chain_kernel(DwPwGeom g)
{
  extern __shared__ __attribute__((aligned(16))) unsigned char dwpw_lds[];
  typedef unsigned v4u __attribute__((ext_vector_type(4)));
  const DwPwTile &T = g.t;
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, lgrp = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const DwPwPlace at = dwpw_place<W>(T, blockIdx.x);
  unsigned char *xin = dwpw_lds + T.x_off;
  const int C = T.C, cgs = C / 16, nitems = cgs * T.nst, nblk = cgs << T.lpxb;

  // the wave's item of the depthwise stage and its block of the pointwise stage
  const int st = (int)fastdiv((unsigned)wave, T.d_n), ch = 16 * (wave - st * cgs), cf = wave >> T.lpxb, px0 = 64 * (wave & ((1 << T.lpxb) - 1));
  const bool dw_on = wave < nitems, pw_on = wave < nblk;

  unsigned char *wl = dwpw_lds + T.w_off + wave * (1024 * DWPW_CHAIN_KP);  // the wave's own weights: four slices of 16 rows of 64 bytes
  unsigned char *par_dw = dwpw_lds + T.par_off, *par_pw = dwpw_lds + T.lds;
  auto load_w = [&](DwPwBlockArg P) {
    typedef __attribute__((address_space(3))) void *lds_ptr_t;
    int ln = lane;  // (opaque: the address is computed when the loads are issued, not kept from block to block)
    asm volatile("" : "+v"(ln));
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)P->pw_w, 0, C * C, 0x00020000);
    const unsigned off = dwpw_w_lane(C, pw_on ? cf : 0, ln, false);
#pragma unroll
    for (int kk = 0; kk < DWPW_CHAIN_KP; kk++) {
      const DwPwWeight at = dwpw_w_slice(C, off, kk);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)(wl + 1024 * kk), 16, at.off, at.add, 0, 0);
    }
  };
  auto load_dw = [&](DwPwBlockArg P) {
    dwpw_par_load(par_dw, P->dw_wt, P->dw_bias, P->e_dw.k, P->e_dw.lambda, P->mode_dw == EPI_BN, C, wave, 16, lane);
  };
  auto load_pw = [&](DwPwBlockArg P) {
    dwpw_par_load(par_pw, nullptr, P->pw_bias, P->e_pw.k, P->e_pw.lambda, P->mode_pw == EPI_BN, C, wave, 16, lane);
  };
  load_dw(dwpw_block(0));
  load_w(dwpw_block(0));
  load_pw(dwpw_block(0));

  // ---- the first input -> LDS ----------------------------------------------------------------------------------------------
  {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(g.in + (dwpw_first_row<1>(T, at) * W) * C), 0, (dwpw_rows_in(T) * W) * C, 0x00020000);
    const int chunks = dwpw_chunks<W>(T);
    constexpr int UN = 2;
#pragma unroll 1
    for (int t0 = tid; t0 < chunks; t0 += 1024 * UN) {
      v4u v[UN];
      int to[UN];
#pragma unroll
      for (int u = 0; u < UN; u++) {
        const DwPwChunk c = dwpw_chunk<W, 1>(T, at, t0 + 1024 * u);
        to[u] = c.lds;
        v[u] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, c.off >= 0 ? (unsigned)c.off : 0x80000000u, 0, 0);
      }
#pragma unroll
      for (int u = 0; u < UN; u++)
        if (t0 + 1024 * u < chunks) *(v4i *)(xin + to[u]) = (v4i){(int)v[u].x, (int)v[u].y, (int)v[u].z, (int)v[u].w} ^ (int)0x80808080;
    }
  }

  // places that stay the same from block to block
  const DwPwLane n = dwpw_lane<W, 1>(T, dw_on ? st : 0, l16, min(lgrp, 2));
  const int src0 = T.x_off + n.x + ch, rowb = (W + 2) * T.pitch;
  const int step = 4096 << T.lpxb, a0 = DWPW_ACT_AT(false, C, step, px0 + l16, 16 * lgrp);
  // (pixels past the last one are written to a spare row)
  const int x0 = pw_on && px0 + lane < at.live ? T.x_off + dwpw_next_x<W>(T, px0 + lane) + 16 * cf : dwpw_chain_spare(T.lds, C) + 16 * lane;
  const int blocks = g.nblocks;
  // every block's pointers into the scalar cache now: a miss between two stages costs all waves a round trip to memory
  {
    int touched = 0;
    for (int j = 1; j < blocks; j++) {
      const DwPwBlockArg P = dwpw_block(j);
      touched ^= P->mode_pw ^ P->e_dw.shift ^ (int)(long long)P->dw_wt;
    }
    asm volatile("" ::"s"(touched));
  }
  __builtin_amdgcn_s_waitcnt(DWPW_WAIT_VM(0));
  dwpw_barrier();

  v4i acc[4];
  bn_t kk[4], ll[4];
  int form;
#pragma unroll 1
  for (int j = 0;; j++) {
    const DwPwBlockArg P = dwpw_block(j);
    const bool last = j + 1 == blocks;
    // ---- depthwise stage -----------------------------------------------------------------------------------------------
    {
      const int mode = P->mode_dw, shift = P->e_dw.shift;
      DwhChannels<1> c;
      const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
      const unsigned char *filter = par_dw + dwpw_par(C, (int)sizeof(bn_t), true).f + ((dw_on ? ch : 0) + l16) * 9 + min(lgrp, 2);
      v4i s = {0, 0, 0, 0};
#pragma unroll
      for (int fy = 0; fy < 3; fy++) {
        const int v = lgrp < 3 ? (int)filter[3 * fy] << (8 * (l16 & 3)) : 0;
#pragma unroll
        for (int d = 0; d < 4; d++) c.A[0][fy][d] = (l16 >> 2) == d ? v : 0;
        s = __builtin_amdgcn_mfma_i32_16x16x64_i8(c.A[0][fy], ones, s, 0, 0, 0);
      }
      const bool ks = dwpw_fold(par_dw, C, (dw_on ? ch : 0) + 4 * lgrp, s, mode, mode == EPI_MULT ? P->e_dw.mult : 1, c.kk[0], c.ll[0]);
      const int form = dwh_form(mode, shift, (bool)__all(ks), true);
      if (dw_on) {
        const unsigned char *src = dwpw_lds + src0;
        int px = n.px;
        auto next = [&]() {
          const v4i v = *(const v4i *)src;
          src += rowb;
          return v;
        };
        auto put = [&](unsigned v) {
          if (n.live) *(unsigned *)(dwpw_lds + DWPW_ACT_AT(false, C, step, px, ch) + 4 * lgrp) = v ^ 0x80808080u;
          px += W;
        };
        dwh_with_form(form, [&](auto f) { dwh_walk<1, decltype(f)::value>(c, shift, T.R, next, put); });
      }
    }
    __builtin_amdgcn_s_waitcnt(DWPW_WAIT_VM(0));  // weights and parameters of the pointwise stage, asked for before the depthwise stage
    dwpw_barrier();
    if (!last) load_dw(dwpw_block(j + 1));  // (everybody has read this block's)

    // ---- pointwise stage ---------------------------------------------------------------------------------------------------
    const int mode = P->mode_pw, shift = P->e_pw.shift;
    const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
    v4i wacc = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; s++) acc[s] = (v4i){0, 0, 0, 0};
    {
      const unsigned char *a = dwpw_lds + a0, *w = wl + l16 * 64 + ((lgrp ^ ((l16 >> 1) & 3)) << 4);
#pragma unroll
      for (int kk = 0; kk < DWPW_CHAIN_KP; kk++) {
        if (64 * kk < C) {
          v4i af[4];
          const v4i wf = *(const v4i *)(w + 1024 * kk);
#pragma unroll
          for (int s = 0; s < 4; s++) af[s] = *(const v4i *)(a + s * 1024);
          a += step;
          wacc = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf, ones, wacc, 0, 0, 0);
#pragma unroll
          for (int s = 0; s < 4; s++) acc[s] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf, af[s], acc[s], 0, 0, 0);
        }
      }
    }
    const bool ks = dwpw_fold(par_pw, C, (pw_on ? 16 * cf : 0) + 4 * lgrp, wacc, mode, mode == EPI_MULT ? P->e_pw.mult : 1, kk, ll);
    form = dwh_form(mode, shift, (bool)__all(ks), true);  // (C <= 256: |acc| < 2^23)
    if (last) break;
    // the next block's weights travel during the requantisation, the barrier and the next depthwise stage
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this block's have been read
    load_w(dwpw_block(j + 1));
    if (pw_on)
      dwh_with_form(form, [&](auto f) {
        unsigned v[4];
#pragma unroll
        for (int s = 0; s < 4; s++) v[s] = dwh_requant<decltype(f)::value>(acc[s], kk, ll, shift);
        *(v4i *)(dwpw_lds + x0) = dwh_pixels(v) ^ (int)0x80808080;
      });
    __builtin_amdgcn_s_waitcnt(DWPW_WAIT_VM(DWPW_CHAIN_KP));  // the next depthwise stage's parameters: all but the weights
    dwpw_barrier();
    load_pw(dwpw_block(j + 1));  // (everybody has read this block's)
  }
  if (pw_on) {
    const int shift = dwpw_block(blocks - 1)->e_pw.shift;
    dwh_with_form(form, [&](auto f) {
      unsigned v[4];
#pragma unroll
      for (int s = 0; s < 4; s++) v[s] = dwh_requant<decltype(f)::value>(acc[s], kk, ll, shift);
      const v4i p = dwh_pixels(v);
      if (px0 + lane < at.live) *(v4i *)(g.out + ((long long)at.b0 * T.Ho * W + px0 + lane) * C + 16 * cf) = p;
    });
  }
}
