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
// one wave only, straight to the wave's own part of LDS, a group of PF K steps ahead of the one it multiplies.  Four lanes fetch the 64
// bytes of a row's step: in MFMA operand layout, sixteen rows side by side, a load keeps the address unit 56 to 64 clocks
// instead of 16, and the layers of many channels were bound by that.  128 * sum(w) comes from one more MFMA per weight fragment against ones.
//
// Everything is asked for in one trip to memory, the input first; a thread walks over the pixels of the band with its chunk of a
// pixel, so a load's place costs it some fifteen instructions.  (Weights first, constants waited for before the input is asked for, each
// place from divisions: 2200 clocks until the constants were asked for, 1600 until the input was, of 11500 in all on 57x43 24 -> 40.)
//
// Bound: layers of up to a few MB, by the chain load -> LDS -> multiply -> store and the instructions of a wave in it; larger ones by
// the vector instructions around each MFMA and by LDS, which holds input, weights and with them the workgroups that share a compute
// unit.  Whole calls, weights in registers in operand layout and tiles for two workgroups a compute unit / now: 57x43 24 -> 40 stride 2 batch 32
// 9.8 / 6.7 us; 15x31 168 -> 16 batch 19 11.3 / 9.7; 56x56 100 -> 100 batch 16 25.9 / 16.7; 40x30 250 -> 250 stride 2 batch 60 115 / 47;
// 13x19 90 -> 192 5x5 batch 70 125 / 36; 24x27 168 -> 176 5x5 stride 2 batch 72 47.4 / 44.6; over 380 layers the mean is 0.90, two of them
// slower by more than 2 % (23x14 144 -> 35 batch 23 8.3 / 8.6, 37x19 48 -> 20 batch 22 5.7 / 5.9); over 60 others of 33 to 64 outputs 0.91, five of them slower by
// 2 to 7 % (10x38 224 -> 48 batch 32 11.4 / 12.3, 34x10 208 -> 62 batch 58 11.9 / 12.7, 15x54 48 -> 40 batch 163 16.8 / 17.6).  (The 128 x 64 tile with a byte gather,
// which these shapes took before: 19.3, 236 and 409 us for the first, the second and the last.)
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

// s_waitcnt vmcnt(n), n < 16; lgkmcnt(0)
#define BAND_WAIT_VM(n) (0x0F70 | (n))
#define BAND_WAIT_LDS 0xC07F

// TN: 16-channel groups per wave; TM: 16-pixel groups per wave; PF: K steps of a group of weights
template <int TN, int TM, int PF>
__global__ __launch_bounds__(256, TN * TM <= 4 ? 4 : TN * TM == 8 ? 3 : 2) void conv_band_kernel(BandGeom g, EpiArgs e)
{
  extern __shared__ __attribute__((aligned(16))) unsigned char band_lds[];
  typedef unsigned v4u __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) void *lds_ptr_t;
  // the launch's numbers at once and opaque (as in dw_mfma_kernel)
  asm volatile("" : "+s"(g.total), "+s"(g.nblocks), "+s"(g.xtiles), "+s"(g.bands), "+s"(g.in), "+s"(g.w), "+s"(g.bias), "+s"(g.N), "+s"(g.K),
               "+s"(g.H), "+s"(g.W), "+s"(g.Ci), "+s"(g.Ho), "+s"(g.Wo), "+s"(g.CG));
  asm volatile("" : "+s"(g.CP), "+s"(g.NK), "+s"(g.R), "+s"(g.PC), "+s"(g.IW), "+s"(g.WN), "+s"(g.cpp), "+s"(g.ppp), "+s"(g.in_bytes),
               "+s"(g.w_off), "+s"(g.sx), "+s"(g.sy), "+s"(e.k), "+s"(e.lambda), "+s"(g.mode));
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lgrp = lane >> 4;
  const int wave_n = wave & (g.WN - 1), wave_m = g.WN == 4 ? 0 : g.WN == 2 ? wave >> 1 : wave;

  const unsigned id = (unsigned)xcd_remap(blockIdx.x, g.total);
  const unsigned t1 = fastdiv(id, g.d_nb), t2 = fastdiv(t1, g.d_xt), b = fastdiv(t2, g.d_band);
  const int nch = 16 * TN * g.WN;                                    // channels of the workgroup
  const int n0 = (int)(id - t1 * g.nblocks) * nch;
  const int ox0 = (int)(t1 - t2 * g.xtiles) * g.PC, oy0 = (int)(t2 - b * g.bands) * g.R;
  const int pc = min(g.PC, g.Wo - ox0), rows = min(g.R, g.Ho - oy0);
  const int px = rows * pc;

  // ---- ask for the input's first part --------------------------------------------------------------------------------
  // A thread keeps its chunk of a pixel and walks over the pixels of the band, ppp a pass.  Offsets count from 16 bytes before the band's
  // first pixel, which may lie in the padding; what is outside the image is out of the buffer's range and reads as zeros.
  const int iy0 = oy0 * g.sy - g.pt, ix0 = ox0 * g.sx - g.pl;
  const int nr = (rows - 1) * g.sy + g.ky;
  const long long first = (long long)b * g.H * g.W * g.Ci + ((long long)iy0 * g.W + ix0) * g.Ci - 16;
  const __amdgpu_buffer_rsrc_t rsrc_x =
      __builtin_amdgcn_make_buffer_rsrc((void *)(g.in + first), 0, (int)min(g.in_bytes - first, 0x7fffffffll), 0x00020000);
  const bool near = g.Ci < 16 && first < 0;                   // chunks may begin in front of the tensor: loaded too late
  const int lo = (int)min(max(-first, 0ll), 0x7fffffffll);
  const int p0 = (int)fastdiv((unsigned)tid, g.d_cpp), c_thr = tid - p0 * g.cpp;
  const int passes = (int)fastdiv((unsigned)(nr * g.IW - 1), g.d_ppp) + 1;
  const int dup = 16 * g.CG - g.Ci;  // bytes of a pixel's last chunk that the one before it has too
  constexpr int UN = 4;
  v4u v[UN];
  int dst[UN], voff[UN];
  int row, col, c16;
  auto start = [&](int cb) {  // chunks cb .. cb + cpp - 1 of all pixels
    row = (int)fastdiv((unsigned)p0, g.d_iw);
    col = p0 - row * g.IW;
    c16 = cb + c_thr;
    if (p0 >= g.ppp || c16 >= g.CG) row = 1 << 20;
  };
  auto load = [&](int pass) {
#pragma unroll
    for (int u = 0; u < UN; u++) {
      if (pass + u >= passes) break;
      const bool in = row < nr && (unsigned)(iy0 + row) < (unsigned)g.H && (unsigned)(ix0 + col) < (unsigned)g.W;
      voff[u] = (row * g.W + col) * g.Ci + min(16 * c16, g.Ci - 16) + 16;
      dst[u] = row < nr ? (row * g.IW + col) * g.CP + 16 * c16 : -1;
      v[u] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_x, in ? (unsigned)(near ? max(voff[u], lo) : voff[u]) : 0xffffffffu, 0, 0);
      if (near && !in) voff[u] = lo;
      col += g.scol;
      row += g.srow;
      if (col >= g.IW) col -= g.IW, row++;
    }
  };
  start(0);
  load(0);

  // ---- ... the constants of the thread's channel -----------------------------------------------------------------------
  int p_bias = 0;
  bn_t p_k = 0, p_l = 0;  // (of batch-norm, and read in that mode alone)
  if (tid < nch && n0 + tid < g.N) {
    if (g.bias) p_bias = (int)g.bias[n0 + tid];
    if (g.mode == EPI_BN) {
      p_k = e.k[n0 + tid];
      p_l = e.lambda[n0 + tid];
    }
  }

  // ---- ... and the first two groups of weights, on their way to the wave's part of LDS --------------------------------------
  // Row i of fragment t is channel wn0 + (i/4)*4*TN + 4*t + i%4.  Four lanes fetch the four chunks of a row's step, 64 bytes side by side.
  const int wn0 = n0 + wave_n * 16 * TN;
  constexpr unsigned OOB = 0x90000000u;  // (out of range whatever a row's offset adds or takes away)
  const int ntaps = g.kx * g.ky, ngroups = (g.NK + PF - 1) / PF;
  unsigned char *wl = band_lds + g.w_off + wave * band_wbytes(TN, PF);
  const int wr = lane >> 2, wj = (lane & 3) ^ ((wr >> 1) & 3);
  unsigned nrow[TN];
#pragma unroll
  for (int t = 0; t < TN; t++) {
    const int n = wn0 + (wr >> 2) * (4 * TN) + 4 * t + (wr & 3);
    nrow[t] = n < g.N ? (unsigned)(n * g.K) : OOB;
  }
  int wtap = (int)fastdiv((unsigned)wj, g.d_cg), wc = wj - wtap * g.CG;  // the lane's tap and chunk in the next step that is asked for
  auto load_w = [&](int half) {
    const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc((void *)g.w, 0, (unsigned)g.N * (unsigned)g.K, 0x00020000);
#pragma unroll
    for (int p = 0; p < PF; p++) {
      const int ko = wtap * g.Ci + min(16 * wc, g.Ci - 16);
#pragma unroll
      for (int t = 0; t < TN; t++)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_w, (lds_ptr_t)(wl + 1024 * ((half * PF + p) * TN + t)), 16,
                                                 (int)(wtap < ntaps ? nrow[t] + (unsigned)ko : OOB), 0, 0, 0);
      wc += g.wc;
      wtap += g.wtap;
      if (wc >= g.CG) wc -= g.CG, wtap++;
    }
  };
  load_w(0);
  if (ngroups > 1) load_w(1);
  // fewer than 16 channels: the first chunks of channel 0 begin in front of the tensor, and are made from its first 16 bytes
  const bool w_near = g.Ci < 16 && wn0 == 0;
  v4i w_head = {0, 0, 0, 0};
  if (w_near) w_head = *(const v4i_u *)g.w;

  // ---- the tap table: LDS offset of chunk q of the filter; its lowest bit: a pixel's last chunk --------------------------------
  int *tab = (int *)(band_lds + g.tab_off);
  for (int q = tid; q < 4 * PF * ngroups; q += 256) {
    const int tap = (int)fastdiv((unsigned)q, g.d_cg), c = q - tap * g.CG;
    const int fy = (int)fastdiv((unsigned)tap, g.d_kx), fx = tap - fy * g.kx;
    tab[q] = tap < ntaps ? (fy * g.IW + fx) * g.CP + 16 * c + (c == g.CG - 1 ? 1 : 0) : 0;  // (chunks past the filter: zero weights)
  }
  // the lanes' pixels
  int base[TM];
#pragma unroll
  for (int s = 0; s < TM; s++) {
    const int p = min((wave_m * TM + s) * 16 + l16, px - 1);
    const int y = (int)fastdiv((unsigned)p, g.d_pc), x = g.R > 1 ? p - y * pc : p;
    base[s] = ((g.R > 1 ? y : 0) * g.sy * g.IW + x * g.sx) * g.CP;
  }
  // ones where a chunk holds a byte that counts: all of it, or the end of a pixel's last chunk
  v4i ones_last;
#pragma unroll
  for (int d = 0; d < 4; d++) ones_last[d] = (int)(0x01010101u & ~low_bytes(dup - 4 * d));
  __builtin_amdgcn_sched_barrier(0);

  // ---- constants and input -> LDS --------------------------------------------------------------------------------------------
  int *c_bias = (int *)(band_lds + g.c_off);
  bn_t *c_k = (bn_t *)(c_bias + nch), *c_l = c_k + nch;
  if (tid < nch) {
    c_bias[tid] = p_bias;
    c_k[tid] = p_k;
    c_l[tid] = p_l;
  }
  for (int cb = 0;;) {
    v4u keep;  // a pixel's last chunk: not the bytes that the chunk before it has
#pragma unroll
    for (int d = 0; d < 4; d++) keep[d] = c16 == g.CG - 1 ? ~low_bytes(dup - 4 * d) : 0xffffffffu;
    for (int pass = 0;;) {
#pragma unroll
      for (int u = 0; u < UN; u++) {
        if (pass + u >= passes) break;
        if (near && __any(voff[u] < lo))
          if (voff[u] < lo) {
            const v4i w = bytes_up((v4i){(int)v[u].x, (int)v[u].y, (int)v[u].z, (int)v[u].w}, lo - voff[u]);
            v[u] = (v4u){(unsigned)w.x, (unsigned)w.y, (unsigned)w.z, (unsigned)w.w};
          }
        if (dst[u] >= 0) *(v4u *)(band_lds + dst[u]) = (v[u] ^ 0x80808080u) & keep;
      }
      pass += UN;
      if (pass >= passes) break;
      load(pass);
    }
    cb += g.cpp;
    if (cb >= g.CG) break;
    start(cb);
    load(0);
  }
  // (not __syncthreads(), which would also wait for the weights, which only their wave reads)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(BAND_WAIT_LDS);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  // ---- multiply -----------------------------------------------------------------------------------------------------------
  v4i acc[TN][TM], wacc[TN];
#pragma unroll
  for (int t = 0; t < TN; t++) {
    wacc[t] = (v4i){0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < TM; s++) acc[t][s] = (v4i){0, 0, 0, 0};
  }
  const v4i ones_all = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
  const unsigned char *wfrag = wl + l16 * 64 + ((lgrp ^ ((l16 >> 1) & 3)) << 4);
  auto steps = [&](int half, int kk0) {
    int toff[PF];
#pragma unroll
    for (int p = 0; p < PF; p++) toff[p] = tab[4 * (kk0 + p) + lgrp];
    if (w_near && kk0 < 4) {
#pragma unroll
      for (int p = 0; p < PF; p++) {
        const int q = 4 * (kk0 + p) + wj, off = q * g.Ci + g.Ci - 16;
        if (wr == 0 && off < 0 && q < ntaps) *(v4i *)(wl + (half * PF + p) * TN * 1024 + 16 * lane) = bytes_up(w_head, -off);
      }
      asm volatile("" ::: "memory");
    }
#pragma unroll
    for (int p = 0; p < PF; p++) {
      v4i ones = ones_all;
      if (dup) {
#pragma unroll
        for (int d = 0; d < 4; d++) ones[d] = toff[p] & 1 ? ones_last[d] : ones_all[d];
      }
      v4i af[TM], wf[TN];
#pragma unroll
      for (int t = 0; t < TN; t++) wf[t] = *(const v4i *)(wfrag + ((half * PF + p) * TN + t) * 1024);
#pragma unroll
      for (int s = 0; s < TM; s++) af[s] = *(const v4i *)(band_lds + base[s] + (toff[p] & ~1));
#pragma unroll
      for (int t = 0; t < TN; t++) wacc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[t], ones, wacc[t], 0, 0, 0);
#pragma unroll
      for (int s = 0; s < TM; s++)
#pragma unroll
        for (int t = 0; t < TN; t++) acc[t][s] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[t], af[s], acc[t][s], 0, 0, 0);
    }
  };
  // a group is waited for behind the one that was asked for after it
  auto ready = [&](bool another) {
    if (another) __builtin_amdgcn_s_waitcnt(BAND_WAIT_VM(PF * TN));
    else __builtin_amdgcn_s_waitcnt(BAND_WAIT_VM(0));
    asm volatile("" ::: "memory");
  };
  auto again = [&](int half) {  // (the group that lies there has been read)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(BAND_WAIT_LDS);
    load_w(half);
  };
#pragma unroll 1
  for (int i = 0; i < ngroups; i += 2) {
    ready(i + 1 < ngroups);
    steps(0, i * PF);
    if (i + 1 >= ngroups) break;
    if (i + 2 < ngroups) again(0);
    ready(i + 2 < ngroups);
    steps(1, (i + 1) * PF);
    if (i + 3 < ngroups) again(1);
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
