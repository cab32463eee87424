// Depthwise convolution (CHW in, HWC out) on the matrix cores, for any plane size, filter up to 8 columns wide,
// padding and stride.
//
// A depthwise layer is no contraction over channels, but one channel's filter is a Toeplitz matrix: sixteen adjacent
// output columns are T[16 x K] * window[K], where K runs over the ky input rows and the ND dwords of each row that
// sixteen columns can see, and T holds a filter tap at (column, row, column * sx + kx).  With the 64 bytes of K of one
// v_mfma_i32_16x16x64_i8 a 3x3 filter at stride 1 fits in one instruction (3 rows x 5 dwords), at stride 2 and 5x5
// filters in two.  The MFMA's sixteen columns are sixteen (row, column group) units of the tile, which all share the
// filter.  So a 16 x 16 block of one channel costs one or two MFMAs and four LDS dwords per lane instead of 48 v_dot4
// and the byte windows they need, and what is left for the vector ALU is the requantisation: 2.5 instructions per
// output.  The rows of T are built per channel from the filter bytes with one v_perm per dword (the selectors depend
// on the lane only).
//
// The accumulator layout gives a lane four neighbouring columns of ONE channel, so four channels computed one after the
// other are four bytes of each pixel: the transposition to HWC is the packing of the requantised bytes, no lane ever
// exchanges data with another.  The bytes are collected in LDS and written in runs of up to CB channels per pixel.
//
// Staging: one unaligned 16-byte load per lane from a row of the plane, at the column a chunk starts at (the row in LDS
// begins at image column x0 - pl), bytes outside the image replaced by zero, all stored as a ^ 0x80.  A thread keeps its
// (row, chunk) for all channels, so the masks are computed once.  The first and last bytes of the tensor are met by
// clamping the address and shifting.
//
// Bound: small layers by the chain input -> LDS, filters -> LDS, constants -> LDS, multiply, LDS -> store (35x29x72: 520 vector
// instructions a wave, most of them set-up, for 13 MFMAs, and 61 % of its time waiting), larger ones by the vector ALU (7x7x512
// batch 256: 1038 instructions a wave are two thirds of the kernel's 23.7 us).  Measured, whole calls, against the
// kernels it replaced (four outputs per lane with v_dot4 for 3x3, a byte loop for rows that are not whole dwords and for
// other filters): 3x3 on 35x29x72 batch 32 36.7 -> 8.5 us; 17x17x408 batch 85 38.3 -> 18.3 (20 MB); 5x5 on 8x23x32 batch
// 9 91 -> 7.0; 5x5 stride 2 on 60x11x416 batch 4 65 -> 7.7.
#pragma once
#include <type_traits>

#include "dw_mfma_geom.h"
#include "igemm.h"
#include "memops.h"
#include "requant.h"

// MODE: requantisation branch; NM: MFMAs per (channel, 16 units) = ceil(ky * ND / 16); CB: channels per workgroup
template <int CB, int NM, int MODE>
__global__ __launch_bounds__(256) void dw_mfma_kernel(DwmGeom g, EpiArgs e)
{
  extern __shared__ __attribute__((aligned(16))) unsigned char dwm_lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lgrp = lane >> 4;
  const DwmTile tile = dwm_tile<CB>(g, (unsigned)xcd_remap(blockIdx.x, g.total));
  const unsigned b = tile.b;
  const int c0 = tile.c0, xg0 = tile.xg0, oy0 = tile.oy0, ncb = tile.ncb, rows = tile.rows, wt = tile.wt;
  const int plane = g.H * g.W;
  const uint8_t *img = g.in + ((long long)b * g.CH + c0) * plane;

  // ---- stage the input rows -------------------------------------------------------------------------------------
  const int slots = g.NR * g.Q;
  const int iy0 = oy0 * g.sy - g.pt, x0 = 16 * xg0 * g.sx - g.pl;
  const int cpi = (int)fastdiv((unsigned)tid, g.d_nper);
  constexpr int UN = CB == 16 ? 4 : 8;  // loads in flight per thread
  auto stage = [&](auto edge) {
    constexpr bool EDGE = decltype(edge)::value;  // a load of this tile may leave the tensor
    const long long before = img - g.in, behind = g.in_bytes - before - 16;
    const int lo_lim = (int)max(-before, -(1ll << 30)), hi_lim = (int)min(behind, 0x7fffffffll);
    for (int s0 = 0; s0 < slots; s0 += g.nper) {
      const int slot = s0 + tid - cpi * g.nper;
      const int row = (int)fastdiv((unsigned)slot, g.d_q), q = slot - row * g.Q;
      const int x = x0 + 16 * q, iy = iy0 + row;
      const bool row_ok = (unsigned)iy < (unsigned)g.H;
      const int base = dwm_load_base(g, iy, x);
      if (cpi < g.cpar && slot < slots) {
        // bytes of the chunk inside the image
        unsigned mask[4];
#pragma unroll
        for (int d = 0; d < 4; d++) mask[d] = row_ok ? low_bytes(g.W - (x + 4 * d)) & ~low_bytes(-(x + 4 * d)) : 0u;
        for (int cb = cpi; cb < ncb; cb += UN * g.cpar) {
          v4i v[UN];
          int off[UN];
#pragma unroll
          for (int u = 0; u < UN; u++) {
            off[u] = min(cb + u * g.cpar, ncb - 1) * plane + base;
            v[u] = *(const v4i_u *)(img + (EDGE ? min(max(off[u], lo_lim), hi_lim) : off[u]));
          }
          unsigned char *dst = dwm_lds + row * g.pitch + 16 * q + cb * g.CS;
#pragma unroll
          for (int u = 0; u < UN; u++) {
            if constexpr (EDGE) {
              // the bytes were loaded up to 15 bytes too late (first bytes of the tensor) or too early (last ones)
              const int sh = min(max(off[u] - min(max(off[u], lo_lim), hi_lim), -16), 16);
              unsigned __int128 t = ((unsigned __int128)((unsigned long long)(unsigned)v[u].z | ((unsigned long long)(unsigned)v[u].w << 32)) << 64) |
                                    ((unsigned long long)(unsigned)v[u].x | ((unsigned long long)(unsigned)v[u].y << 32));
              if (sh > 0) t = sh < 16 ? t >> (8 * sh) : 0;
              if (sh < 0) t = sh > -16 ? t << (-8 * sh) : 0;
              v[u] = (v4i){(int)(unsigned)t, (int)(unsigned)(t >> 32), (int)(unsigned)(t >> 64), (int)(unsigned)(t >> 96)};
            }
            if (cb + u * g.cpar < ncb)
              *(v4i *)(dst + u * g.cpar * g.CS) =
                  (v4i){(int)(((unsigned)v[u].x & mask[0]) ^ 0x80808080u), (int)(((unsigned)v[u].y & mask[1]) ^ 0x80808080u),
                        (int)(((unsigned)v[u].z & mask[2]) ^ 0x80808080u), (int)(((unsigned)v[u].w & mask[3]) ^ 0x80808080u)};
          }
        }
      }
    }
  };
  if (dwm_edge(g, tile, img - g.in, iy0, x0)) stage(std::true_type{});
  else stage(std::false_type{});

  // ---- filter rows (8 bytes each, bytes past kx zero) and per-channel constants -> LDS ------------------------
  for (int t = tid; t < CB * g.ky; t += 256) {
    const int first = (c0 * g.ky + t) * g.kx;  // the filters of all channels back to back
    v2i w = {0, 0};
    if ((int)fastdiv((unsigned)t, g.d_ky) < ncb) {
      if (g.kx <= 4 && g.wt_bytes >= 4) {
        const int at = min(first, g.wt_bytes - 4);
        w.x = (int)(((unsigned)*(const i32_u *)(g.wt + at) >> (8 * (first - at))) & low_bytes(g.kx));
      } else {
        for (int j = 0; j < g.kx; j++) {
          const unsigned v = (unsigned)(uint8_t)g.wt[first + j] << (8 * (j & 3));
          if (j < 4) w.x |= (int)v;
          else w.y |= (int)v;
        }
      }
    }
    *(v2i *)(dwm_lds + g.w_off + t * 8) = w;
  }
  int *c_bias = (int *)(dwm_lds + g.c_off);
  bn_t *c_k = (bn_t *)(c_bias + CB), *c_l = c_k + CB;
  if (tid < CB) {
    const bool ok = tid < ncb;
    c_bias[tid] = (g.bias && ok) ? (int)g.bias[c0 + tid] : 0;
    if (MODE == EPI_BN) {
      c_k[tid] = ok ? e.k[c0 + tid] : (bn_t)0;
      c_l[tid] = ok ? e.lambda[c0 + tid] : (bn_t)0;
    }
  }

  // ---- lane constants: dword d = 16 mm + 4 lgrp + i of K is dword d % ND of filter row d / ND -----------------
  int boff[NM][4], wrow[NM][4];
  unsigned sel[NM][4];
#pragma unroll
  for (int mm = 0; mm < NM; mm++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int d = 16 * mm + 4 * lgrp + i, r = (d * g.rND) >> 16, xd = d - r * g.ND;
      const bool ok = r < g.ky;
      boff[mm][i] = ok ? r * g.pitch + 4 * xd : 0;
      wrow[mm][i] = ok ? 8 * r : 0;
      // this dword holds filter columns t .. t + 3 of the row; v_perm selectors: byte 0 .. 7 of the row, 12 = zero
      const int t = ok ? min(max(4 * xd - l16 * g.sx, -4), 8) + 4 : 0;
      const unsigned lo = t >= 4 && t < 8 ? 0x03020100u : t >= 8 && t < 12 ? 0x07060504u : 0x0c0c0c0cu;
      const unsigned hi = t < 4 ? 0x03020100u : t < 8 ? 0x07060504u : 0x0c0c0c0cu;
      sel[mm][i] = __builtin_amdgcn_alignbyte(hi, lo, t & 3);
    }
  __syncthreads();

  // (an output pixel takes one dword more than its channels in LDS: a store's lanes are multiples of four pixels apart)
  constexpr int PP = CB + 4;
  // ---- multiply ---------------------------------------------------------------------------------------------------
  const int units = rows * g.XT, shift = e.shift;
  const v4i b64 = {0x40404040, 0x40404040, 0x40404040, 0x40404040};
  for (int qd = wave; qd < (ncb + 3) / 4; qd += 4) {
    v4i a[4][NM];
    int corr[4];
    bn_t kk[4], ll[4];
    bool ks = true;
#pragma unroll
    for (int cc = 0; cc < 4; cc++) {
      const unsigned char *wl = dwm_lds + g.w_off + (4 * qd + cc) * g.ky * 8;
      v4i s = {0, 0, 0, 0};
#pragma unroll
      for (int mm = 0; mm < NM; mm++) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const v2i w = *(const v2i *)(wl + wrow[mm][i]);
          a[cc][mm][i] = (int)__builtin_amdgcn_perm((unsigned)w.y, (unsigned)w.x, sel[mm][i]);
        }
        // 128 * (sum of the filter), in every element
        s = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[cc][mm], b64, s, 0, 0, 0);
        s = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[cc][mm], b64, s, 0, 0, 0);
      }
      corr[cc] = c_bias[4 * qd + cc] + s[0];
      if (MODE == EPI_BN) {
        kk[cc] = c_k[4 * qd + cc];
        ll[cc] = c_l[4 * qd + cc];
      } else {
        kk[cc] = MODE == EPI_MULT ? (bn_t)e.mult : (bn_t)1;
        ll[cc] = 0;
      }
      ks = ks && bn_k_small(kk[cc]);
      // k * (acc + corr) + lambda = k * acc + (k * corr + lambda), exact in the wrapping arithmetic of the type
#if PULPNN_BN_BITS == 64
      if (MODE == EPI_BN) ll[cc] = (bn_t)((unsigned long long)kk[cc] * (unsigned long long)(long long)corr[cc] + (unsigned long long)ll[cc]);
      else
#endif
        ll[cc] = (bn_t)(int)((unsigned)kk[cc] * (unsigned)corr[cc] + (unsigned)ll[cc]);
    }
    auto tiles = [&](auto fast) {
      constexpr bool FAST = decltype(fast)::value;  // BN: k fits 24 (64-bit build: 32) bits; MULT: shift >= 16
      for (int u0 = 0; u0 < units; u0 += 16) {
        const int u = min(u0 + l16, units - 1);
        const int y = (int)fastdiv((unsigned)u, g.d_xg), xg = u - y * g.XT;
        const unsigned char *src = dwm_lds + (4 * qd) * g.CS + y * g.sy * g.pitch + xg * 16 * g.sx;
        int v[4][4];
#pragma unroll
        for (int cc = 0; cc < 4; cc++) {
          v4i acc = {0, 0, 0, 0};
#pragma unroll
          for (int mm = 0; mm < NM; mm++) {
            v4i bf;
#pragma unroll
            for (int i = 0; i < 4; i++) bf[i] = *(const int *)(src + cc * g.CS + boff[mm][i]);
            acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[cc][mm], bf, acc, 0, 0, 0);
          }
#pragma unroll
          for (int i = 0; i < 4; i++) {
            if constexpr (MODE == EPI_BN && PULPNN_BN_BITS == 64) {
              if constexpr (FAST) {
                const long long t = (long long)(int)kk[cc] * (long long)acc[i] + (long long)ll[cc];
                v[cc][i] = shift >= 32 ? (int)(t >> 32) : (int)__builtin_amdgcn_alignbit((unsigned)(t >> 32), (unsigned)t, shift);
              } else {
                const unsigned long long t = (unsigned long long)kk[cc] * (unsigned long long)(long long)acc[i] + (unsigned long long)ll[cc];
                v[cc][i] = (int)(unsigned)(unsigned long long)((long long)t >> shift);
              }
            } else if constexpr (MODE == EPI_BN && !FAST) {
              v[cc][i] = (int)((unsigned)kk[cc] * (unsigned)acc[i] + (unsigned)ll[cc]);
            } else {
              v[cc][i] = __mul24(acc[i], (int)kk[cc]) + (int)ll[cc];
              if (MODE == EPI_MULT && !FAST) v[cc][i] = (int)(short)(v[cc][i] >> shift);
            }
          }
        }
        // what is left of the shift
        const int sh = (MODE == EPI_BN && PULPNN_BN_BITS == 64) ? (FAST && shift >= 32 ? shift - 32 : 0) : (MODE == EPI_MULT && !FAST) ? 0 : shift;
        if (u0 + l16 < units) {
          unsigned char *dst = dwm_lds + g.o_off + (y * wt + 16 * xg + 4 * lgrp) * PP + 4 * qd;
#pragma unroll
          for (int i = 0; i < 4; i++)
            if (16 * xg + 4 * lgrp + i < wt) *(unsigned *)(dst + i * PP) = ashr_sat_pack4(v[0][i], v[1][i], v[2][i], v[3][i], sh);
        }
      }
    };
    if (MODE == EPI_RAW || (MODE == EPI_BN ? __all(ks) : shift >= 16)) tiles(std::true_type{});
    else tiles(std::false_type{});
  }
  __syncthreads();

  // ---- HWC out: the channels of a pixel in pieces of 16 ---------------------------------------------------------
  {
    constexpr int NCH = CB / 16;
    const int px = rows * wt, ch = 16 * (tid % NCH), n = ncb - ch;
    uint8_t *ob = g.out + ((long long)b * g.Ho * g.Wo + (long long)oy0 * g.Wo + 16 * xg0) * g.CH + c0 + ch;
    if (n > 0)
      for (int p = tid / NCH; p < px; p += 256 / NCH) {
        const int y = dwm_out_row(g, tile, p);
        const int *src = (const int *)(dwm_lds + g.o_off + p * PP + ch);
        const v4i v = {src[0], src[1], src[2], src[3]};
        uint8_t *dst = ob + (long long)(p + y * (g.Wo - wt)) * g.CH;
        if (n >= 16) {
          *(v4i_u *)dst = v;
        } else {
#pragma unroll
          for (int j = 0; j < 16; j++)
            if (j < n) dst[j] = (uint8_t)((unsigned)v[j / 4] >> (8 * (j & 3)));
        }
      }
  }
}
