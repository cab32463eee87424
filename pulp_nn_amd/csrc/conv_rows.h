// Convolution with a filter of up to four rows of up to 16 bytes (the 3x3 stem of a network on RGB or RGBA, pointwise layers of up to 16
// channels) on the matrix cores.
//
// A filter row of a pixel is kx * Ci contiguous bytes of the HWC input, so the four 16-byte slots of K of one v_mfma_i32_16x16x64_i8
// are the filter's rows: a lane fetches 16 bytes from the dword below a row's first byte and shifts them into place, and 16 pixels x 16 channels are one instruction, whatever the geometry.
// Bytes behind a row's end meet zero weights; columns outside the image are cleared, and rows outside it, where a wave has any; the
// first and the last bytes of the tensor are met by clamping the address and shifting.  The filters are fetched the same way.  No barrier:
// a wave is an independent item.  LDS is used in two places, a part of it per wave, and relies on a wave's accesses being served in order: for
// the input of rows of 64 output pixels (ROWS_ROW64 below), and for results of 33 to 63 channels.
//
// Rows of the MFMA are dealt so that a lane ends up with 4 * NT consecutive channels of its pixel (dw_hwc.h); with NT == 1 and 16
// channels in all, the four pixels of a lane's four units change places between lanes and a store is 16 bytes a lane, 1 KB in memory order.
//
// Replaces v_dot4 with one pixel per lane, which took 370 vector instructions per 64 pixels and 16 channels, and the band in LDS
// (conv_band.h) for such filters of more than 32 channels.  Bound: memory latency, at one to eight groups of 64 pixels per wave (rows_shape).
// Call by call, before / now: 128x128x3 -> 16 stride 2 batch 256 15.8 / 13.1 us, batch 1 4.2 / 4.0; 32x32x3 -> 64 batch 64 8.9 / 5.8, batch 1 5.7 / 4.7;
// 57x43x3 -> 40 batch 64 21.8 / 11.0; 64x64x4 -> 256 batch 32 37.5 / 18.7; 64x64x5 -> 16 stride 2 batch 64 6.5 / 4.1; 64x64x16 -> 32 1x1 6.9 / 3.6.  A few
// small filters of few channels are slower: 64x64x1 -> 6 batch 256 13.8 / 15.3, 191x16x3 -> 16 3x1 batch 286 14.1 / 15.8, 5x20x1 -> 16 2x2 3.6 / 4.0.
// Reference semantics:
// 32bit/src/pulp_nn_conv_Ho_parallel.c:76-183 (im2col order ky, kx, ci) and pulp_nn_matmul.c:144-216 (requantisation).
#pragma once
#include "conv_rows_geom.h"
#include "dw_hwc.h"

// v moved towards byte 0 by n bytes (n < 0: away from it), zeros behind; |n| <= 16
__device__ __forceinline__ v4i bytes_shift(v4i v, int n)
{
  unsigned __int128 t = ((unsigned __int128)((unsigned long long)(unsigned)v.z | ((unsigned long long)(unsigned)v.w << 32)) << 64) |
                        ((unsigned long long)(unsigned)v.x | ((unsigned long long)(unsigned)v.y << 32));
  if (n > 0) t = n < 16 ? t >> (8 * n) : 0;
  if (n < 0) t = n > -16 ? t << (-8 * n) : 0;
  return (v4i){(int)(unsigned)t, (int)(unsigned)(t >> 32), (int)(unsigned)(t >> 64), (int)(unsigned)(t >> 96)};
}

// all ones below byte n of a dword's four bytes (n any number); no branch
__device__ __forceinline__ unsigned below(int n)
{
  const unsigned m = (1u << (8 * max(n, 0) & 31)) - 1u;
  return n >= 4 ? ~0u : m;
}

// PLACE: where the units of 16 pixels lie.  ROWS_ROW16: inside one output row each, scalar arithmetic.  ROWS_ROW64: four of them side by side;
// the filter rows of the 64 pixels are then fetched as whole pieces of memory, 64 contiguous bytes by four lanes, and handed out through
// a part of LDS that belongs to the wave: a lane's own 16 bytes, at a stride of a few bytes from lane to lane, cost the address unit a
// cycle each (128x128x3 -> 16 stride 2 at batch 256 14.7 us without, 13.3 with).
enum { ROWS_ANY = 0, ROWS_ROW16 = 1, ROWS_ROW64 = 2 };
template <int NT, int PLACE>
__global__ __launch_bounds__(256, NT == 4 ? 2 : 4) void conv_rows_kernel(RowsGeom g, EpiArgs e, int mode)
{
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, lgrp = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = blockIdx.y * (16 * NT);

  // ---- the first pixels ------------------------------------------------------------------------------------------------------
  constexpr bool ROW16 = PLACE != ROWS_ANY, STAGED = PLACE == ROWS_ROW64;
  // Whether results can be put together in LDS: with four tiles.  (With fewer tiles the way there is longer than their few odd stores, 13x30x2 -> 7
  // 3x2 batch 13 4.6 / 5.2 us, 102x128x5 -> 26 3x3 batch 18 8.6 / 9.4; in the 64-bit build it takes the registers of a third wave per SIMD, 20x16x4 ->
  // 261 4x3 batch 45 10.5 / 11.5.)
  constexpr bool GATHER = NT == 4 && sizeof(bn_t) == 4;
  __shared__ __attribute__((aligned(16))) unsigned char rows_l[4][GATHER ? 1024 * NT : STAGED ? 4 * ROWS_PITCH : 16];
  unsigned char *mine = rows_l[wave];
  int grp = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 * g.npass + wave);
  RowsWindow win[4];
  v4i v[4];
  int more[4] = {0, 0, 0, 0};
  // The slots of rows that the filter does not have meet zero weights: they repeat its last row, and ask neither for memory of their own nor
  // for a look at the image's edges; 158x198x2 -> 7 4x1 batch 253 111 us with rows of their own, 80 so.  (Leaving them out of the load is worse: a
  // load that not all lanes take part in is waited for as a whole, 5x20x1 -> 16 2x2 4.0 / 4.5.)
  const bool has_row = lgrp < g.ky;
  const int slot = min(lgrp, g.ky - 1);
  const int loff = rows_lane(g, ROW16 ? l16 : 0, slot);
  typedef v4i v4i_4 __attribute__((aligned(4)));
  auto request = [&]() {
    if constexpr (STAGED) {
      const RowsWindow w = rows_window(g, (unsigned)min(64 * grp, g.M - 64));
#pragma unroll
      for (int u = 0; u < 4; u++) win[u] = RowsWindow{w.at + 16 * u * g.sx * g.Ci, w.iy, w.ix + 16 * u * g.sx};
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const int fy = min(2 * i + (lane >> 5), g.ky - 1);
        v[i] = *(const v4i_4 *)(g.in + (unsigned)rows_chunk_at(g, w.at + fy * g.W * g.Ci, min(lane & 31, rows_chunks(g) - 1)));
      }
      return;
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      // (units past the last pixel repeat it: fetched, not stored)
      const int m = 64 * grp + 16 * u + (ROW16 ? 0 : l16);
      win[u] = rows_window(g, (unsigned)min(m, ROW16 ? g.M - 16 : g.M - 1));
      const int at = win[u].at + loff;
      v[u] = *(const v4i_4 *)(g.in + (unsigned)rows_fetch(g, at));
      if (rows_long(g)) more[u] = *(const int *)(g.in + (unsigned)rows_more(g, at));
    }
  };
  request();

  // ---- filters and constants, all of them requested before the first is used ---------------------------------------------------------
  // Row i of tile t is channel 4 * NT * (i / 4) + 4 * t + i % 4; slot lgrp of it the channel's filter row lgrp.
  v4i A[NT];
  const int wbytes = g.N * g.K;
  int off[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) {
    off[t] = (n0 + 4 * NT * (l16 >> 2) + 4 * t + (l16 & 3)) * g.K + lgrp * g.L;
    A[t] = *(const v4i_u *)(g.w + (unsigned)max(min(off[t], wbytes - 16), 0));
  }
  const int cb = n0 + 4 * NT * lgrp;  // the lane's channels
  typedef bn_t bn4 __attribute__((ext_vector_type(4), aligned(sizeof(bn_t))));
  const bn_t same = mode == EPI_MULT ? (bn_t)e.mult : (bn_t)1;
  bn_t kk[NT][4], ll[NT][4];
  int bias[NT];  // four bytes
#pragma unroll
  for (int t = 0; t < NT; t++) {
    bias[t] = 0;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      kk[t][r] = same;
      ll[t][r] = 0;
    }
  }
  if (g.N >= 4) {
    // (past the last channel the last four, turned into place further down)
#pragma unroll
    for (int t = 0; t < NT; t++) {
      const int c = min(cb + 4 * t, g.N - 4);
      if (g.bias) bias[t] = *(const i32_u *)(g.bias + c);
      if (mode == EPI_BN) {
        const bn4 k = *(const bn4 *)(e.k + c), l = *(const bn4 *)(e.lambda + c);
#pragma unroll
        for (int r = 0; r < 4; r++) {
          kk[t][r] = k[r];
          ll[t][r] = l[r];
        }
      }
    }
  } else {
    for (int c = 0; c < g.N; c++) {
      if (g.bias) bias[0] |= (int)(uint8_t)g.bias[c] << (8 * c);
      if (mode == EPI_BN) {
#pragma unroll
        for (int r = 0; r < 3; r++) {
          if (r != c) continue;
          kk[0][r] = e.k[c];
          ll[0][r] = e.lambda[c];
        }
      }
    }
  }
  if (g.N >= 4 && n0 + 16 * NT > g.N && (g.N & 3)) {
#pragma unroll
    for (int t = 0; t < NT; t++) {
      const int by = cb + 4 * t - min(cb + 4 * t, g.N - 4);  // (channels from by = 4 on do not exist)
      bias[t] = (int)((unsigned)bias[t] >> (8 * (by & 3)));
#pragma unroll
      for (int turn = 1; turn < 4; turn *= 2) {
        bn_t k[4], l[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          k[r] = by & turn ? kk[t][(r + turn) & 3] : kk[t][r];
          l[r] = by & turn ? ll[t][(r + turn) & 3] : ll[t][r];
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
          kk[t][r] = k[r];
          ll[t][r] = l[r];
        }
      }
    }
  }
#pragma unroll
  for (int t = 0; t < NT; t++) {
    const bool ok = has_row && off[t] < wbytes;
    const int late = ok ? off[t] - max(min(off[t], wbytes - 16), 0) : 0, keep = ok ? -1 : 0;
    if (__any(late > 0)) A[t] = bytes_shift(A[t], max(late, 0));
#pragma unroll
    for (int d = 0; d < 4; d++) A[t][d] &= (int)below(g.L - 4 * d) & keep;
  }
  bool ks = true;
#pragma unroll
  for (int t = 0; t < NT; t++) {
    const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101}, zero = {0, 0, 0, 0};
    const v4i s = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[t], ones, zero, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int corr = 128 * s[r] + (int)(int8_t)((unsigned)bias[t] >> (8 * r));
      const bn_t k = kk[t][r];
      ks = ks && bn_k_small(k);
#if PULPNN_BN_BITS == 64
      if (mode == EPI_BN) ll[t][r] = (bn_t)((unsigned long long)k * (unsigned long long)(long long)corr + (unsigned long long)ll[t][r]);
      else
#endif
        ll[t][r] = (bn_t)(int)((unsigned)k * (unsigned)corr + (unsigned)ll[t][r]);
    }
  }
  const int form = dwh_form(mode, e.shift, (bool)__all(ks), true);  // |acc| <= 64 * 128 * 128

  for (int pass = 0; pass < g.npass && grp < g.groups; pass++) {
    // ---- the operands -------------------------------------------------------------------------------------------------------
    v4i px[4];
    if constexpr (STAGED) {
#pragma unroll
      for (int i = 0; i < 2; i++) *(v4i *)(mine + ROWS_PITCH * (2 * i + (lane >> 5)) + 16 * (lane & 31)) = v[i];
      __builtin_amdgcn_wave_barrier();
      asm volatile("" ::: "memory");
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int *p = (const int *)(mine + ROWS_PITCH * slot + (((win[0].at + slot * g.W * g.Ci) & 3) + (16 * u + l16) * g.sx * g.Ci & ~3));
        v[u] = (v4i){p[0], p[1], p[2], p[3]};
        if (rows_long(g)) more[u] = p[4];
      }
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int at = win[u].at + loff, sh = at & 3;
#pragma unroll
      for (int d = 0; d < 4; d++) px[u][d] = (int)__builtin_amdgcn_alignbyte((unsigned)(d < 3 ? v[u][d < 3 ? d + 1 : 3] : more[u]), (unsigned)v[u][d], (unsigned)sh);
      if (ROW16 ? rows_edge(g, win[u]) : true) {
        RowsWindow w = win[u];
        if (ROW16) w.ix += l16 * g.sx;
        const RowsKeep n = rows_keep(g, w, slot);
        const bool end = has_row && n.row && rows_near_end(g, at);
        if (ROW16 || __any(has_row && (!n.row || end || n.lo > 0 || n.hi < g.L))) {
          if (__any(end)) {  // (first and last rows of the whole tensor)
            const int from = rows_exact(g, at);
            const v4i exact = bytes_shift(*(const v4i_u *)(g.in + (unsigned)from), min(max(at - from, -16), 16));
#pragma unroll
            for (int d = 0; d < 4; d++) px[u][d] = end ? exact[d] : px[u][d];
          }
#pragma unroll
          for (int d = 0; d < 4; d++) px[u][d] = n.row ? (int)((unsigned)px[u][d] & below(n.hi - 4 * d) & ~below(n.lo - 4 * d)) : 0;
        }
      }
      px[u] = px[u] ^ (int)0x80808080;
    }
    if constexpr (STAGED) {
      __builtin_amdgcn_wave_barrier();
      asm volatile("" ::: "memory");
    }
    const int m0 = 64 * grp;
    grp += 4;
    if (pass + 1 < g.npass && grp < g.groups) request();
    // ---- multiply, requantise, store ------------------------------------------------------------------------------------------
    unsigned q[4][NT];
    dwh_with_form(form, [&](auto f) {
#pragma unroll
      for (int u = 0; u < 4; u++)
#pragma unroll
        for (int t = 0; t < NT; t++) {
          const v4i zero = {0, 0, 0, 0};
          const v4i acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[t], px[u], zero, 0, 0, 0);
          q[u][t] = dwh_requant<decltype(f)::value>(acc, kk[t], ll[t], e.shift);
        }
    });
    if (NT == 1 && g.N == 16) {
      const unsigned p[4] = {q[0][0], q[1][0], q[2][0], q[3][0]};
      const v4i o = dwh_pixels(p);
      if (m0 + lane < g.M) *(v4i_u *)(g.out + (long long)(m0 + lane) * 16) = o;
    } else if (GATHER && g.gather) {
      // the results of the 64 pixels are 64 * N contiguous bytes: put together in the wave's part of LDS
      // (the channels left as a value that the compiler does not know: it would keep all comparisons with it in scalar registers)
      int left = g.N - cb;
      asm volatile("" : "+v"(left));
#pragma unroll
      for (int u = 0; u < 4; u++) {
        unsigned char *o = mine + (16 * u + l16) * g.N + cb;
#pragma unroll
        for (int t = 0; t < NT; t++) {
          if (4 * t + 4 <= left) *(i32_u *)(o + 4 * t) = (int)q[u][t];
          else
#pragma unroll
            for (int r = 0; r < 4; r++)
              if (4 * t + r < left) o[4 * t + r] = (unsigned char)(q[u][t] >> (8 * r));
        }
      }
      __builtin_amdgcn_wave_barrier();
      asm volatile("" ::: "memory");
      const int bytes = min(64, g.M - m0) * g.N;
      uint8_t *o = g.out + (long long)m0 * g.N;
      for (int i = 16 * lane; i < bytes; i += 1024) {
        if (i + 16 <= bytes) *(v4i_u *)(o + i) = *(const v4i *)(mine + i);
        else
          for (int j = i; j < bytes; j++) o[j] = mine[j];
      }
      __builtin_amdgcn_wave_barrier();
      asm volatile("" ::: "memory");
    } else {
      int left = g.N - cb;
      asm volatile("" : "+v"(left));
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int m = m0 + 16 * u + l16;
        uint8_t *o = g.out + (long long)m * g.N + cb;
        if (m >= g.M) continue;
        if (4 * NT <= left) {
          if constexpr (NT == 4) *(v4i_u *)o = (v4i){(int)q[u][0], (int)q[u][1 % NT], (int)q[u][2 % NT], (int)q[u][3 % NT]};
          else if constexpr (NT == 2) *(v2i_u *)o = (v2i){(int)q[u][0], (int)q[u][1 % NT]};
          else *(i32_u *)o = (int)q[u][0];
        } else {
#pragma unroll
          for (int t = 0; t < NT; t++) {
            if (4 * t + 4 <= left) *(i32_u *)(o + 4 * t) = (int)q[u][t];
            else
#pragma unroll
              for (int r = 0; r < 4; r++)
                if (4 * t + r < left) o[4 * t + r] = (uint8_t)(q[u][t] >> (8 * r));
          }
        }
      }
    }
  }
}
