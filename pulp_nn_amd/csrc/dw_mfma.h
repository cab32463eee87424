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
// output.  The rows of T are read per channel from the filter rows in LDS, two dwords and a byte shift for each of theirs (the
// places depend on the lane only).
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
// Bound: small layers by the instructions of one wave, one after the other: a dependent one takes 8 clocks whichever unit executes it,
// and nothing covers that with one wave per SIMD (10x8x48: some 9000 clocks from the first instruction to the last).  So: the launch's
// numbers are read at once; a wave fetches the filters and constants of its own channels and builds the matrix rows while its part of
// the input is on the way; the input travels by buffer loads, whose addresses take two instructions, and parts of a pass that no channel
// needs are left out.  (The same set-up with every array going through LDS behind one barrier and each number read where it is used:
// 10x8x48 batch 5 5.3 us, now 4.2; 28x7x8 batch 35 5.18, 3.84; 35x29x72 batch 32 8.7, 7.6.)
// Larger layers by the vector ALU (13x39x408 batch 208 43.6 us, now 38.3, 85 MB).  Measured, whole calls, against the kernels
// it replaced (four outputs per lane with v_dot4 for 3x3, a byte loop for rows that are not whole dwords and for other filters): 3x3
// on 35x29x72 batch 32 36.7 -> 7.6 us; 5x5 on 8x23x32 batch 9 91 -> 5; 5x5 stride 2 on 60x11x416 batch 4 65 -> 7.
#pragma once
#include <type_traits>

#include "dw_mfma_geom.h"
#include "igemm.h"
#include "memops.h"
#include "requant.h"

// Bytes of a chunk that was loaded `sh` bytes away from where it is: moved down (sh > 0: loaded too early) or up, zeros behind.
typedef unsigned v4u __attribute__((ext_vector_type(4)));
__device__ __forceinline__ v4u dwm_shift(v4u v, int sh)
{
  const int n = min(max(sh, -16), 16), up = n < 0 ? -1 : 0;
  // moving up by m bytes is moving {zeros, chunk} down by 16 - m
  const int down = n + (up & 16);
  unsigned w[8];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    w[i] = up ? 0u : v[i];
    w[4 + i] = up ? v[i] : 0u;
  }
  if (down & 16)
#pragma unroll
    for (int i = 0; i < 4; i++) w[i] = w[4 + i], w[4 + i] = 0u;
  if (down & 8)
#pragma unroll
    for (int i = 0; i < 6; i++) w[i] = w[i + 2];
  if (down & 4)
#pragma unroll
    for (int i = 0; i < 5; i++) w[i] = w[i + 1];
  v4u r;
#pragma unroll
  for (int i = 0; i < 4; i++) r[i] = __builtin_amdgcn_alignbyte(w[i + 1], w[i], down & 3);
  return r;
}

__device__ __forceinline__ bn_t readlane_bn(bn_t v, int l)
{
#if PULPNN_BN_BITS == 64
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, l), hi = (unsigned)__builtin_amdgcn_readlane((int)(v >> 32), l);
  return (bn_t)((unsigned long long)hi << 32 | lo);
#else
  return __builtin_amdgcn_readlane(v, l);
#endif
}

// MODE: requantisation branch; NM: MFMAs per (channel, 16 units) = ceil(ky * ND / 16); CB: channels per workgroup
template <int CB, int NM, int MODE>
__global__ __launch_bounds__(256, CB == 16 ? (NM == 1 ? 5 : NM <= 3 ? 4 : 1) : NM <= 2 ? 4 : NM == 3 ? 3 : 1) void dw_mfma_kernel(DwmGeom g, EpiArgs e)
{
  extern __shared__ __attribute__((aligned(16))) unsigned char dwm_lds[];
  // The launch's numbers, all at once: left to itself the compiler asks for each where it is first needed (and again where it is
  // needed later), twenty trips to the scalar cache one after the other.  (Opaque, so that it cannot.)
  asm volatile("" : "+s"(g.total), "+s"(g.cblocks), "+s"(g.xtiles), "+s"(g.bands), "+s"(g.in), "+s"(g.wt), "+s"(g.bias), "+s"(g.CH),
               "+s"(g.H), "+s"(g.W), "+s"(g.ky), "+s"(g.kx), "+s"(e.k), "+s"(e.lambda), "+s"(g.RB));
  asm volatile("" : "+s"(g.NR), "+s"(g.Q), "+s"(g.XT), "+s"(g.ND), "+s"(g.rND), "+s"(g.nper), "+s"(g.cpar), "+s"(g.pitch), "+s"(g.CS),
               "+s"(g.w_off), "+s"(g.in_bytes), "+s"(g.wt_bytes), "+s"(e.shift), "+s"(g.sx), "+s"(g.sy));
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lgrp = lane >> 4;
  const DwmTile tile = dwm_tile<CB>(g, (unsigned)xcd_remap(blockIdx.x, g.total));
  const unsigned b = tile.b;
  const int c0 = tile.c0, xg0 = tile.xg0, oy0 = tile.oy0, ncb = tile.ncb, rows = tile.rows, wt = tile.wt;
  const int plane = g.H * g.W;
  const long long before = ((long long)b * g.CH + c0) * plane;
  const uint8_t *img = g.in + before;

  // ---- ask for what the set-up reads: the wave's filters and constants, then the first input rows -------------------
  // (What is asked for first comes back first.  A wave has nq quads of channels, cw and those behind it; channels that do not
  // exist read as the last one and are not written.)
  const int nq = CB == 16 ? 1 : (ncb + 15) / 16, cw = 4 * nq * wave;
  const int nrow = 4 * nq * g.ky;  // filter rows, those of all channels back to back
  auto filter_at = [&](int t) { return dwm_filter_at(g, tile, cw, t); };
  const int wlast = g.wt_bytes - 8;
  v2i w_raw = {0, 0};
  if (wlast >= 0) w_raw = *(const v2i_u *)(g.wt + min(filter_at(lane), wlast));
  int p_bias = 0;
  bn_t p_k = 0, p_l = 0;
  {
    const int c = c0 + min(cw + (lane & (CB / 4 - 1)), ncb - 1);
    if (g.bias) p_bias = (int)g.bias[c];
    if (MODE == EPI_BN) {
      p_k = e.k[c];
      p_l = e.lambda[c];
    }
  }

  const int slots = g.NR * g.Q;
  const int iy0 = oy0 * g.sy - g.pt, x0 = 16 * xg0 * g.sx - g.pl;
  const int cpi = (int)fastdiv((unsigned)tid, g.d_nper);
  constexpr int UN = DWM_LOADS;
  const bool edge = dwm_edge(g, tile, before);  // a load of this tile may leave the tensor
  // Inside: buffer loads (dwm_buffer_off)
  const __amdgpu_buffer_rsrc_t rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void *)(img - 64), 0, (int)min(g.in_bytes - before + 64, 0x7fffffffll), 0x00020000);
  const long long behind = g.in_bytes - before - 16;
  const int lo_lim = (int)max(-before, -(1ll << 30)), hi_lim = (int)min(behind, 0x7fffffffll);
  // one pass: a thread's (row, chunk) of UN channels; s0: the pass's first slot, cj: the pass's first channel
  int base, lds_at, ch;     // ch: the thread's first channel, out of reach where it has no slot
  unsigned mask[4];         // the chunk's bytes inside the image
  auto place = [&](int s0) {
    const int slot = s0 + tid - cpi * g.nper;
    const int row = (int)fastdiv((unsigned)slot, g.d_q), q = slot - row * g.Q;
    const int x = x0 + 16 * q, iy = iy0 + row;
    base = dwm_load_base(g, iy, x);
    lds_at = row * g.pitch + 16 * q + cpi * g.CS;
    ch = dwm_thread_channel(CB, cpi, slot < slots);
    const int n = (unsigned)iy < (unsigned)g.H ? 8 * (g.W - x) : 0;
#pragma unroll
    for (int d = 0; d < 4; d++) mask[d] = low_bits(n - 32 * d) & high_bits(-8 * x - 32 * d);
  };
  v4u v[UN];
  auto chan_off = [&](int cb) { return min(cb, ncb - 1) * plane + base; };
  auto load = [&](int cj) {
    if (edge) {
#pragma unroll
      for (int u = 0; u < UN; u++) {
        if (u != 0 && cj + u * g.cpar >= ncb) break;
        const v4i t = *(const v4i_u *)(img + min(max(chan_off(cpi + cj + u * g.cpar), lo_lim), hi_lim));
        v[u] = (v4u){(unsigned)t.x, (unsigned)t.y, (unsigned)t.z, (unsigned)t.w};
      }
    } else {
      const unsigned at = dwm_buffer_first(plane, ch, cpi, base), at_last = dwm_buffer_last(plane, ncb, ch, cpi, base);
#pragma unroll
      for (int u = 0; u < UN; u++)
        if (u == 0 || cj + u * g.cpar < ncb) v[u] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, dwm_buffer_off(at, at_last, plane, cj + u * g.cpar), 0, 0);
    }
  };
  auto stage = [&](int cj) {
#pragma unroll
    for (int u = 0; u < UN; u++) {
      if (u != 0 && cj + u * g.cpar >= ncb) break;
      if (edge) {
        // the bytes were loaded up to 15 bytes too late (first bytes of the tensor) or too early (last ones)
        const int off = chan_off(cpi + cj + u * g.cpar), sh = off - min(max(off, lo_lim), hi_lim);
        if (__builtin_amdgcn_ballot_w64(sh != 0)) v[u] = dwm_shift(v[u], sh);
      }
      if (ch < ncb - cj - u * g.cpar)
        *(v4u *)(dwm_lds + lds_at + (cj + u * g.cpar) * g.CS) = (v4u){(v[u].x & mask[0]) ^ 0x80808080u, (v[u].y & mask[1]) ^ 0x80808080u,
                                                                     (v[u].z & mask[2]) ^ 0x80808080u, (v[u].w & mask[3]) ^ 0x80808080u};
    }
  };
  place(0);
  load(0);

  // ---- lane constants: dword d = 16 mm + 4 lgrp + i of K is dword d % ND of filter row d / ND -----------------
  // In that row it holds the filter columns 4 (d % ND) - l16 * sx to the third behind: four bytes that begin wsh bytes into
  // dword f of the filter row, f = d % ND - (l16 * sx + 3) / 4.  They are read as two whole dwords (a dword read at an odd
  // address takes the LDS some 200 clocks); a row in LDS is two dwords of zeros and its two dwords, and zeros follow it.
  const int wsh = (-l16 * g.sx) & 3, wq = (l16 * g.sx + 3) >> 2;
  int boff[NM][4], woff[NM][4];
#pragma unroll
  for (int mm = 0; mm < NM; mm++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int d = 16 * mm + 4 * lgrp + i, r = (d * g.rND) >> 16, xd = d - r * g.ND;
      const bool ok = r < g.ky;
      boff[mm][i] = ok ? r * g.pitch + 4 * xd : 0;
      woff[mm][i] = ok ? r * DWM_WROW + 4 * min(max(xd - wq + 2, 0), 4) : 0;
      // (here, not where it is used: the compiler would keep r and xd until then, and spill with three MFMAs a unit.  With two it has registers to spare,
      // and the 64-bit kernels are up to 14 % slower with this.)
      if constexpr (NM == 3) asm volatile("" : "+v"(boff[mm][i]));
    }
  __builtin_amdgcn_sched_barrier(0);

  // ---- the wave's filter rows -> its part of LDS ---------------------------------------------------------------------
  unsigned char *wl = dwm_lds + g.w_off + wave * dwm_wpart(CB, g.ky);
  auto filter_put = [&](int t, unsigned long long w) {  // w: the row, `late` bytes too early if it is one of the tensor's last
    w = w >> (8 * max(filter_at(t) - wlast, 0)) & ~0ull >> (64 - 8 * g.kx);
    *(v4i *)(wl + t * DWM_WROW) = (v4i){0, 0, (int)(unsigned)w, (int)(unsigned)(w >> 32)};
  };
  auto row64 = [](v2i w) { return (unsigned)w.x | (unsigned long long)(unsigned)w.y << 32; };
  if (wlast >= 0) {
    if (lane < nrow) filter_put(lane, row64(w_raw));
    for (int t = lane + 64; t < nrow; t += 64) filter_put(t, row64(*(const v2i_u *)(g.wt + min(filter_at(t), wlast))));
  } else {  // a layer of fewer bytes of filters than one load
    for (int t = lane; t < nrow; t += 64) {
      unsigned long long w = 0;
      for (int i = g.wt_bytes - 1; i >= 0; i--) w = w << 8 | (uint8_t)g.wt[i];
      filter_put(t, w << (8 * -wlast));
    }
  }
  if (lane < 2) *(int *)(wl + nrow * DWM_WROW + 4 * lane) = 0;
  __builtin_amdgcn_wave_barrier();  // (from here on the wave reads its own part)

  // ---- a quad of channels: filters as matrix rows, constants of the epilogue -----------------------------------------
  const v4i b64 = {0x40404040, 0x40404040, 0x40404040, 0x40404040};
  v4i a[4][NM];
  bn_t kk[4], ll[4];
  bool ks;
  auto filters = [&](int j) {  // quad j of the wave
#pragma unroll
    for (int cc = 0; cc < 4; cc++)
#pragma unroll
      for (int mm = 0; mm < NM; mm++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const unsigned *w = (const unsigned *)(wl + (4 * j + cc) * g.ky * DWM_WROW + woff[mm][i]);
          a[cc][mm][i] = (int)__builtin_amdgcn_alignbyte(w[1], w[0], wsh);
        }
    v4i s[4];
#pragma unroll
    for (int cc = 0; cc < 4; cc++) {
      s[cc] = (v4i){0, 0, 0, 0};
#pragma unroll
      for (int mm = 0; mm < NM; mm++) s[cc] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[cc][mm], b64, s[cc], 0, 0, 0);
    }
    ks = true;
#pragma unroll
    for (int cc = 0; cc < 4; cc++) {
      // (s: 64 times the sum of the filter, in every element)
      const int corr = __builtin_amdgcn_readlane(p_bias, 4 * j + cc) + 2 * __builtin_amdgcn_readfirstlane(s[cc][0]);
      if (MODE == EPI_BN) {
        kk[cc] = readlane_bn(p_k, 4 * j + cc);
        ll[cc] = readlane_bn(p_l, 4 * j + cc);
      } else {
        kk[cc] = MODE == EPI_MULT ? (bn_t)e.mult : (bn_t)1;
        ll[cc] = 0;
      }
      ks = ks && bn_k_small(kk[cc]);
      // k * (acc + corr) + lambda = k * acc + (k * corr + lambda), exact in the wrapping arithmetic of the type
#if PULPNN_BN_BITS == 64
      if (MODE == EPI_BN) ll[cc] = (bn_t)((unsigned long long)kk[cc] * (unsigned long long)(long long)corr + (unsigned long long)ll[cc]);
      else
#endif
        ll[cc] = (bn_t)(int)((unsigned)kk[cc] * (unsigned)corr + (unsigned)ll[cc]);
    }
  };
  filters(0);  // (the first quad's while the input is on its way)

  // ---- input rows -> LDS ----------------------------------------------------------------------------------------
  for (int s0 = 0;;) {
    for (int cj = 0;;) {
      stage(cj);
      cj += UN * g.cpar;
      if (cj >= ncb) break;
      load(cj);
    }
    s0 += g.nper;
    if (s0 >= slots) break;
    place(s0);
    load(0);
  }
  __syncthreads();

  // (an output pixel takes one dword more than its channels in LDS: a store's lanes are multiples of four pixels apart)
  constexpr int PP = CB + 4;
  // ---- multiply ---------------------------------------------------------------------------------------------------
  const int units = rows * g.XT, shift = e.shift;
  for (int j = 0; cw + 4 * j < ncb;) {
    const int qd = cw / 4 + j;
    auto tiles = [&](auto fast) {
      constexpr bool FAST = decltype(fast)::value;  // BN: k fits 24 (64-bit build: 32) bits; MULT: shift >= 16
      for (int u0 = 0; u0 < units; u0 += 16) {
        const int u = min(u0 + l16, units - 1);
        const int y = (int)fastdiv((unsigned)u, g.d_xg), xg = u - y * g.XT;
        const unsigned char *src = dwm_lds + (4 * qd) * g.CS + y * g.sy * g.pitch + xg * 16 * g.sx;
        int v[4][4];
        v4i bf[4][NM], accs[4];
#pragma unroll
        for (int cc = 0; cc < 4; cc++)
#pragma unroll
          for (int mm = 0; mm < NM; mm++)
#pragma unroll
            for (int i = 0; i < 4; i++) bf[cc][mm][i] = *(const int *)(src + cc * g.CS + boff[mm][i]);
#pragma unroll
        for (int cc = 0; cc < 4; cc++) {
          accs[cc] = (v4i){0, 0, 0, 0};
#pragma unroll
          for (int mm = 0; mm < NM; mm++) accs[cc] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[cc][mm], bf[cc][mm], accs[cc], 0, 0, 0);
        }
#pragma unroll
        for (int cc = 0; cc < 4; cc++) {
          const v4i acc = accs[cc];
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
    if (++j == nq) break;
    filters(j);
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
