// 3x3 depthwise (padding 1, stride 1 or 2), HWC in, HWC out, on the matrix cores.
//
// In HWC a lane's 16-byte load is sixteen channels of one pixel, and a depthwise layer is a contraction over (filter column,
// channel) with a diagonal weight matrix: D[16 channels][16 pixels] += A[16 x 64] B[64 x 16], K = (column kx, channel), A holding
// filter byte (fy, kx) of a channel at the channel's own place in K and zero elsewhere.  One v_mfma_i32_16x16x64_i8 per filter
// row; the fourth 16-byte slot of K is empty.  One multiply in 21 counts, but the matrix cores have nothing else to do here, and
// the vector ALU is left with the ^ 0x80 of the input, the requantisation and a few addresses: 12 instructions per 256 outputs,
// where v_dot4 needs 38 and transposes four by four bytes on the way in and out (dw3x3_rows_kernel, which this replaces for
// channel counts of whole tiles).
//
// A wave walks down R rows of one image in full width, 16 * NT channels at a time, so that an input row is one 16-byte load per
// lane, four rows ahead.  The row passes through a two-row ring in LDS that belongs to the wave (no barrier), from where a lane
// reads its pixel's left, own and right neighbour, and it serves the up to three output rows above, at and below it.
//
// Rows of the MFMA are dealt so that a lane ends up with 4 * NT consecutive channels of its pixel: row i of tile t is
// channel (i / 4) * 4 * NT + 4 * t + i % 4, and the operand of tile t is every NT-th dword of the pixel's 16 * NT bytes.
//
// Bound: the memory system for large layers, call by call at batch 256 64x64x16 12.6 -> 9.2 us (33.5 MB, of which some 3 us are the
// launch), 64x64x32 stride 2 12.0 -> 8.8, 32x32x64 11.3 -> 8.7, 32x32x64 stride 2 6.7 -> 6.0, 16x16x128 6.8 -> 6.5; the chain load ->
// LDS -> multiply -> store for small ones, at batch 16 6.6 -> 3.8, 6.2 -> 3.4, 5.9 -> 4.2, 5.9 -> 3.5, 5.6 -> 4.8.
#pragma once
#include <type_traits>

#include "dw_hwc_geom.h"
#include "memops.h"
#include "requant.h"

// The forms of kk * acc + ll, shift, saturation: with the 24-bit multiplier (|acc| < 2^23 and kk of 24 bits, no narrowing), with the
// 32-bit one, the same with the reference's narrowing to int16_t behind the shift (multiplier branch, shifts below 16), and in
// the 64-bit build batch-norm with kk of 32 bits and with any kk.
enum { DWH_FAST = 0, DWH_MUL32 = 1, DWH_NARROW = 2, DWH_BN64_SMALL = 3, DWH_BN64 = 4 };
// k_small: all kk fit 24 (64-bit build: 32) bits; acc24: |acc| < 2^23
__device__ __forceinline__ int dwh_form(int mode, int shift, bool k_small, bool acc24)
{
#if PULPNN_BN_BITS == 64
  if (mode == EPI_BN) return k_small ? DWH_BN64_SMALL : DWH_BN64;
#else
  if (mode == EPI_BN) return k_small && acc24 ? DWH_FAST : DWH_MUL32;
#endif
  if (mode == EPI_MULT && shift < 16) return DWH_NARROW;
  return acc24 ? DWH_FAST : DWH_MUL32;
}
// f(std::integral_constant<int, form>)
template <class F>
__device__ __forceinline__ void dwh_with_form(int form, F f)
{
  if (form == DWH_FAST) f(std::integral_constant<int, DWH_FAST>{});
#if PULPNN_BN_BITS == 64
  else if (form == DWH_BN64_SMALL) f(std::integral_constant<int, DWH_BN64_SMALL>{});
  else if (form == DWH_BN64) f(std::integral_constant<int, DWH_BN64>{});
#endif
  else if (form == DWH_MUL32) f(std::integral_constant<int, DWH_MUL32>{});
  else f(std::integral_constant<int, DWH_NARROW>{});
}

// four requantised bytes (four consecutive channels of one pixel)
template <int FORM>
__device__ __forceinline__ unsigned dwh_requant(const v4i &acc, const bn_t (&kk)[4], const bn_t (&ll)[4], int shift)
{
  int v[4], sh = shift;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    if constexpr (FORM == DWH_FAST) {
      v[r] = __mul24(acc[r], (int)kk[r]) + (int)ll[r];
    } else if constexpr (FORM == DWH_MUL32 || FORM == DWH_NARROW) {
      v[r] = (int)((unsigned)acc[r] * (unsigned)kk[r] + (unsigned)ll[r]);
      if (FORM == DWH_NARROW) v[r] = (int)(short)(v[r] >> shift);
    } else if constexpr (FORM == DWH_BN64_SMALL) {
      const long long x = (long long)(int)kk[r] * (long long)acc[r] + (long long)ll[r];
      v[r] = shift >= 32 ? (int)(x >> 32) : (int)__builtin_amdgcn_alignbit((unsigned)(x >> 32), (unsigned)x, shift);
    } else {
      const unsigned long long x = (unsigned long long)kk[r] * (unsigned long long)(long long)acc[r] + (unsigned long long)ll[r];
      v[r] = (int)(unsigned)(unsigned long long)((long long)x >> shift);
    }
  }
  if (FORM == DWH_NARROW || FORM == DWH_BN64) sh = 0;
  if (FORM == DWH_BN64_SMALL) sh = shift >= 32 ? shift - 32 : 0;
  return ashr_sat_pack4(v[0], v[1], v[2], v[3], sh);
}

// v[s] of lane (l16, lgrp): four bytes, channels 4 * lgrp .., of pixel 16 * s + l16.  Afterwards v[q] of lane (l16, lgrp) is channels 4 * q ..
// of pixel 16 * lgrp + l16: sixteen contiguous bytes of pixel `lane`.
__device__ __forceinline__ v4i dwh_pixels(const unsigned (&v)[4])
{
  const auto a = __builtin_amdgcn_permlane32_swap(v[0], v[2], false, false), b = __builtin_amdgcn_permlane32_swap(v[1], v[3], false, false);
  const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false), d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  return (v4i){(int)c[0], (int)c[1], (int)d[0], (int)d[1]};
}

// What a wave keeps per 16 * NT channels.
template <int NT>
struct DwhChannels {
  v4i A[NT][3];                 // weight operands, per filter row
  bn_t kk[NT][4], ll[NT][4];    // requantisation of channel 4 * NT * (lane / 16) + 4 * t + r: kk * acc + ll, then the shift
  int form;
};

// The raw parameters of the channels: requested early, turned into DwhChannels behind the first input.
template <int NT>
struct DwhParams {
  int w[NT][3], bias[NT];
  bn_t k[NT][4], l[NT][4];
};
template <int NT>
__device__ __forceinline__ void dwh_request(DwhParams<NT> &p, const int8_t *wt, const int8_t *bias, const EpiArgs &e, int mode, int c0, int lane)
{
  const int l16 = lane & 15, lgrp = lane >> 4;
  const int8_t *w = wt + (long long)(c0 + (l16 >> 2) * (4 * NT) + (l16 & 3)) * 9 + min(lgrp, 2);
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int fy = 0; fy < 3; fy++) p.w[t][fy] = (int)w[36 * t + 3 * fy];
  const int cb = c0 + 4 * NT * lgrp;
#pragma unroll
  for (int t = 0; t < NT; t++) p.bias[t] = bias ? *(const i32_u *)(bias + cb + 4 * t) : 0;
  if (mode == EPI_BN) {
    typedef bn_t bn4 __attribute__((ext_vector_type(4), aligned(sizeof(bn_t))));
#pragma unroll
    for (int t = 0; t < NT; t++) {
      const bn4 k = *(const bn4 *)(e.k + cb + 4 * t), l = *(const bn4 *)(e.lambda + cb + 4 * t);
#pragma unroll
      for (int r = 0; r < 4; r++) {
        p.k[t][r] = k[r];
        p.l[t][r] = l[r];
      }
    }
  } else {
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        p.k[t][r] = mode == EPI_MULT ? (bn_t)e.mult : (bn_t)1;
        p.l[t][r] = 0;
      }
  }
}
template <int NT>
__device__ __forceinline__ void dwh_channels(DwhChannels<NT> &c, const DwhParams<NT> &p, int mode, int shift, int lane)
{
  const int l16 = lane & 15, lgrp = lane >> 4;
  const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
  bool ks = true;
#pragma unroll
  for (int t = 0; t < NT; t++) {
    v4i s = {0, 0, 0, 0};
#pragma unroll
    for (int fy = 0; fy < 3; fy++) {
      const int v = lgrp < 3 ? (p.w[t][fy] & 255) << (8 * (l16 & 3)) : 0;
#pragma unroll
      for (int d = 0; d < 4; d++) c.A[t][fy][d] = (l16 >> 2) == d ? v : 0;
      s = __builtin_amdgcn_mfma_i32_16x16x64_i8(c.A[t][fy], ones, s, 0, 0, 0);  // sum of the filter
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int corr = 128 * s[r] + (int)(int8_t)((unsigned)p.bias[t] >> (8 * r));
      const bn_t k = p.k[t][r];
      ks = ks && bn_k_small(k);
      c.kk[t][r] = k;
      // k * (acc + corr) + lambda = k * acc + (k * corr + lambda), exact in the wrapping arithmetic of the type
#if PULPNN_BN_BITS == 64
      if (mode == EPI_BN) c.ll[t][r] = (bn_t)((unsigned long long)k * (unsigned long long)(long long)corr + (unsigned long long)p.l[t][r]);
      else
#endif
        c.ll[t][r] = (bn_t)(int)((unsigned)k * (unsigned)corr + (unsigned)p.l[t][r]);
    }
  }
  c.form = dwh_form(mode, shift, (bool)__all(ks), true);  // |acc| <= 9 * 128 * 128
}

// Walks a strip of one tile of 16 channels down `rows` output rows: next() is the operand of the next input row (one more than needed
// is asked for), put(bytes) takes four requantised channels of the next output row.
template <int S, int FORM, class Next, class Put>
__device__ __forceinline__ void dwh_walk(const DwhChannels<1> &c, int shift, int rows, Next next, Put put)
{
  const v4i zero = {0, 0, 0, 0};
  // N: the output row that the last input row started; M (stride 1): the one before it
  v4i M = zero, N, F, cur = next(), nxt = next();
  N = __builtin_amdgcn_mfma_i32_16x16x64_i8(c.A[0][0], cur, zero, 0, 0, 0);
  if constexpr (S == 1) {
    cur = next();
    M = __builtin_amdgcn_mfma_i32_16x16x64_i8(c.A[0][1], nxt, N, 0, 0, 0);
    N = __builtin_amdgcn_mfma_i32_16x16x64_i8(c.A[0][0], nxt, zero, 0, 0, 0);
  } else {
    cur = next();
  }
  for (int r = 0; r < rows; r++) {
    if constexpr (S == 1) {
      F = __builtin_amdgcn_mfma_i32_16x16x64_i8(c.A[0][2], cur, M, 0, 0, 0);
      M = __builtin_amdgcn_mfma_i32_16x16x64_i8(c.A[0][1], cur, N, 0, 0, 0);
      N = __builtin_amdgcn_mfma_i32_16x16x64_i8(c.A[0][0], cur, zero, 0, 0, 0);
      cur = next();
    } else {
      N = __builtin_amdgcn_mfma_i32_16x16x64_i8(c.A[0][1], nxt, N, 0, 0, 0);
      F = __builtin_amdgcn_mfma_i32_16x16x64_i8(c.A[0][2], cur, N, 0, 0, 0);
      N = __builtin_amdgcn_mfma_i32_16x16x64_i8(c.A[0][0], cur, zero, 0, 0, 0);
      if (r + 1 < rows) {
        nxt = next();
        cur = next();
      }
    }
    put(dwh_requant<FORM>(F, c.kk[0], c.ll[0], shift));
  }
}

template <int W, int S>
__global__ __launch_bounds__(256, 2) void dw_hwc_kernel(DwhGeom g, EpiArgs e, int mode)
{
  constexpr int NT = 64 / W, WO = W / S, XS = WO / 16;  // tiles of 16 channels, strips of 16 columns
  constexpr int PD = 4;                                 // input rows in flight
  constexpr int ROW = dwh_row_bytes<W>();
  __shared__ __attribute__((aligned(16))) unsigned char rows_l[4][2 * ROW];  // per wave: two input rows
  const int lane = threadIdx.x & 63, l16 = lane & 15, lgrp = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int q8 = (int)gridDim.x >> 3, rem = (int)gridDim.x & 7, x8 = blockIdx.x & 7;  // a contiguous range per XCD
  const int id = 4 * (x8 * q8 + min(x8, rem) + (int)(blockIdx.x >> 3)) + wave;
  if (id >= g.total) return;
  const DwhItem it = dwh_item<NT>(g, (unsigned)id);

  // ---- the first rows and the channels' parameters are requested ----------------------------------------------------------
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(g.in - g.lead), 0, g.size, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_o = __builtin_amdgcn_make_buffer_rsrc((void *)g.out, 0, g.out_size, 0x00020000);
  const unsigned voff = dwh_in_offset<W, S>(g, it, lane);
  const int rowb = W * g.C;
  v4i q[PD];
  auto request = [&](v4i &d, int ir) {
    typedef unsigned v4u __attribute__((ext_vector_type(4)));
    const bool ok = dwh_row_ok<S>(g, it, ir);  // (the same for all lanes)
    const v4u v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, ok ? voff : DWH_OOB, ok ? ir * rowb : 0, 0);
    d = (v4i){(int)v.x, (int)v.y, (int)v.z, (int)v.w};
  };
  DwhParams<NT> p;
  dwh_request<NT>(p, g.wt, g.bias, e, mode, it.c0, lane);
#pragma unroll
  for (int i = 0; i < PD; i++) request(q[i], i);

  unsigned char *lds = rows_l[wave];
  if (lane < 4 * NT) {  // columns -1 and W of both rows: outside the image
    const int chunk = lane % NT, side = (lane / NT) & 1, slot = lane / NT / 2;
    *(v4i *)(lds + slot * ROW + dwh_lds<W>(side ? W + 1 : 0, chunk)) = (v4i){(int)0x80808080, (int)0x80808080, (int)0x80808080, (int)0x80808080};
  }
  unsigned char *to = lds + dwh_lds<W>(lane / NT + 1, lane % NT);
  const unsigned char *from[XS][NT];  // (the lanes of the empty K slot read what their neighbours read)
#pragma unroll
  for (int x = 0; x < XS; x++)
#pragma unroll
    for (int j = 0; j < NT; j++) from[x][j] = lds + dwh_lds<W>((16 * x + l16) * S + min(lgrp, 2), j);
  const unsigned ooff = dwh_out_offset<W, S>(g, it, lane);
  DwhChannels<NT> c;
  dwh_channels<NT>(c, p, mode, e.shift, lane);

  // ---- down the rows ------------------------------------------------------------------------------------------------------
  // stage(i): row i, requested PD rows ago, goes to LDS as a ^ 0x80 and its registers are asked for row i + PD; px(): row i's
  // operands.  LDS serves a wave's accesses in order, so the rows of a wave need no barrier, only their order in the program.
  auto stage = [&](v4i &d, int slot, int ir) {
    *(v4i *)(to + slot * ROW) = d ^ (int)0x80808080;
    request(d, ir + PD);
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
  };
  const v4i zero = {0, 0, 0, 0};
  // N: the output row that the last input row started; M (stride 1): the one before it
  v4i M[XS][NT], N[XS][NT], F[XS][NT];
  auto walk = [&](auto form) {
    constexpr int FORM = decltype(form)::value;
    auto row = [&](int slot, auto role_tag) {
      constexpr int ROLE = decltype(role_tag)::value;  // bits: the filter rows that this input row takes part in
#pragma unroll
      for (int x = 0; x < XS; x++) {
        int px[4 * NT];
#pragma unroll
        for (int j = 0; j < NT; j++) {
          const v4i v = *(const v4i *)(from[x][j] + slot * ROW);
#pragma unroll
          for (int d = 0; d < 4; d++) px[4 * j + d] = v[d];
        }
#pragma unroll
        for (int t = 0; t < NT; t++) {
          const v4i b = {px[t], px[NT + t], px[2 * NT + t], px[3 * NT + t]};
          if (ROLE & 4) F[x][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(c.A[t][2], b, S == 1 ? M[x][t] : N[x][t], 0, 0, 0);
          if (ROLE & 2) (S == 1 ? M[x][t] : N[x][t]) = __builtin_amdgcn_mfma_i32_16x16x64_i8(c.A[t][1], b, N[x][t], 0, 0, 0);
          if (ROLE & 1) N[x][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(c.A[t][0], b, zero, 0, 0, 0);
        }
      }
    };
    // one tile: the 64 pixels of a row, or with stride 2 of two rows, change places between lanes so that one store writes their
    // 1 KB in memory order, instead of four of 256 bytes in 4-byte pieces
    unsigned v1[4];
    // u: which of the rows that are put together this is
    auto emit = [&](int r, int u) {
      typedef unsigned v4u __attribute__((ext_vector_type(4)));
      typedef unsigned vnt __attribute__((ext_vector_type(NT)));
#pragma unroll
      for (int x = 0; x < XS; x++) {
        vnt v;
#pragma unroll
        for (int t = 0; t < NT; t++) v[t] = dwh_requant<FORM>(F[x][t], c.kk[t], c.ll[t], e.shift);
        if constexpr (NT == 1) {
          v1[2 * u + x] = v[0];
        } else {
          const bool ok = dwh_out_ok<W, S>(it, r, lane);
          const int soff = ok ? (r * WO + 16 * x) * g.C : 0;
          if constexpr (NT == 2) __builtin_amdgcn_raw_buffer_store_b64(v, rsrc_o, ok ? ooff : DWH_OOB, soff, 0);
          else __builtin_amdgcn_raw_buffer_store_b128(v, rsrc_o, ok ? ooff : DWH_OOB, soff, 0);
        }
      }
      if constexpr (NT == 1) {
        if (u == S - 1) {
          const v4i p = dwh_pixels(v1);
          const int r0 = r - u;
          __builtin_amdgcn_raw_buffer_store_b128((v4u){(unsigned)p.x, (unsigned)p.y, (unsigned)p.z, (unsigned)p.w}, rsrc_o, dwh_out_ok<W, S>(it, r0, lane) ? ooff : DWH_OOB,
                                                 r0 < it.rows ? r0 * WO * g.C : 0, 0);
        }
      }
    };
    const std::integral_constant<int, 1> start{};
    const std::integral_constant<int, 2> middle{};
    const std::integral_constant<int, 3> two{};
    const std::integral_constant<int, 5> both{};
    const std::integral_constant<int, 7> all{};
    stage(q[0], 0, 0);
    stage(q[1], 1, 1);
    row(0, start);
    if constexpr (S == 1) {
      stage(q[2], 0, 2);
      row(1, two);
      for (int r = 0; r < it.rows; r += 4) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
          stage(q[(u + 3) & 3], (u + 1) & 1, r + u + 3);
          row(u & 1, all);
          emit(r + u, 0);
        }
      }
    } else {
      for (int r = 0; r < it.rows; r += 2) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
          stage(q[(2 * u + 2) & 3], 0, 2 * (r + u) + 2);
          row(1, middle);
          stage(q[(2 * u + 3) & 3], 1, 2 * (r + u) + 3);
          row(0, both);
          emit(r + u, u);
        }
      }
    }
  };
  dwh_with_form(c.form, walk);
}
