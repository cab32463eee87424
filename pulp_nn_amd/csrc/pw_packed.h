// Weights-stationary streaming kernel for large pointwise convolutions 16 -> 16, 16 -> 32 and 32 -> 64
// (pulp_nn_pointwise_HoWo_parallel; the first layers of a MobileNet).
//
// The four 16-byte slots of K of one v_mfma_i32_16x16x64_i8 hold four pixels of 16 channels, or two of 32, instead of one: a load
// is 1 KB of memory in which every lane has a part, and which of the pixels a row of the product sees is decided by the slot its weights
// lie in (zeros in the others).  The rows are dealt so that four products leave a lane 16 consecutive channels of one pixel:
// one 16-byte store a lane, 1 KB in memory order, and no exchange between lanes.  Weights and constants live in registers, a wave
// streams a contiguous run of pixels two loads ahead; no LDS, no barrier.
//
// Bound: HBM and the vector ALU, which has 125 instructions per 64 pixels of 16 -> 32 where pw_stream_kernel has 213 (one pixel a column, three of four lanes of a load
// without a part, 8-byte stores).  Whole calls, that / this: 64x64 16 -> 32 batch 256 12.0 / 10.0 us (50 MB; scalar multiplier 11.7 / 9.2), 16 -> 16
// 10.8 / 7.3 (34 MB, 4.6 TB/s), 32x32 32 -> 64 batch 256 7.8 / 7.1; MobileNet chain at batch 256 166.1 / 163.5.
#pragma once
#include "dw_hwc.h"
#include "pw_stream.h"

// K16: 16-byte chunks of a pixel; Q: 16-channel groups of the output; g.units: loads (of 64 / K16 pixels) in the launch
template <int K16, int Q, bool NT>
__global__ __launch_bounds__(256, 4) void pw_packed_kernel(PwGeom g, EpiArgs e, int mode)
{
  constexpr int K = 16 * K16, N = 16 * Q;
  constexpr int P = 4 / K16, PX = 16 * P;  // pixels of a column, of a load
  constexpr int PS = 4 / Q, SETS = P / PS; // pixels of a column that four products finish; fours of products
  static_assert(SETS >= 1, "a store takes more pixels than a load has");
  const int lane = threadIdx.x & 63, l16 = lane & 15, lgrp = lane >> 4;
  const int wave = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = 4 * (int)gridDim.x;
  int u = (int)((long long)g.units * wave / waves);
  const int u_end = (int)((long long)g.units * (wave + 1) / waves), u_last = max(u_end - 1, 0);

  // (loads past the wave's last one repeat it, pixels past the last one of the launch that one: no branch, a fixed number of loads)
  auto request = [&](int i) {
    const int m = min(PX * min(i, u_last) + 16 * (lgrp / K16) + l16, g.M - 1);
    return *(const v4i *)(g.in + (long long)m * K + 16 * (lgrp % K16));
  };
  v4i b0 = request(u), b1 = request(u + 1);

  // ---- weights and constants -------------------------------------------------------------------------------------------------
  // Row i of product t: channel 16 * ((i / 4) % Q) + 4 * t + i % 4 of pixel PS * h + i / 4 / Q of the column, h the four.
  v4i w[4];
#pragma unroll
  for (int t = 0; t < 4; t++) w[t] = *(const v4i *)(g.w + (16 * ((l16 >> 2) % Q) + 4 * t + (l16 & 3)) * K + 16 * (lgrp % K16));
  typedef bn_t bn4 __attribute__((ext_vector_type(4), aligned(sizeof(bn_t))));
  const int cb = 16 * (lgrp % Q);  // the lane's channels
  v4i bias = {0, 0, 0, 0};
  bn_t kk[4][4], ll[4][4];
  if (g.bias) bias = *(const v4i_u *)(g.bias + cb);
  const bn_t same = mode == EPI_MULT ? (bn_t)e.mult : (bn_t)1;
#pragma unroll
  for (int t = 0; t < 4; t++) {
    bn4 k = {same, same, same, same}, l = {0, 0, 0, 0};
    if (mode == EPI_BN) {
      k = *(const bn4 *)(e.k + cb + 4 * t);
      l = *(const bn4 *)(e.lambda + cb + 4 * t);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
      kk[t][r] = k[r];
      ll[t][r] = l[r];
    }
  }
  v4i A[SETS][4];
#pragma unroll
  for (int h = 0; h < SETS; h++) {
    const int in = lgrp / K16 == PS * h + (l16 >> 2) / Q ? -1 : 0;
#pragma unroll
    for (int t = 0; t < 4; t++) A[h][t] = w[t] & in;
  }
  // k * (acc + corr) + lambda = k * acc + (k * corr + lambda), exact in the wrapping arithmetic of the type
  const v4i zero = {0, 0, 0, 0}, ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
  bool ks = true;
#pragma unroll
  for (int t = 0; t < 4; t++) {
    const v4i s = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[0][t], ones, zero, 0, 0, 0);
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
  const int form = dwh_form(mode, e.shift, (bool)__all(ks), true);  // |acc| <= 32 * 128 * 128

  // ---- pixels ------------------------------------------------------------------------------------------------------------------
  dwh_with_form(form, [&](auto f) {
#pragma unroll 1
    for (; u < u_end; u++) {
      const v4i b2 = request(u + 2);
      const v4i px = b0 ^ (int)0x80808080;
#pragma unroll
      for (int h = 0; h < SETS; h++) {
        v4i o;
#pragma unroll
        for (int t = 0; t < 4; t++) {
          const v4i acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[h][t], px, zero, 0, 0, 0);
          o[t] = (int)dwh_requant<decltype(f)::value>(acc, kk[t], ll[t], e.shift);
        }
        const int m = min(PX * u + 16 * (PS * h + lgrp / Q) + l16, g.M - 1);
        store16<NT>((uint8_t *)g.out + (long long)m * N + cb, o);
        __builtin_amdgcn_sched_barrier(0);  // (the products of the next four stay behind: their registers would be spilled)
      }
      b0 = b1;
      b1 = b2;
    }
  });
}
