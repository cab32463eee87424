// Depthwise 3x3 + pointwise 1x1 in one kernel: the block of a MobileNet-style network.
//
// The reference runs the two layers as separate calls with the depthwise result written to memory in
// HWC (32bit/src/pulp_nn_depthwise_generic.c:179) and read back pixel by pixel by the next layer
// (pulp_nn_pointwise_HoWo_parallel.c:103).  Here the intermediate tensor never exists in memory, and a block is one launch
// instead of two.  Both layers apply their own requantisation exactly as the separate kernels do, so the result is
// bit-identical to the two-call sequence.
//
// A workgroup brings its tile's input into LDS as a ^ 0x80, with the padding around it, and the depthwise layer's parameters; the depthwise
// stage multiplies on the matrix cores with diagonal weight operands (dw_hwc.h): a wave takes 16 channels of a strip of 16 pixels
// down the strip's rows, an operand is one ds_read_b128 and serves up to three output rows; the requantised bytes go to LDS in the form
// of the pointwise layer's activation operand.  The pointwise stage multiplies blocks of 64 pixels x 16 channels.  A wave's weights
// travel to its own part of LDS from the start of the kernel on, four lanes fetching the 64 contiguous bytes of a row: fetched in operand
// layout, sixteen rows side by side, every lane's 16 bytes cost the address unit a cycle of their own, four times as long.
// 128 * (sum of the weights) comes from one more MFMA per operand against ones and is folded into lambda.  Four bytes of four
// pixels change places between lanes before the store, so that a lane writes 16 bytes of one pixel.
//
// Several blocks of one shape (stride 1, as many channels out as in) run back to back in one launch: tiles are whole images then,
// a block's output goes to LDS where the input was, and only the last block's output leaves the chip (dwpw_chain.h for runs whose
// stages give each wave one item).
//
// Bound: the chain parameters and input -> LDS -> multiply -> LDS -> multiply -> store, and the instructions of a wave in it, some 900
// with 128 channels, 8 clocks for one that needs the one before; large batches by that chain too, two to four workgroups per compute unit
// covering each other.  What a block reads from memory is asked for in one trip, the input first (some 2000 clocks from another XCD's
// writes), then the parameters straight to LDS, the weights, and the constants of the pointwise stage; two 16-byte loads of input a lane at a
// time (four cost 14 registers, one wave of five per SIMD and on 64x64x16 -> 32 batch 256 2.5 us).  With the parameters through
// registers, array by array, and each number of the launch read where it is used, a wave took 10800 clocks from end to end on 64x64x16 ->
// 32, now 8200.  Call by call, before that / now: 64x64x16 -> 32 batch 1 5.0 / 4.15 us, batch 256 24.7 / 23.0; 64x64x32 -> 64 stride 2
// batch 256 21.0 / 17.8; 32x32x64 batch 1 5.3 / 4.5; 16x16x128 batch 64 6.4 / 5.9; 16x16x64 -> 128 6.1 / 5.2.  (With the vector-ALU
// depthwise stage 64x64x16 -> 32 was 13.6 and 42.4.)
#pragma once
#include <stddef.h>

#include "dw_hwc.h"
#include "dwpw_geom.h"

#define DWPW_MAX_BLOCKS 8  // blocks of one launch (pulp_nn_hip_dw_pw_chain_hwc)

// one depthwise + pointwise block
struct DwPwBlock {
  const int8_t *dw_wt;    // [C][3][3]
  const int8_t *dw_bias;  // int8 [C] or null
  const int8_t *pw_w;     // [Co][C]
  const int8_t *pw_bias;  // int8 [Co] or null
  EpiArgs e_dw, e_pw;     // k, lambda, multiplier, shift of either layer
  int mode_dw, mode_pw;   // requantisation branch of either layer (EPI_BN, EPI_MULT, EPI_RAW)
};

struct DwPwGeom {
  const uint8_t *in;      // HWC [B][H][W][C]
  uint8_t *out;           // HWC [B][Ho][Wo][Co]
  DwPwTile t;
  int nblocks;
  DwPwBlock blk[DWPW_MAX_BLOCKS];
};

// Requantisation of channels first .. first + 3 as kk * acc + ll, from the parameters in LDS and the sums of their weights.  Returns
// whether the multipliers are small.
__device__ __forceinline__ bool dwpw_fold(const unsigned char *par, int C, int first, const v4i &wsum, int mode, int mult, bn_t (&kk)[4], bn_t (&ll)[4])
{
  const DwPwPar at = dwpw_par(C, (int)sizeof(bn_t), false);
  const unsigned b = *(const unsigned *)(par + first);
  typedef bn_t bn4 __attribute__((ext_vector_type(4)));
  const bn4 k = *(const bn4 *)(par + at.k + first * (int)sizeof(bn_t)), l = *(const bn4 *)(par + at.l + first * (int)sizeof(bn_t));
  bool ks = true;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int corr = 128 * wsum[r] + (int)(int8_t)(b >> (8 * r));
    kk[r] = mode == EPI_BN ? k[r] : (bn_t)mult;
    ks = ks && bn_k_small(kk[r]);
#if PULPNN_BN_BITS == 64
    if (mode == EPI_BN) ll[r] = (bn_t)((unsigned long long)kk[r] * (unsigned long long)(long long)corr + (unsigned long long)l[r]);
    else
#endif
      ll[r] = (bn_t)(int)((unsigned)kk[r] * (unsigned)corr + (unsigned)l[r]);  // (lambda: zero without batch-norm)
  }
  return ks;
}

// s_waitcnt vmcnt(n), n < 16
#define DWPW_WAIT_VM(n) (0x0F70 | (n))

// This wave's LDS accesses done, then the workgroup's barrier.  (__syncthreads() would also wait for the weights on their way to LDS, which
// only the wave that asked for them reads.)
__device__ __forceinline__ void dwpw_barrier()
{
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// One block's parameters in the kernel's argument segment, through a pointer the compiler cannot see through: loaded when a stage
// needs them, not all of them up front into scalar registers that there are not enough of.
typedef const __attribute__((address_space(4))) DwPwBlock *DwPwBlockArg;
__device__ __forceinline__ DwPwBlockArg dwpw_block(int j)
{
  typedef const __attribute__((address_space(4))) char *bytes_t;
  bytes_t p = (bytes_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return (DwPwBlockArg)(p + offsetof(DwPwGeom, blk)) + j;
}
// ... and bytes per 64-byte slice of K of the activation operand.
__device__ __forceinline__ int dwpw_act_step()
{
  typedef const __attribute__((address_space(4))) char *bytes_t;
  bytes_t p = (bytes_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return 64 * *(const __attribute__((address_space(4))) int *)(p + offsetof(DwPwGeom, t) + offsetof(DwPwTile, act_px));
}

// One layer's parameters to LDS (DwPwPar) by the workgroup as a whole, 1 KB an instruction: sixteen waves that each fetch their own 16
// channels' into registers keep the address units busy for 2500 cycles a block.
// Every one of the waves asks for its share (loads without a source are out of range: zeros).  Filter and bias 4-byte aligned.
__device__ __forceinline__ void dwpw_par_load(unsigned char *par, const int8_t *filter, const int8_t *bias, const bn_t *k, const bn_t *lambda, bool bn, int C, int wave,
                                              int waves, int lane)
{
  typedef __attribute__((address_space(3))) void *lds_ptr_t;
  const DwPwPar at = dwpw_par(C, (int)sizeof(bn_t), filter != nullptr);
  for (int to = 1024 * wave; to < at.bytes; to += waves * 1024) {
    const DwPwParPiece p = dwpw_par_piece(at, C, (int)sizeof(bn_t), bias != nullptr, bn, to);
    const char *src = (p.array == 0 ? (const char *)bias : p.array == 1 ? (const char *)k : p.array == 2 ? (const char *)lambda : (const char *)filter) + p.first;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)src, 0, p.bytes, 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)(par + to), 16, 16 * lane, 0, 0, 0);
  }
}

// W, S: input width, stride.  KP: slices of K whose weights are in LDS at once.  CHAIN: g.nblocks blocks back to back; otherwise the
// one block g.blk[0].
template <int W, int S, int KP, bool CHAIN, bool LEAN = false>
__global__ __launch_bounds__(1024) void dwpw_kernel(DwPwGeom g)
{
  extern __shared__ __attribute__((aligned(16))) unsigned char dwpw_lds[];
  typedef unsigned v4u __attribute__((ext_vector_type(4)));
  typedef bn_t bn4 __attribute__((ext_vector_type(4), aligned(sizeof(bn_t))));
  typedef __attribute__((address_space(3))) void *lds_ptr_t;
  constexpr int WO = W / S;
  DwPwTile &T = g.t;
  // The launch's numbers at once and opaque (as in dw_mfma_kernel), the block's pointers with them.
  asm volatile("" : "+s"(T.C), "+s"(T.H), "+s"(T.Ho), "+s"(T.Co), "+s"(T.whole), "+s"(T.NI), "+s"(T.TR), "+s"(T.lpxb), "+s"(T.R), "+s"(T.nst),
               "+s"(T.CS), "+s"(T.XR), "+s"(T.pitch), "+s"(T.x_off), "+s"(T.waves));
  asm volatile("" : "+s"(T.lsplit), "+s"(T.cf_per), "+s"(T.par_off), "+s"(T.w_off), "+s"(T.bands), "+s"(T.slabs), "+s"(T.act_px), "+s"(g.in),
               "+s"(T.nrb), "+s"(T.B));
  DwPwBlock only = g.blk[0];
  if constexpr (!CHAIN)
    asm volatile("" : "+s"(only.dw_wt), "+s"(only.dw_bias), "+s"(only.pw_w), "+s"(only.pw_bias), "+s"(only.e_dw.k), "+s"(only.e_dw.lambda),
                 "+s"(only.e_pw.k), "+s"(only.e_pw.lambda), "+s"(only.e_dw.shift), "+s"(only.e_pw.shift), "+s"(only.mode_dw), "+s"(only.mode_pw));
  auto block = [&](int j) {
    if constexpr (CHAIN) return dwpw_block(j);
    else return (const DwPwBlock *)&only;
  };
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, lgrp = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), NWV = T.waves, NTH = 64 * NWV;
  const int part = blockIdx.x & ((1 << T.lsplit) - 1);
  const DwPwPlace at = dwpw_place<WO>(T, blockIdx.x >> T.lsplit);
  const bool narrow = KP == 1 && T.C < 64;
  const int KT = (T.C + 63) / 64;
  unsigned char *xin = dwpw_lds + T.x_off, *par = dwpw_lds + T.par_off;
  const int nblocks = CHAIN ? g.nblocks : 1;
  // The input's first part (10 registers) and the pointwise constants (9, of 64 bits 17) are asked for ahead of the depthwise stage, unless they do not
  // fit beside it.  In chains with constants of 64 bits they were spilled, 14 to 22 registers a lane, and in single blocks they left four
  // waves a SIMD where there had been five; with eight slices of weights they hold those up.  There they are asked for where they are
  // used.  Ahead / so: chains 8x8x320 two blocks batch 64 21.0 / 18.1 us, four batch 128 36.0 / 31.8; 8x8x64 four batch 256 17.1 / 14.6; blocks
  // 64x64x16 -> 32 batch 256 33.2 / 30.0, 8x8x256 batch 64 8.3 / 7.5, 4x4x512 11.0 / 10.6; 32 bits, eight slices: 8x8x512 -> 64 stride 2 9.1 /
  // 8.7.  (With 32 bits otherwise ahead is the better: 8x8x64 two blocks batch 64 7.5 / 7.95; 64x64x16 -> 32 23.2 / 24.6.)
  constexpr bool WIDE = sizeof(bn_t) == 8, X_AHEAD = !WIDE || (!CHAIN && KP > 1), PW_AHEAD = !WIDE && KP < 8 && !LEAN;
  // Weights: one slice, behind the input; eight, in front of it; four, behind the input and the parameters, where those have been waited for (constants of
  // 64 bits: at once).  Eight waited for / in front: 8x8x512 -> 64 stride 2 batch 64 9.15 / 8.9; four at once, 32 bits: 8x8x256 -> 512 stride
  // 2 6.7 / 7.0, 64 bits 7.8 / 7.7.
  constexpr bool W_FIRST = KP == 8, W_AT_ONCE = WIDE && !CHAIN && KP == 4;

  // the pointwise stage's blocks of 64 pixels x 16 channels, dealt to the waves
  const int cf_lo = part * T.cf_per, nblk = max(min(T.cf_per, T.Co / 16 - cf_lo), 0) << T.lpxb;
  unsigned char *wl = dwpw_lds + T.w_off + wave * (1024 * KP);  // the wave's own weights: KP slices of 16 rows of 64 bytes
  int w_cf = -1;                                                // channels whose first slices are there, or on their way
  auto load_w = [&](auto P, int cf, int kt0) {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)P->pw_w, 0, (unsigned)T.Co * (unsigned)T.C, 0x00020000);
    const unsigned off = dwpw_w_lane(T.C, cf, lane, KP == 1);
#pragma unroll
    for (int kk = 0; kk < KP; kk++) {
      const DwPwWeight at = KP == 1 ? DwPwWeight{off, 64 * kt0} : dwpw_w_slice(T.C, off, kt0 + kk);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)(wl + 1024 * kk), 16, at.off, at.add, 0, 0);
    }
  };
  const int cgs = T.CS / 16, nitems = cgs * T.nst;  // items of the depthwise stage: 16 channels of a strip

#pragma unroll 1
  for (int j = 0; j < nblocks; j++) {
    const bool first = !CHAIN || j == 0, last = !CHAIN || j == nblocks - 1;
    // ---- one trip to memory: the input's first part, weights and depthwise parameters on their way to LDS, the constants of the wave's
    // first block of the pointwise stage ------------------------------------------------------------------------------------------
    const auto P = block(j);
    const int cf_first = cf_lo + (wave >> T.lpxb);
    constexpr int UN = 2;  // 16-byte loads in flight per lane
    v4u v[UN];
    int to[UN];
    const int chunks = dwpw_chunks<W>(T);
    // (t0: the wave's first chunk; what none of its lanes needs is left out)
    auto load_x = [&](int slab, int t0) {
      const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(g.in + (dwpw_first_row<S>(T, at) * W) * T.C + slab * T.CS), 0,
                                                                            (dwpw_rows_in(T) * W) * T.C - slab * T.CS, 0x00020000);
#pragma unroll
      for (int u = 0; u < UN; u++) {
        if (t0 + NTH * u >= chunks) break;
        const DwPwChunk c = dwpw_chunk<W, S>(T, at, t0 + lane + NTH * u);
        to[u] = c.lds;
        v[u] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, c.off >= 0 ? (unsigned)c.off : 0x80000000u, 0, 0);
      }
    };
    if constexpr (W_FIRST)
      if (wave < nblk) load_w(P, w_cf = cf_first, 0);
    if (X_AHEAD && first) load_x(0, 64 * wave);
    if (KP == 1 && wave < nblk) load_w(P, w_cf = cf_first, 0);
    if ((((unsigned)(unsigned long long)P->dw_wt | (unsigned)(unsigned long long)P->dw_bias) & 3) == 0) {
      dwpw_par_load(par, P->dw_wt, P->dw_bias, P->e_dw.k, P->e_dw.lambda, P->mode_dw == EPI_BN, T.C, wave, NWV, lane);
    } else {
      const DwPwPar off = dwpw_par(T.C, (int)sizeof(bn_t), true);
      const int8_t *wt = P->dw_wt, *bias = P->dw_bias;
      for (int i = tid; i < 9 * T.C; i += NTH) par[off.f + i] = (unsigned char)wt[i];
      for (int i = tid; i < T.C; i += NTH) par[i] = bias ? (unsigned char)bias[i] : 0;
      const bool bn = P->mode_dw == EPI_BN;
      const bn_t *k = P->e_dw.k, *l = P->e_dw.lambda;
      for (int i = tid; i < T.C; i += NTH) {
        *(bn_t *)(par + off.k + i * (int)sizeof(bn_t)) = bn ? k[i] : (bn_t)0;
        *(bn_t *)(par + off.l + i * (int)sizeof(bn_t)) = bn ? l[i] : (bn_t)0;
      }
    }
    // the constants of the lane's four channels of output
    int bias = 0;
    bn4 k = {0, 0, 0, 0}, l = {0, 0, 0, 0};
    auto load_pw = [&](int cf) {
      const int n = 16 * cf + 4 * lgrp;
      if (P->pw_bias) bias = *(const i32_u *)(P->pw_bias + n);
      if (P->mode_pw == EPI_BN) {
        k = *(const bn4 *)(P->e_pw.k + n);
        l = *(const bn4 *)(P->e_pw.lambda + n);
      }
    };
    if constexpr (W_AT_ONCE)
      if (wave < nblk) load_w(P, w_cf = cf_first, 0);
    if constexpr (PW_AHEAD)
      if (wave < nblk) load_pw(cf_first);
#pragma unroll 1
    for (int slab = 0; slab < (CHAIN ? 1 : T.slabs); slab++) {
      // ---- input -> LDS ------------------------------------------------------------------------------------------------
      if (first) {
        if (slab) dwpw_barrier();  // everybody is done with the slab before
#pragma unroll 1
        for (int t0 = 64 * wave; t0 < chunks; t0 += NTH * UN) {
          if (!X_AHEAD || slab || t0 != 64 * wave) load_x(slab, t0);
#pragma unroll
          for (int u = 0; u < UN; u++) {
            if (t0 + NTH * u >= chunks) break;
            if (t0 + lane + NTH * u < chunks) *(v4i *)(xin + to[u]) = (v4i){(int)v[u].x, (int)v[u].y, (int)v[u].z, (int)v[u].w} ^ (int)0x80808080;
          }
        }
      }
      if (slab == 0) {
        __builtin_amdgcn_s_waitcnt(DWPW_WAIT_VM(0));  // (a wave without input has parameters on their way to LDS)
        if (KP == 4 && !W_AT_ONCE && wave < nblk) load_w(P, w_cf = cf_first, 0);
      }
      dwpw_barrier();

      // ---- depthwise stage ---------------------------------------------------------------------------------------------
      const int mode = P->mode_dw, shift = P->e_dw.shift;
      const unsigned char *filter = par + dwpw_par(T.C, (int)sizeof(bn_t), true).f + l16 * 9 + min(lgrp, 2);
      const int act_step = CHAIN ? 4096 << T.lpxb : dwpw_act_step();
      DwhChannels<1> c;
      int set = -1;  // channel group that c holds
#pragma unroll 1
      for (int it = wave; it < nitems; it += NWV) {
        const int st = (int)fastdiv((unsigned)it, T.d_n), cg = it - st * cgs, ch = slab * T.CS + 16 * cg;
        if (!CHAIN && ch >= T.C) continue;  // (the last slab may have fewer channels)
        if (set != cg) {
          const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
          v4i s = {0, 0, 0, 0};
#pragma unroll
          for (int fy = 0; fy < 3; fy++) {
            const int v = lgrp < 3 ? (int)filter[9 * ch + 3 * fy] << (8 * (l16 & 3)) : 0;
#pragma unroll
            for (int d = 0; d < 4; d++) c.A[0][fy][d] = (l16 >> 2) == d ? v : 0;
            s = __builtin_amdgcn_mfma_i32_16x16x64_i8(c.A[0][fy], ones, s, 0, 0, 0);
          }
          const bool ks = dwpw_fold(par, T.C, ch + 4 * lgrp, s, mode, mode == EPI_MULT ? P->e_dw.mult : 1, c.kk[0], c.ll[0]);
          c.form = dwh_form(mode, shift, (bool)__all(ks), true);
          set = cg;
        }
        const DwPwLane n = dwpw_lane<W, S>(T, st, l16, min(lgrp, 2));
        const unsigned char *src = xin + n.x + 16 * cg;
        const int rowb = (W + 2) * T.pitch;
        int px = n.px;
        auto next = [&]() {
          const v4i v = *(const v4i *)src;
          src += rowb;
          return v;
        };
        auto put = [&](unsigned v) {
          if (n.live) *(unsigned *)(dwpw_lds + DWPW_ACT_AT(narrow, T.C, act_step, px, ch) + 4 * lgrp) = v ^ 0x80808080u;
          px += WO;
        };
        dwh_with_form(c.form, [&](auto form) { dwh_walk<S, decltype(form)::value>(c, shift, T.R, next, put); });
      }
    }
    // ---- pointwise stage ---------------------------------------------------------------------------------------------------
    const int mode = P->mode_pw, shift = P->e_pw.shift, act_step = CHAIN ? 4096 << T.lpxb : dwpw_act_step();
    __builtin_amdgcn_s_waitcnt(DWPW_WAIT_VM(0));  // this wave's weights
    dwpw_barrier();
#pragma unroll 1
    for (int blk = wave; blk < nblk; blk += NWV) {
      const int cf = cf_lo + (blk >> T.lpxb), px0 = 64 * (blk & ((1 << T.lpxb) - 1));
      if constexpr (!PW_AHEAD) {
        bias = 0;
        k = l = (bn4){0, 0, 0, 0};
        load_pw(cf);
      } else if (blk != wave) {
        load_pw(cf);
      }
      const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
      v4i acc[4], wacc = {0, 0, 0, 0};
#pragma unroll
      for (int s = 0; s < 4; s++) acc[s] = (v4i){0, 0, 0, 0};
      // (fewer than 64 channels: the lanes whose chunk does not exist read chunk 0, and meet zero weights)
      const unsigned char *a0 = dwpw_lds + (narrow ? (px0 + l16) * T.C + (16 * lgrp < T.C ? 16 * lgrp : 0) : (px0 + l16) * 64 + ((lgrp ^ ((l16 >> 1) & 3)) << 4));
      const unsigned char *w0 = wl + l16 * 64 + ((lgrp ^ ((l16 >> 1) & 3)) << 4);
      const int sstep = narrow ? 16 * T.C : 1024;
      for (int kt0 = 0; kt0 < KT; kt0 += KP) {
        if (kt0 || w_cf != cf) {
          __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the weights that lie there have been read
          load_w(P, cf, kt0);
          __builtin_amdgcn_s_waitcnt(DWPW_WAIT_VM(0));
          asm volatile("" ::: "memory");
        }
#pragma unroll
        for (int kk = 0; kk < KP; kk++) {
          if (KP == 1 || kt0 + kk < KT) {
            const v4i wf = *(const v4i *)(w0 + 1024 * kk);
            v4i af[4];
#pragma unroll
            for (int s = 0; s < 4; s++) af[s] = *(const v4i *)(a0 + s * sstep);
            a0 += act_step;
            wacc = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf, ones, wacc, 0, 0, 0);
#pragma unroll
            for (int s = 0; s < 4; s++) acc[s] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf, af[s], acc[s], 0, 0, 0);
          }
        }
      }
      w_cf = KT <= KP ? cf : -1;
      // kk * acc + ll, as in the depthwise stage; |acc| <= K * 128 * 128
      const int mult = mode == EPI_MULT ? P->e_pw.mult : 1;
      bn_t kk[4], ll[4];
      bool ks = true;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int corr = 128 * wacc[r] + (int)(int8_t)((unsigned)bias >> (8 * r));
        kk[r] = mode == EPI_BN ? k[r] : (bn_t)mult;
        ks = ks && bn_k_small(kk[r]);
#if PULPNN_BN_BITS == 64
        if (mode == EPI_BN) ll[r] = (bn_t)((unsigned long long)kk[r] * (unsigned long long)(long long)corr + (unsigned long long)l[r]);
        else
#endif
          ll[r] = (bn_t)(int)((unsigned)kk[r] * (unsigned)corr + (unsigned)l[r]);
      }
      // lane: one pixel's 16 channels
      const int px = px0 + lane;
      dwh_with_form(dwh_form(mode, shift, (bool)__all(ks), T.C < 512), [&](auto f) {
        unsigned v[4];
#pragma unroll
        for (int s = 0; s < 4; s++) v[s] = dwh_requant<decltype(f)::value>(acc[s], kk, ll, shift);
        const v4i p = dwh_pixels(v);
        if (px < at.live) {
          if (last) *(v4i *)(g.out + (((long long)at.b0 * T.Ho + at.oy0) * WO + px) * T.Co + 16 * cf) = p;
          else *(v4i *)(xin + dwpw_next_x<W>(T, px) + 16 * cf) = p ^ (int)0x80808080;
        }
      });
    }
  }
}
