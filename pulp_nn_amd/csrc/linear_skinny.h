// Skinny GEMM for linear layers with few rows (batch <= 256): weights stream, activations stay.
//
// pulp_nn_linear / pulp_nn_linear_out_32 (32bit/src/pulp_nn_linear.c:58-108, pulp_nn_linear_out_32.c) at small batch are
// bound by reading the weight matrix once; a tiled GEMM with a barrier per 64-byte K slice spends its time on per-slice
// latency instead (16 sequential slices for K = 1024).  Here a workgroup of four waves owns 16 output neurons.  The waves
// split the work by blocks of 64 rows and, when there are fewer than four such blocks, by parts of K as well (when the
// neurons alone make too few workgroups for the machine, the row blocks go to separate workgroups and K is always split in
// four).  A K slice of 64 bytes is up to five fragments: 16 weight rows and four times 16 activation rows (as many as there
// are; shared by all workgroups and therefore cache resident).  They travel straight to the wave's own part of LDS, four
// slices in flight, four lanes to the 64 bytes of a row: in MFMA operand layout, sixteen rows side by side, a load keeps the
// address unit 56 to 64 clocks instead of 16.  The sums of the weight rows come from one more MFMA against ones.  The K parts
// meet in LDS at the end, and each of the waves that share a block of rows finishes a part of it, with the channel
// constants that it has asked for at the start.
//
// Rows of any length from 16 bytes on at any address (ANY): the last chunk of a row is its LAST 16 bytes, so that no load leaves a
// tensor; the bytes the chunk before has counted already are zeroed in the weight operand.
//
// Bound: one trip to memory, the instructions of a wave, launch.  Whole calls, operands straight to registers in operand layout, then bias,
// k and lambda as a second trip and the epilogue of all rows on one wave of four / now: 64 rows 1024 -> 4096 64-bit 6.26 / 5.0 us (4.5 MB), 256 rows 4096 -> 4096 38.9 / 25.7,
// 256 rows 1024 -> 1000 5.9 / 4.7, 1 row 4096 -> 4096 7.2 / 7.0; rows that are not whole chunks: 178 rows 258 -> 1712 18.4 / 4.3, 64 rows 4001 ->
// 3001 28.5 / 11.2, 64 rows 1000 -> 1000 5.2 / 4.6; over 90 layers the mean is 0.75, none slower.
// (Rows that are not whole chunks, on the tiled kernel with its byte gather: 1 row 1003 -> 1000 62.6 us, 64 rows 1000 -> 1000 64.6.)
//
// Arithmetic as in igemm.h: activations as a ^ 0x80 with bias + 128 * sum_k w added back.
#pragma once
#include "igemm.h"
#include "requant.h"

struct SkinnyGeom {
  const uint8_t *in;   // [M][K]
  const int8_t *w;     // [N][K]
  const int8_t *bias;  // int8 [N]; int32 [N] for EPI_OUT32; may be null
  void *out;           // [M][N] uint8, or int32 for EPI_OUT32
  int M, N, K;         // M <= 256, K >= 16
  int kparts, lkparts; // 4, 2 or 1 parts of K (and its logarithm); a workgroup takes 4 / kparts blocks of 64 rows, gridDim.y the rest
  int vec4;            // N and the output are multiples of 4
};
#define SKINNY_SLOT (5 * 1024)            // one K slice: weights, four groups of 16 rows
#define SKINNY_LDS (4 * 4 * SKINNY_SLOT)  // four slices of four waves: two workgroups fill a compute unit

template <int MODE, bool ANY>
__device__ __forceinline__ void linear_skinny(SkinnyGeom g, EpiArgs e)
{
  extern __shared__ __attribute__((aligned(16))) unsigned char skinny_lds[];
  typedef __attribute__((address_space(3))) void *lds_ptr_t;
  asm volatile("" : "+s"(g.in), "+s"(g.w), "+s"(g.bias), "+s"(g.out), "+s"(g.M), "+s"(g.N), "+s"(g.K), "+s"(g.kparts), "+s"(g.lkparts), "+s"(g.vec4),
               "+s"(e.k), "+s"(e.lambda), "+s"(e.mult), "+s"(e.shift));
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, lgrp = lane >> 4;
  const int n0 = blockIdx.x * 16;  // this workgroup's 16 neurons
  const int KT = (g.K + 63) / 64;
  // block of 64 rows (blockIdx.y counts the row blocks that other workgroups of the same neurons take), part of K
  const int rb = (blockIdx.y << (2 - g.lkparts)) + (wave >> g.lkparts), kp = wave & (g.kparts - 1);
  const int mb = rb * 64;
  const int kt0 = (KT * kp) >> g.lkparts, kt1 = (KT * (kp + 1)) >> g.lkparts;
  const int ns = min(max((g.M - mb + 15) >> 4, 0), 4);  // groups of 16 rows that exist
  const int slices = ns ? kt1 - kt0 : 0;

  // ---- the K slices on their way to LDS --------------------------------------------------------------------------------
  // Lane: 16 bytes of row lane / 4; which of the four fetches which depends on the row, so that fragment reads meet different banks.
  // Rows and chunks that do not exist are out of range.
  unsigned char *stage = skinny_lds + wave * (4 * SKINNY_SLOT);
  const int lrow = lane >> 2, lchunk = 16 * ((lane & 3) ^ ((lrow >> 1) & 3));
  const int wrows = min(16, g.N - n0), arows = min(64, g.M - mb);
  auto issue = [&](int i) {
    const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc((void *)(g.w + (long long)n0 * g.K), 0, wrows * g.K, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void *)(g.in + (long long)mb * g.K), 0, arows * g.K, 0x00020000);
    unsigned char *slot = stage + (i & 3) * SKINNY_SLOT;
    const int p = 64 * (kt0 + i) + lchunk;
    const unsigned off = p < g.K ? (unsigned)(lrow * g.K + (ANY ? min(p, g.K - 16) : p)) : 0x80000000u;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_w, (lds_ptr_t)slot, 16, (int)off, 0, 0, 0);
#pragma unroll
    for (int s = 0; s < 4; s++)
      if (s < ns) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_ptr_t)(slot + 1024 * (s + 1)), 16, (int)(off + (unsigned)(16 * s * g.K)), 0, 0, 0);
  };
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (i < slices) issue(i);

  // ---- the constants of the lane's four neurons ---------------------------------------------------------------------------
  const int nb = n0 + 4 * lgrp;
  int bias[4] = {0, 0, 0, 0};
  bn_t kk[4] = {0, 0, 0, 0}, ll[4] = {0, 0, 0, 0};
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int n = min(nb + r, g.N - 1);
    if (g.bias) bias[r] = (MODE == EPI_OUT32) ? ((const int *)g.bias)[n] : (int)g.bias[n];
    if (MODE == EPI_BN) {
      kk[r] = e.k[n];
      ll[r] = e.lambda[n];
    }
  }

  // ---- multiply -----------------------------------------------------------------------------------------------------------
  // the bytes of a row's last chunk that the chunk before does not hold
  [[maybe_unused]] v4i tail;
  if constexpr (ANY) {
    const int skip = (16 - g.K % 16) % 16;
#pragma unroll
    for (int d = 0; d < 4; d++) tail[d] = (int)high_bits(8 * skip - 32 * d);
  }
  v4i acc[4], wacc = {0, 0, 0, 0};
#pragma unroll
  for (int s = 0; s < 4; s++) acc[s] = (v4i){0, 0, 0, 0};
  const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
  const int frag = l16 * 64 + ((lgrp ^ ((l16 >> 1) & 3)) << 4);
#pragma unroll 1
  for (int i = 0; i < slices; i++) {
    // this slice has arrived when no more than the three behind it are on their way (vmcnt: 3 * (1 + ns))
    if (i + 3 >= slices) __builtin_amdgcn_s_waitcnt(0x0F70);
    else if (ns == 4) __builtin_amdgcn_s_waitcnt(0x0F70 | 15);
    else if (ns == 3) __builtin_amdgcn_s_waitcnt(0x0F70 | 12);
    else if (ns == 2) __builtin_amdgcn_s_waitcnt(0x0F70 | 9);
    else __builtin_amdgcn_s_waitcnt(0x0F70 | 6);
    asm volatile("" ::: "memory");
    const unsigned char *slot = stage + (i & 3) * SKINNY_SLOT + frag;
    v4i wf = *(const v4i *)slot, af[4];
#pragma unroll
    for (int s = 0; s < 4; s++) af[s] = *(const v4i *)(slot + 1024 * (s + 1));  // (groups that do not exist: whatever is there)
    if (i + 4 < slices) {
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the slice has been read
      issue(i + 4);
    }
    if (ANY && 64 * (kt0 + i) + 16 * lgrp + 16 > g.K) wf &= tail;
    wacc = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf, ones, wacc, 0, 0, 0);
#pragma unroll
    for (int s = 0; s < 4; s++) acc[s] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf, af[s] ^ (int)0x80808080, acc[s], 0, 0, 0);
  }

  // ---- the K parts of a block of rows meet in LDS, and each of its waves takes 4 / kparts groups of 16 rows -----------------------
  v4i *part = (v4i *)skinny_lds;  // [wave][weights, s][lane]
  if (g.kparts > 1) {
    __syncthreads();  // (everybody has read the slices that lay there)
    part[(wave * 5) * 64 + lane] = wacc;
#pragma unroll
    for (int s = 0; s < 4; s++) part[(wave * 5 + 1 + s) * 64 + lane] = acc[s];
    __syncthreads();
  }
  const int per = 4 >> g.lkparts, first = wave - kp;
  if (g.kparts > 1) {
    wacc = part[(first * 5) * 64 + lane];
    for (int q = 1; q < g.kparts; q++) wacc += part[((first + q) * 5) * 64 + lane];
  }

  // ---- epilogue: acc[s][r] = neuron nb + r of row mb + 16*s + l16 ------------------------------------------------------------------
  int corr[4];
  bool ks = true;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    corr[r] = 128 * wacc[r] + bias[r];
    ks = ks && bn_k_small(kk[r]);
  }
  const bool k_small = __all(ks);
  const bool acc24 = g.K <= 256;
  constexpr int QM = MODE == EPI_OUT32 ? EPI_RAW : MODE;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int s = kp * per + j, m = mb + 16 * s + l16;
    if (j >= per || s >= ns) break;
    v4i a = acc[j];
    if (g.kparts > 1) {
      a = part[(first * 5 + 1 + s) * 64 + lane];
      for (int q = 1; q < g.kparts; q++) a += part[((first + q) * 5 + 1 + s) * 64 + lane];
    }
    if (m >= g.M) continue;
    const int a0 = a[0] + corr[0], a1 = a[1] + corr[1], a2 = a[2] + corr[2], a3 = a[3] + corr[3];
    if constexpr (MODE == EPI_OUT32) {
      int *o = (int *)g.out + (long long)m * g.N + nb;
      const int v[4] = {a0, a1, a2, a3};
#pragma unroll
      for (int r = 0; r < 4; r++)
        if (nb + r < g.N) o[r] = v[r];
    } else {
      const unsigned p = acc24 ? requant4<QM, true>(a0, a1, a2, a3, kk, ll, k_small, e.mult, e.shift)
                               : requant4<QM, false>(a0, a1, a2, a3, kk, ll, k_small, e.mult, e.shift);
      uint8_t *o = (uint8_t *)g.out + (long long)m * g.N + nb;
      if (g.vec4 && nb < g.N) {
        *(unsigned *)o = p;
      } else {
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (nb + r < g.N) o[r] = (uint8_t)(p >> (8 * r));
      }
    }
  }
}

template <int MODE>
__global__ __launch_bounds__(256) void linear_skinny_kernel(SkinnyGeom g, EpiArgs e) { linear_skinny<MODE, false>(g, e); }
template <int MODE>
__global__ __launch_bounds__(256) void linear_skinny_any_kernel(SkinnyGeom g, EpiArgs e) { linear_skinny<MODE, true>(g, e); }
