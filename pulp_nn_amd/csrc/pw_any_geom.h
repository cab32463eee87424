// Blocks of channels, grid and the waves' runs of pw_any_kernel.  Plain C++: the kernel and its launcher use it, and a host
// program can walk the same numbers.
#pragma once
#include <stdint.h>

#include <algorithm>

#include "fastdiv.h"

// Most pixels of a layer that pw_any_kernel and pw_stream_kernel take: a run's counter goes up to three steps (of 16 and of 32
// pixels) past its end.
static constexpr long long PW_MOST_PIXELS = 0x7fffffffLL - 128;

struct PwAnyGeom {
  const uint8_t *in;   // [M][K]
  const int8_t *w;     // [N][K]
  const int8_t *bias;  // may be null
  uint8_t *out;        // [M][N]
  int M, N, K;
  int NB, nblk;        // channels per block (a multiple of 4 unless nblk == 1), blocks
  int nt;              // write the output with non-temporal stores
  int units;           // 16-pixel units
  int nwg;             // workgroups per block of channels
  FastDiv d_cpr, d_cpr_last;  // division by the 16-byte pieces of a pixel (of a block, of the last block)
};

// LDS: weights, k and lambda, corr, then a private output tile per wave (16 rows of 64 * NP + 20 bytes)
#define PW_ANY_OROW(np) (64 * (np) + 20)
static inline int pw_any_lds(int ks, int np, int nw, int bn_bytes)
{
  return np * 64 * (ks * 64 + 4 + 2 * bn_bytes) + nw * 16 * PW_ANY_OROW(np) + 16;
}

// The pixels [*px, *px_end) of a wave: the units are dealt to the workgroups of a block of channels, and theirs to the waves.
PULPNN_HD void pw_any_run(const PwAnyGeom &g, int wg, int wave, int nw, int *px, int *px_end)
{
  const int ub0 = (int)((long long)g.units * wg / g.nwg), nu = (int)((long long)g.units * (wg + 1) / g.nwg) - ub0;
  const int end = (ub0 + nu * (wave + 1) / nw) * 16;
  *px = (ub0 + nu * wave / nw) * 16;
  *px_end = end < g.M ? end : g.M;
}

// ks: 64-byte slices of K the kernel is made for; np: groups of 64 channels of a block.  False for a layer the kernel does
// not take.
inline bool pw_any_shape(long long M, int N, int K, int cus, int bn_bytes, PwAnyGeom *out, int *ks_out, int *np_out)
{
  if (K > 512 || N < 16 || M * K < 16 || (long long)N * K < 16) return false;
  if (M > PW_MOST_PIXELS) return false;
  PwAnyGeom &g = *out;
  g = PwAnyGeom{};
  g.M = (int)M;
  g.N = N;
  g.K = K;
  const int ks = K <= 64 ? 1 : K <= 128 ? 2 : K <= 256 ? 4 : 8;
  const int nw = ks <= 2 ? 16 : 8;
  // blocks of at most 256 channels whose weights fit LDS beside the output tiles
  int np_max = 4;
  while (np_max > 1 && pw_any_lds(ks, np_max, nw, bn_bytes) > 160 * 1024 - 512) np_max--;
  g.nblk = (N + 64 * np_max - 1) / (64 * np_max);
  g.NB = g.nblk == 1 ? N : ((N + g.nblk - 1) / g.nblk + 3) & ~3;
  if (g.nblk > 1 && N - (g.nblk - 1) * g.NB < 16) return false;  // (a last block of fewer channels than a piece)
  if (g.nblk > 1 && (N & 3)) return false;
  const int np = (g.NB + 63) / 64;
  g.units = (int)((M + 15) / 16);
  // persistent workgroups, one per compute unit, each with at least four units; fewer pixels than give half of the
  // compute units that are better off with kernels that stage no weights
  g.nwg = std::max(1, cus / g.nblk);
  if (g.nblk > 1) g.nwg = std::max(8, g.nwg / 8 * 8);
  const int most = (g.units + 3) / 4;
  if (2 * most < g.nwg) return false;
  // (whole 16-byte chunks: the tiled kernel gathers those well and wins on fewer than eight units per compute unit)
  if (K % 16 == 0 && N % 16 == 0 && g.units < 8 * cus) return false;
  if (g.nblk == 1) g.nwg = std::min(g.nwg, most);
  g.d_cpr = fastdiv_make((unsigned)((g.NB + 15) / 16));
  g.d_cpr_last = fastdiv_make((unsigned)((N - (g.nblk - 1) * g.NB + 15) / 16));
  *ks_out = ks;
  *np_out = np;
  return true;
}
