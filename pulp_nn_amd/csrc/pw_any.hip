// Host side of pw_any.h: blocks of channels, grid and launch.
#include "host.h"

#include <algorithm>

#include "pw_any.h"

namespace {

template <int KS, int NP, int NW>
bool launch_mode(int mode, const PwAnyGeom &g, const EpiArgs &e, hipStream_t s)
{
  const dim3 grid((unsigned)(g.nwg * g.nblk)), block(64 * NW);
  const size_t lds = (size_t)pw_any_lds(KS, NP, NW);
  switch (mode) {
    case EPI_BN:
      if (!raise_lds_limit<pw_any_kernel<KS, NP, EPI_BN, NW>>(lds)) return false;
      hipLaunchKernelGGL((pw_any_kernel<KS, NP, EPI_BN, NW>), grid, block, lds, s, g, e);
      break;
    case EPI_MULT:
      if (!raise_lds_limit<pw_any_kernel<KS, NP, EPI_MULT, NW>>(lds)) return false;
      hipLaunchKernelGGL((pw_any_kernel<KS, NP, EPI_MULT, NW>), grid, block, lds, s, g, e);
      break;
    default:
      if (!raise_lds_limit<pw_any_kernel<KS, NP, EPI_RAW, NW>>(lds)) return false;
      hipLaunchKernelGGL((pw_any_kernel<KS, NP, EPI_RAW, NW>), grid, block, lds, s, g, e);
      break;
  }
  return true;
}

template <int KS, int NW>
bool launch_np(int np, int mode, const PwAnyGeom &g, const EpiArgs &e, hipStream_t s)
{
  if (np == 1) return launch_mode<KS, 1, NW>(mode, g, e, s);
  if (np == 2) return launch_mode<KS, 2, NW>(mode, g, e, s);
  if (np == 3) return launch_mode<KS, 3, NW>(mode, g, e, s);
  return launch_mode<KS, 4, NW>(mode, g, e, s);
}

}  // namespace

bool launch_pw_any(int mode, const uint8_t *in, const int8_t *w, const int8_t *bias, uint8_t *out, long long M, int N, int K,
                   const EpiArgs &e, int cus, hipStream_t s)
{
  if (K > 512 || N < 16 || M * K < 16 || (long long)N * K < 16 || M > 0x7fffffffLL || mode == EPI_OUT32) return false;
  PwAnyGeom g = {};
  g.in = in;
  g.w = w;
  g.bias = bias;
  g.out = out;
  g.M = (int)M;
  g.N = N;
  g.K = K;
  const int ks = K <= 64 ? 1 : K <= 128 ? 2 : K <= 256 ? 4 : 8;
  const int nw = ks <= 2 ? 16 : 8;
  // blocks of at most 256 channels whose weights fit LDS beside the output tiles
  int np_max = 4;
  while (np_max > 1 && pw_any_lds(ks, np_max, nw) > 160 * 1024 - 512) np_max--;
  g.nblk = (N + 64 * np_max - 1) / (64 * np_max);
  g.NB = g.nblk == 1 ? N : ((N + g.nblk - 1) / g.nblk + 3) & ~3;
  if (g.nblk > 1 && N - (g.nblk - 1) * g.NB < 16) return false;  // (a last block of fewer channels than a piece)
  if (g.nblk > 1 && (N & 3)) return false;
  const int np = (g.NB + 63) / 64;
  g.units = (int)((M + 15) / 16);
  g.nt = M * N >= PULPNN_NT_BYTES;
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
  if (ks == 1) return launch_np<1, 16>(np, mode, g, e, s);
  if (ks == 2) return launch_np<2, 16>(np, mode, g, e, s);
  if (ks == 4) return launch_np<4, 8>(np, mode, g, e, s);
  return launch_np<8, 8>(np, mode, g, e, s);
}
