// Host side of pw_any.h: blocks of channels, grid and launch.
#include "host.h"

#include "pw_any.h"

namespace {

template <int KS, int NP, int NW>
bool launch_mode(int mode, const PwAnyGeom &g, const EpiArgs &e, hipStream_t s)
{
  const dim3 grid((unsigned)(g.nwg * g.nblk)), block(64 * NW);
  const size_t lds = (size_t)pw_any_lds(KS, NP, NW, (int)sizeof(bn_t));
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
  PwAnyGeom g;
  int ks, np;
  if (mode == EPI_OUT32 || !pw_any_shape(M, N, K, cus, (int)sizeof(bn_t), &g, &ks, &np)) return false;
  g.in = in;
  g.w = w;
  g.bias = bias;
  g.out = out;
  g.nt = M * N >= PULPNN_NT_BYTES;
  if (ks == 1) return launch_np<1, 16>(np, mode, g, e, s);
  if (ks == 2) return launch_np<2, 16>(np, mode, g, e, s);
  if (ks == 4) return launch_np<4, 8>(np, mode, g, e, s);
  return launch_np<8, 8>(np, mode, g, e, s);
}
