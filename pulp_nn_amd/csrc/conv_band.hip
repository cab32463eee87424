// Host side of conv_band.h: tile shape and launch.
#include "host.h"

#include "conv_band.h"

namespace {

template <int TN>
bool launch_tm(int tm, const BandGeom &g, const EpiArgs &e, size_t lds, hipStream_t s)
{
  const dim3 grid((unsigned)g.total), block(256);
  if (tm == 2) {
    if (!raise_lds_limit<conv_band_kernel<TN, 2>>(lds)) return false;
    hipLaunchKernelGGL((conv_band_kernel<TN, 2>), grid, block, lds, s, g, e);
  } else if (tm == 4) {
    if (!raise_lds_limit<conv_band_kernel<TN, 4>>(lds)) return false;
    hipLaunchKernelGGL((conv_band_kernel<TN, 4>), grid, block, lds, s, g, e);
  } else {
    if (!raise_lds_limit<conv_band_kernel<TN, 8>>(lds)) return false;
    hipLaunchKernelGGL((conv_band_kernel<TN, 8>), grid, block, lds, s, g, e);
  }
  return true;
}

}  // namespace

bool launch_conv_band(int mode, const ConvLayer &L, const EpiArgs &e, int cus, hipStream_t s)
{
  BandGeom g;
  int tn, tm;
  size_t lds;
  if (mode == EPI_OUT32 || !band_shape(L, cus, (int)sizeof(bn_t), &g, &tn, &tm, &lds)) return false;
  g.mode = mode;
  if (tn == 1) return launch_tm<1>(tm, g, e, lds, s);
  if (tn == 2) return launch_tm<2>(tm, g, e, lds, s);
  return launch_tm<4>(tm, g, e, lds, s);
}
