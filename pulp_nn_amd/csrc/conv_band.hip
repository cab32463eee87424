// Host side of conv_band.h: tile shape and launch.
#include "host.h"

#include "conv_band.h"

namespace {

template <int TN, int TM, int PF>
bool launch(const BandGeom &g, const EpiArgs &e, size_t lds, hipStream_t s)
{
  if (!raise_lds_limit<conv_band_kernel<TN, TM, PF>>(lds)) return false;
  hipLaunchKernelGGL((conv_band_kernel<TN, TM, PF>), dim3((unsigned)g.total), dim3(256), lds, s, g, e);
  return true;
}
template <int TN>
bool launch_tm(int tm, int pf, const BandGeom &g, const EpiArgs &e, size_t lds, hipStream_t s)
{
  if constexpr (TN == 1)
    if (tm == 2 && pf != 2) return pf == 4 ? launch<1, 2, 4>(g, e, lds, s) : launch<1, 2, 1>(g, e, lds, s);
  if constexpr (TN < 4)  // (64 channels a wave: four groups of pixels at the most)
    if (tm == 8) return launch<TN, 8, band_pf(TN, 8)>(g, e, lds, s);
  return tm == 2 ? launch<TN, 2, band_pf(TN, 2)>(g, e, lds, s) : launch<TN, 4, band_pf(TN, 4)>(g, e, lds, s);
}

}  // namespace

bool launch_conv_band(int mode, const ConvLayer &L, const EpiArgs &e, int cus, hipStream_t s)
{
  BandGeom g;
  int tn, tm, pf;
  size_t lds;
  if (mode == EPI_OUT32 || !band_shape(L, cus, (int)sizeof(bn_t), &g, &tn, &tm, &lds, &pf)) return false;
  g.mode = mode;
  if (tn == 1) return launch_tm<1>(tm, pf, g, e, lds, s);
  if (tn == 2) return launch_tm<2>(tm, pf, g, e, lds, s);
  return launch_tm<4>(tm, pf, g, e, lds, s);
}
