// Host side of dw_mfma.h: launch (the tile's shape: dw_mfma_geom.h).
#include "dw_mfma.h"

#include "host.h"

namespace {

template <int CB, int NM>
void launch_mode(int mode, const DwmGeom &g, const EpiArgs &e, size_t lds, hipStream_t s)
{
  const dim3 grid((unsigned)g.total), block(256);
  switch (mode) {
    case EPI_BN: hipLaunchKernelGGL((dw_mfma_kernel<CB, NM, EPI_BN>), grid, block, lds, s, g, e); break;
    case EPI_MULT: hipLaunchKernelGGL((dw_mfma_kernel<CB, NM, EPI_MULT>), grid, block, lds, s, g, e); break;
    default: hipLaunchKernelGGL((dw_mfma_kernel<CB, NM, EPI_RAW>), grid, block, lds, s, g, e); break;
  }
}

template <int CB>
bool launch_cb(int mode, const DwLayer &L, const EpiArgs &e, int cus, hipStream_t s)
{
  DwmGeom g;
  int nm;
  size_t lds;
  if (!dwm_shape<CB>(L, cus, &g, &nm, &lds) || (CB == 64 && !dwm_wide(L, g, cus))) return false;
  if (nm == 1) launch_mode<CB, 1>(mode, g, e, lds, s);
  else if (nm == 2) launch_mode<CB, 2>(mode, g, e, lds, s);
  else if (nm == 3) launch_mode<CB, 3>(mode, g, e, lds, s);
  else launch_mode<CB, 5>(mode, g, e, lds, s);
  return true;
}

}  // namespace

bool launch_dw_mfma(int mode, const DwLayer &L, const EpiArgs &e, int cus, hipStream_t s)
{
  return (L.Ho * L.Wo <= 64 && launch_cb<64>(mode, L, e, cus, s)) || launch_cb<16>(mode, L, e, cus, s);
}
