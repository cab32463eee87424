// Host side of dw_hwc.h: launch (the split of the work: dw_hwc_geom.h).
#include "dw_hwc.h"

#include "host.h"

namespace {

template <int W, int S>
bool launch(int mode, const DwLayer &L, const EpiArgs &e, int cus, hipStream_t s)
{
  DwhGeom g;
  if (!dwh_shape<W, S>(L, cus, &g)) return false;
  hipLaunchKernelGGL((dw_hwc_kernel<W, S>), dim3((unsigned)((g.total + 3) / 4)), dim3(256), 0, s, g, e, mode);
  return true;
}

}  // namespace

bool launch_dw_hwc(int mode, const DwLayer &L, const EpiArgs &e, int cus, hipStream_t s)
{
  if (!aligned(L.in, 16) || !aligned(L.out, 16) || dwh_wide(L)) return false;
  if (L.sx == 1) return launch<64, 1>(mode, L, e, cus, s) || launch<32, 1>(mode, L, e, cus, s) || launch<16, 1>(mode, L, e, cus, s);
  return launch<64, 2>(mode, L, e, cus, s) || launch<32, 2>(mode, L, e, cus, s);
}
