// Host side of conv_rows.h: launch (addresses: conv_rows_geom.h).
#include "conv_rows.h"

#include "host.h"

bool launch_conv_rows(int mode, const ConvLayer &L, const EpiArgs &e, int cus, hipStream_t s)
{
  const long long M = (long long)L.B * L.Ho * L.Wo;
  // 16-channel groups per wave: all of them up to four, fewer while that leaves SIMDs without a wave
  int nt = L.N <= 16 ? 1 : L.N <= 32 ? 2 : 4;
  while (nt > 1 && (M + 63) / 64 * ((L.N + 16 * nt - 1) / (16 * nt)) < 4ll * cus) nt /= 2;
  RowsGeom g;
  if (mode == EPI_OUT32 || !rows_shape(L.in, L.w, L.bias, L.out, M, L.N, L.H, L.W, L.Ci, L.Ho, L.Wo, L.kx, L.ky, L.pt, L.pl, L.sx, L.sy, cus, nt, &g)) return false;
  const dim3 grid((unsigned)((g.groups + 4 * g.npass - 1) / (4 * g.npass)), (unsigned)((L.N + 16 * nt - 1) / (16 * nt))), block(256);
  const int place = L.Wo % 64 == 0 && rows_chunks(g) <= 32 ? ROWS_ROW64 : L.Wo % 16 == 0 ? ROWS_ROW16 : ROWS_ANY;
#define ROWS_NT(NT)                                                                                                               \
  if (place == ROWS_ROW64) hipLaunchKernelGGL((conv_rows_kernel<NT, ROWS_ROW64>), grid, block, 0, s, g, e, mode);                 \
  else if (place == ROWS_ROW16) hipLaunchKernelGGL((conv_rows_kernel<NT, ROWS_ROW16>), grid, block, 0, s, g, e, mode);            \
  else hipLaunchKernelGGL((conv_rows_kernel<NT, ROWS_ANY>), grid, block, 0, s, g, e, mode);
  if (nt == 1) { ROWS_NT(1) }
  else if (nt == 2) { ROWS_NT(2) }
  else { ROWS_NT(4) }
#undef ROWS_NT
  return true;
}
