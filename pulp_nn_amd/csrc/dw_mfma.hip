// Host side of dw_mfma.h: tile shape and launch.
#include "dw_mfma.h"

#include <algorithm>

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
  const long long plane = (long long)L.H * L.W;
  if (L.kx > 8 || L.kx * L.ky > 256 || L.sx > 4 || L.pl > 64 || plane * CB > (1 << 29) || (long long)L.B * L.CH * plane < 16) return false;
  DwmGeom g = {};
  g.in = L.in;
  g.wt = L.wt;
  g.bias = L.bias;
  g.out = L.out;
  g.B = L.B;
  g.CH = L.CH;
  g.H = L.H;
  g.W = L.W;
  g.Ho = L.Ho;
  g.Wo = L.Wo;
  g.kx = L.kx;
  g.ky = L.ky;
  g.pt = L.pt;
  g.pl = L.pl;
  g.sx = L.sx;
  g.sy = L.sy;
  g.in_bytes = L.B * L.CH * plane;
  g.wt_bytes = L.CH * L.kx * L.ky;
  g.ND = (15 * L.sx + L.kx + 3) / 4;
  g.rND = 65536 / g.ND + 1;
  const int nm = (L.ky * g.ND + 15) / 16;
  if (nm > 5) return false;
  g.cblocks = (L.CH + CB - 1) / CB;
  const int xg = (L.Wo + 15) / 16;
  const int fixed = CB * L.ky * 8 + CB * (4 + 2 * (int)sizeof(bn_t));
  auto shape = [&](int xt, int rb) {
    g.XT = xt;
    g.RB = rb;
    g.NR = (rb - 1) * L.sy + L.ky;
    g.Q = ((xt - 1) * 16 * L.sx + 4 * g.ND + 15) / 16;
    g.pitch = 16 * (g.Q | 1);  // an odd number of 16-byte chunks: the rows of a tile start in different banks
    g.CS = g.NR * g.pitch;
    g.xtiles = (xg + xt - 1) / xt;
    g.bands = (L.Ho + rb - 1) / rb;
    return CB * g.CS + fixed + rb * std::min(16 * xt, L.Wo) * (CB + 4);
  };
  // Rows of the full width, all rows of the plane, unless that takes more than 32 KB of LDS (four workgroups of a
  // compute unit cover each other's load, multiply and store phases) ...
  constexpr int LDS = CB == 16 ? 32 * 1024 : 48 * 1024;
  int xt = xg, rb = L.Ho;
  while (xt > 1 && shape(xt, 1) > LDS) xt = (xt + 1) / 2;
  if (shape(xt, 1) > 64 * 1024) return false;
  while (rb > 1 && shape(xt, rb) > LDS) rb--;
  // ... and fewer rows while that leaves compute units without a workgroup and a tile still fills an MFMA
  auto count = [&] { return (long long)L.B * g.cblocks * ((xg + xt - 1) / xt) * ((L.Ho + rb - 1) / rb); };
  while (rb * xt > 16 && rb > 1 && count() < 2ll * cus) rb = (rb + 1) / 2;
  rb = (L.Ho + (L.Ho + rb - 1) / rb - 1) / ((L.Ho + rb - 1) / rb);  // rows spread evenly over the bands
  const int lds_bytes = shape(xt, rb);
  const long long total = (long long)L.B * g.cblocks * g.xtiles * g.bands;
  if (total > 0x7fffffffLL) return false;
  g.total = (int)total;
  g.w_off = CB * g.CS;
  g.c_off = g.w_off + CB * L.ky * 8;
  g.o_off = (g.c_off + CB * (4 + 2 * (int)sizeof(bn_t)) + 15) & ~15;
  g.d_cb = fastdiv_make((unsigned)g.cblocks);
  g.d_xt = fastdiv_make((unsigned)g.xtiles);
  g.d_band = fastdiv_make((unsigned)g.bands);
  g.nper = std::min(g.NR * g.Q, 256);
  g.cpar = 256 / g.nper;
  g.d_nper = fastdiv_make((unsigned)g.nper);
  g.d_ky = fastdiv_make((unsigned)L.ky);
  g.d_q = fastdiv_make((unsigned)g.Q);
  g.d_xg = fastdiv_make((unsigned)g.XT);
  g.d_wt = fastdiv_make((unsigned)std::min(16 * xt, L.Wo));
  const size_t lds = (size_t)lds_bytes + 32;
  if (nm == 1) launch_mode<CB, 1>(mode, g, e, lds, s);
  else if (nm == 2) launch_mode<CB, 2>(mode, g, e, lds, s);
  else if (nm == 3) launch_mode<CB, 3>(mode, g, e, lds, s);
  else launch_mode<CB, 5>(mode, g, e, lds, s);
  return true;
}

}  // namespace

bool launch_dw_mfma(int mode, const DwLayer &L, const EpiArgs &e, int cus, hipStream_t s)
{
  // 64 channels per workgroup instead of 16 where a plane is so small (up to 64 output pixels) that the set-up of a
  // workgroup, some 400 instructions per wave, is most of its work, and enough workgroups remain.  Measured, kernel time
  // at 16 / 64 channels: 7x7x512 batch 256 33.8 / 23.8 us, 8x8x256 18.9 / 14.5; but 17x17x408 batch 85 18.8 / 27.9,
  // 28x28x256 batch 64 11.8 / 17.9 (fewer workgroups to cover each other's load, multiply and store phases).
  if (L.Ho * L.Wo <= 64 && (long long)L.B * ((L.CH + 63) / 64) >= 4ll * cus && launch_cb<64>(mode, L, e, cus, s)) return true;
  return launch_cb<16>(mode, L, e, cus, s);
}
