// Host side of conv_band.h: tile shape and launch.
#include "host.h"

#include <algorithm>

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
  if (mode == EPI_OUT32 || (long long)L.N * L.kx * L.ky * L.Ci >= 0x7fffffffLL || (long long)L.kx * L.ky * L.Ci < 16) return false;
  if ((long long)L.B * L.H * L.W * L.Ci < 16 || (long long)L.H * L.W * L.Ci >= (1ll << 40)) return false;
  BandGeom g = {};
  g.in = L.in;
  g.w = L.w;
  g.bias = L.bias;
  g.out = L.out;
  g.N = L.N;
  g.K = L.kx * L.ky * L.Ci;
  g.H = L.H;
  g.W = L.W;
  g.Ci = L.Ci;
  g.Ho = L.Ho;
  g.Wo = L.Wo;
  g.kx = L.kx;
  g.ky = L.ky;
  g.pt = L.pt;
  g.pl = L.pl;
  g.sx = L.sx;
  g.sy = L.sy;
  g.mode = mode;
  int B = L.B;
  if (L.kx == 1 && L.ky == 1 && L.sx == 1 && L.sy == 1 && !L.pt && !L.pl && L.Ho == L.H && L.Wo == L.W) {
    // pointwise: the batch is one row of pixels
    const long long m = (long long)B * L.H * L.W;
    if (m > 0x7fffffffLL) return false;
    g.H = g.Ho = B = 1;
    g.W = g.Wo = (int)m;
  }
  g.CG = (L.Ci + 15) / 16;
  g.CP = 16 * (g.CG | 1);  // an odd number of chunks: neighbouring pixels start in different banks
  g.NK = (L.kx * L.ky * g.CG + 3) / 4;
  // waves along the channels, 16-channel groups per wave
  g.WN = L.N <= 16 ? 1 : L.N <= 32 ? 2 : 4;
  int tn = L.N <= 64 ? 1 : L.N <= 128 ? 2 : 4;
  const int wm = 4 / g.WN;
  auto lds_for = [&](int r, int pc) {
    g.R = r;
    g.PC = pc;
    g.IW = (pc - 1) * L.sx + L.kx;
    g.NR = (r - 1) * L.sy + L.ky;
    g.tab_off = g.NR * g.IW * g.CP;
    g.c_off = g.tab_off + 16 * g.NK;
    return (long long)g.c_off + 16ll * tn * g.WN * (4 + 2 * (int)sizeof(bn_t));
  };
  // the largest run of pixels whose input fits; fewer while that leaves compute units idle
  int tm = 0, r = 1, pc = 1;
  const int tries[] = {8, 4, 2};
  for (const int t : tries) {
    const int px = 16 * t * wm;
    pc = std::min(px, g.Wo);
    r = std::max(1, std::min(px / pc, g.Ho));
    if (pc < g.Wo) r = 1;
    while (r > 1 && lds_for(r, pc) > 64 * 1024) r--;
    const long long lds = lds_for(r, pc);
    const long long wgs = (long long)B * ((g.Ho + r - 1) / r) * ((g.Wo + pc - 1) / pc) * ((g.N + 16 * tn * g.WN - 1) / (16 * tn * g.WN));
    tm = t;
    if (lds <= (t == 2 ? 150 : 64) * 1024 && (wgs >= 2ll * cus || t == 2)) break;
  }
  g.xtiles = (g.Wo + pc - 1) / pc;
  // a row split evenly, rows spread evenly over the bands
  if (g.xtiles > 1) pc = (g.Wo + g.xtiles - 1) / g.xtiles;
  g.bands = (g.Ho + r - 1) / r;
  r = (g.Ho + g.bands - 1) / g.bands;
  const long long lds = lds_for(r, pc);
  if (lds > 150 * 1024) return false;
  g.nblocks = (g.N + 16 * tn * g.WN - 1) / (16 * tn * g.WN);
  const long long total = (long long)B * g.bands * g.xtiles * g.nblocks;
  if (total > 0x7fffffffLL) return false;
  g.total = (int)total;
  g.d_nb = fastdiv_make((unsigned)g.nblocks);
  g.d_xt = fastdiv_make((unsigned)g.xtiles);
  g.d_band = fastdiv_make((unsigned)g.bands);
  g.d_cg = fastdiv_make((unsigned)g.CG);
  g.d_iw = fastdiv_make((unsigned)g.IW);
  g.d_pc = fastdiv_make((unsigned)g.PC);
  g.d_kx = fastdiv_make((unsigned)g.kx);
  if (tn == 1) return launch_tm<1>(tm, g, e, (size_t)lds, s);
  if (tn == 2) return launch_tm<2>(tm, g, e, (size_t)lds, s);
  return launch_tm<4>(tm, g, e, (size_t)lds, s);
}
