// Tile shape of conv_band_kernel.  Plain C++: the launcher uses it, and a host program can walk the same numbers.
#pragma once
#include <stdint.h>

#include <algorithm>

#include "fastdiv.h"

struct ConvLayer {
  const uint8_t *in;
  const int8_t *w;
  const int8_t *bias;
  uint8_t *out;
  int B, H, W, Ci, Ho, Wo, N, kx, ky, pt, pl, sx, sy;
};

struct BandGeom {
  const uint8_t *in;
  const int8_t *w;
  const int8_t *bias;  // may be null
  uint8_t *out;
  int N, K, H, W, Ci, Ho, Wo;
  int kx, ky, pt, pl, sx, sy;
  int CG, CP;          // 16-byte chunks per pixel, LDS bytes per pixel
  int NK;              // MFMA steps: ceil(kx * ky * CG / 4)
  int R, PC;           // output rows and columns per workgroup (R == 1 if PC < Wo)
  int IW, NR;          // input columns and rows behind them
  int WN;              // waves along the channels (1, 2 or 4 of four)
  int mode;
  int tab_off, c_off;  // LDS offsets: tap table, per-channel constants
  int nblocks, xtiles, bands, total;
  FastDiv d_nb, d_xt, d_band, d_cg, d_iw, d_pc, d_kx;
};

// Tile shape; bn_bytes: bytes of a batch-norm parameter.  tn, tm: 16-channel and 16-pixel groups per wave; lds: dynamic LDS
// of the launch.  False for a layer the kernel does not take.
inline bool band_shape(const ConvLayer &L, int cus, int bn_bytes, BandGeom *out, int *tn_out, int *tm_out, size_t *lds_out)
{
  if ((long long)L.N * L.kx * L.ky * L.Ci >= 0x7fffffffLL || (long long)L.kx * L.ky * L.Ci < 16) return false;
  if ((long long)L.B * L.H * L.W * L.Ci < 16 || (long long)L.H * L.W * L.Ci >= (1ll << 40)) return false;
  BandGeom &g = *out;
  g = BandGeom{};
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
  int B = L.B;
  if (L.kx == 1 && L.ky == 1 && L.sx == 1 && L.sy == 1 && !L.pt && !L.pl && L.Ho == L.H && L.Wo == L.W) {
    // pointwise: the batch is one row of pixels
    const long long m = (long long)B * L.H * L.W;
    if (m > 0x7fffffffLL - 1024) return false;  // (a tile's pixels are counted past the last one)
    g.H = g.Ho = B = 1;
    g.W = g.Wo = (int)m;
  }
  g.CG = (L.Ci + 15) / 16;
  g.CP = 16 * (g.CG | 1);  // an odd number of chunks: neighbouring pixels start in different banks
  g.NK = (L.kx * L.ky * g.CG + 3) / 4;
  // waves along the channels, 16-channel groups per wave
  g.WN = L.N <= 16 ? 1 : L.N <= 32 ? 2 : 4;
  const int tn = L.N <= 64 ? 1 : L.N <= 128 ? 2 : 4;
  const int wm = 4 / g.WN;
  // LDS of a tile, in 64 bits: strides and filters far larger than the image give more bytes than an int counts (the fields
  // are what they should be for tiles that fit)
  auto lds_for = [&](int r, int pc) -> long long {
    const long long iw = (pc - 1) * (long long)L.sx + L.kx, nr = (r - 1) * (long long)L.sy + L.ky;
    const long long tab = nr * iw * g.CP, c = tab + 16ll * g.NK;
    g.R = r;
    g.PC = pc;
    g.IW = (int)iw;
    g.NR = (int)nr;
    g.tab_off = (int)tab;
    g.c_off = (int)c;
    return c + 16ll * tn * g.WN * (4 + 2 * bn_bytes);
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
  if (g.xtiles > 1) pc = (int)(((long long)g.Wo + g.xtiles - 1) / g.xtiles);
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
  *tn_out = tn;
  *tm_out = tm;
  *lds_out = (size_t)lds;
  return true;
}
