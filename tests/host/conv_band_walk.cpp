// Walks the tiles of conv_band_kernel on the host with the launcher's own tile shape (csrc/conv_band_geom.h) and reports
// tiles whose staged input or fragments leave their LDS range, and output pixels that no tile or more than one computes.
// Layers on stdin, one a line: B H W Ci Ho Wo N kx ky pt pl sx sy bn_bytes cus.  One line out per layer: "ok LDS TILES", with "odd" behind it where
// band_for_odd_channels says so, "no"
// (not taken by the kernel) or what is wrong.
#include <stdio.h>

#include <string>

#include "../../pulp_nn_amd/csrc/conv_band_geom.h"

static std::string check(const ConvLayer &L, int bn_bytes, int cus)
{
  BandGeom g;
  int tn, tm;
  size_t lds;
  if (!band_shape(L, cus, bn_bytes, &g, &tn, &tm, &lds)) return "no";
  typedef long long ll;
  const ll iw = (g.PC - 1) * (ll)g.sx + g.kx, nr = (g.R - 1) * (ll)g.sy + g.ky, nch = 16ll * tn * g.WN;
  const ll staged = nr * iw * g.CP;
  if (g.IW != iw || staged > g.tab_off || g.tab_off + 16ll * g.NK > g.c_off || g.c_off + nch * (4 + 2 * bn_bytes) > (ll)lds || lds > 160 * 1024 - 512)
    return "LDS ranges: " + std::to_string(staged) + " bytes staged, " + std::to_string(lds) + " asked for";
  // the farthest fragment: last pixel of a tile at the last tap, last chunk
  const ll far = ((g.R - 1) * (ll)g.sy * iw + (g.PC - 1) * (ll)g.sx) * g.CP + ((g.ky - 1) * iw + g.kx - 1) * g.CP + 16ll * (g.CG - 1);
  if (far + 16 > staged) return "fragment outside the staged input";
  if (g.R > 1 && g.PC < g.Wo) return "several part rows in a tile";
  if ((ll)g.R * g.PC > 16ll * tm * (4 / g.WN)) return "more pixels than the waves compute";
  const bool flat = g.Ho != L.Ho || g.Wo != L.Wo;  // a pointwise layer as one row of pixels
  const ll B = flat ? 1 : L.B;
  if (flat && (ll)g.Ho * g.Wo != (ll)L.B * L.Ho * L.Wo) return "pixels of the flattened batch";
  if ((ll)g.xtiles * g.PC < g.Wo || (ll)(g.xtiles - 1) * g.PC >= g.Wo || (ll)g.bands * g.R < g.Ho || (ll)(g.bands - 1) * g.R >= g.Ho ||
      g.nblocks * nch < g.N || (g.nblocks - 1) * nch >= g.N || B * g.bands * g.xtiles * g.nblocks != g.total)
    return "tiles: " + std::to_string(g.total);
  return "ok " + std::to_string(lds) + " " + std::to_string(g.total) + (L.N > 64 && band_for_odd_channels(L, cus, bn_bytes) ? " odd" : "");
}

int main()
{
  ConvLayer L = {};
  int bn_bytes, cus;
  while (scanf("%d %d %d %d %d %d %d %d %d %d %d %d %d %d %d", &L.B, &L.H, &L.W, &L.Ci, &L.Ho, &L.Wo, &L.N, &L.kx, &L.ky, &L.pt, &L.pl, &L.sx,
               &L.sy, &bn_bytes, &cus) == 15)
    puts(check(L, bn_bytes, cus).c_str());
  return 0;
}
