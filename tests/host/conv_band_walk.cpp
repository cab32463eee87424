// Walks the tiles of conv_band_kernel on the host with the launcher's own tile shape (csrc/conv_band_geom.h) and reports
// tiles whose staged input, tap table, constants, weights or fragments leave their LDS range, output pixels that no tile or more than one
// computes, and, for the first, the last and some tiles between of layers that are not large, chunks of the band that a workgroup stages twice or
// not at all and loads inside the image that leave the input.
// Layers on stdin, one a line: B H W Ci Ho Wo N kx ky pt pl sx sy bn_bytes cus.  One line out per layer: "ok LDS TILES", with "odd" behind it where
// band_for_odd_channels (up to 64 output channels: band_for_up_to_64) says so, "no"
// (not taken by the kernel) or what is wrong.
#include <stdio.h>

#include <string>
#include <vector>

#include "../../pulp_nn_amd/csrc/conv_band_geom.h"

// One tile's staging, thread by thread as the kernel does it.
static std::string staging(const BandGeom &g, unsigned id)
{
  typedef long long ll;
  const unsigned t1 = fastdiv(id, g.d_nb), t2 = fastdiv(t1, g.d_xt), b = fastdiv(t2, g.d_band);
  const int ox0 = (int)(t1 - t2 * g.xtiles) * g.PC, oy0 = (int)(t2 - b * g.bands) * g.R;
  const int pc = std::min(g.PC, g.Wo - ox0), rows = std::min(g.R, g.Ho - oy0);
  if (pc <= 0 || rows <= 0) return "empty tile";
  // (strides far larger than the image: products past an int are negative ones, outside the image like what they stand for)
  const int iy0 = (int)((unsigned)oy0 * g.sy - g.pt), ix0 = (int)((unsigned)ox0 * g.sx - g.pl), nr = (rows - 1) * g.sy + g.ky;
  const ll first = (ll)b * g.H * g.W * g.Ci + ((ll)iy0 * g.W + ix0) * g.Ci - 16, range = std::min(g.in_bytes - first, 0x7fffffffll);
  const bool near = g.Ci < 16 && first < 0;
  const int lo = (int)std::min(std::max(-first, 0ll), 0x7fffffffll), passes = (int)fastdiv((unsigned)(nr * g.IW - 1), g.d_ppp) + 1;
  std::vector<unsigned char> seen((size_t)nr * g.IW * g.CG);
  for (int cb = 0; cb < g.CG; cb += g.cpp)
    for (int tid = 0; tid < 256; tid++) {
      const int p0 = (int)fastdiv((unsigned)tid, g.d_cpp), c16 = cb + tid - p0 * g.cpp;
      int row = (int)fastdiv((unsigned)p0, g.d_iw), col = p0 - row * g.IW;
      if (p0 >= g.ppp || c16 >= g.CG) row = 1 << 20;
      for (int pass = 0; pass < passes; pass++) {
        if (row < nr) {
          const bool in = (unsigned)(iy0 + row) < (unsigned)g.H && (unsigned)(ix0 + col) < (unsigned)g.W;
          const ll want = ((ll)row * g.W + col) * g.Ci + std::min(16 * c16, g.Ci - 16) + 16, off = near ? std::max(want, (ll)lo) : want;
          if (in && (want > 0x7fffffff || off < 0 || off + 16 > range || first + off < 0 || first + off + 16 > g.in_bytes || off - want > 15))
            return "load of row " + std::to_string(row) + " column " + std::to_string(col) + " at " + std::to_string(first + off);
          const ll dst = ((ll)row * g.IW + col) * g.CP + 16 * c16;
          if (col >= g.IW || dst + 16 > g.tab_off) return "staged outside the input's LDS";
          if (seen[((size_t)row * g.IW + col) * g.CG + c16]++) return "chunk staged twice";
        }
        col += g.scol;
        row += g.srow;
        if (col >= g.IW) col -= g.IW, row++;
      }
    }
  for (const unsigned char s : seen)
    if (!s) return "chunk not staged";
  return "";
}

static std::string check(const ConvLayer &L, int bn_bytes, int cus)
{
  BandGeom g;
  int tn, tm, pf;
  size_t lds;
  if (!band_shape(L, cus, bn_bytes, &g, &tn, &tm, &lds, &pf)) return "no";
  typedef long long ll;
  const ll iw = (g.PC - 1) * (ll)g.sx + g.kx, nr = (g.R - 1) * (ll)g.sy + g.ky, nch = 16ll * tn * g.WN;
  const ll staged = nr * iw * g.CP;
  // (the table has an entry for every chunk of whole groups of pf steps; two groups of weights for each of four waves)
  if (g.IW != iw || staged > g.tab_off || g.tab_off + 16ll * ((g.NK + pf - 1) / pf * pf) > g.c_off || g.c_off + nch * (4 + 2 * bn_bytes) > g.w_off ||
      g.w_off + 4ll * band_wbytes(tn, pf) > (ll)lds || lds > 160 * 1024 - 512)
    return "LDS ranges: " + std::to_string(staged) + " bytes staged, " + std::to_string(lds) + " asked for";
  // the farthest fragment: last pixel of a tile at the last tap, last chunk
  const ll far = ((g.R - 1) * (ll)g.sy * iw + (g.PC - 1) * (ll)g.sx) * g.CP + ((g.ky - 1) * iw + g.kx - 1) * g.CP + 16ll * (g.CG - 1);
  if (far + 16 > staged) return "fragment outside the staged input";
  if (g.R > 1 && g.PC < g.Wo) return "several part rows in a tile";
  if ((ll)g.R * g.PC > 16ll * tm * (4 / g.WN)) return "more pixels than the waves compute";
  if (tm != 2 && tm != 4 && (tm != 8 || tn == 4)) return "no kernel for so many groups of pixels";
  const bool flat = g.Ho != L.Ho || g.Wo != L.Wo;  // a pointwise layer as one row of pixels
  const ll B = flat ? 1 : L.B;
  if (flat && (ll)g.Ho * g.Wo != (ll)L.B * L.Ho * L.Wo) return "pixels of the flattened batch";
  if ((ll)g.xtiles * g.PC < g.Wo || (ll)(g.xtiles - 1) * g.PC >= g.Wo || (ll)g.bands * g.R < g.Ho || (ll)(g.bands - 1) * g.R >= g.Ho ||
      g.nblocks * nch < g.N || (g.nblocks - 1) * nch >= g.N || B * g.bands * g.xtiles * g.nblocks != g.total)
    return "tiles: " + std::to_string(g.total);
  if (nr * iw * g.CG <= 30000 && (ll)g.IW * 256 < 0x7fffffff)
    for (const int id : {0, g.total / 3, g.total / 2, g.total - 1}) {
      const std::string s = staging(g, (unsigned)id);
      if (!s.empty()) return "tile " + std::to_string(id) + ": " + s;
    }
  return "ok " + std::to_string(lds) + " " + std::to_string(g.total) + ((L.N > 64 ? band_for_odd_channels(L, cus, bn_bytes) : band_for_up_to_64(L, cus, bn_bytes)) ? " odd" : "");
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
