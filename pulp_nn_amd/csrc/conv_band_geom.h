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
  int tab_off, c_off, w_off;  // LDS offsets: tap table, per-channel constants, weights of the four waves
  int nblocks, xtiles, bands, total;
  int cpp, ppp, srow, scol;   // staging: chunks of a pixel side by side, pixels of a pass, and those as rows and columns of the band
  int wtap, wc;               // four chunks further: taps and chunks
  long long in_bytes;
  FastDiv d_nb, d_xt, d_band, d_cg, d_iw, d_pc, d_kx, d_cpp, d_ppp;
};

// K steps whose weights a wave asks for together (two such groups are in LDS), by its 16-channel and 16-pixel groups.  With one 16-channel
// group and two of pixels: four or one, see there.
PULPNN_HD constexpr int band_pf(int tn, int tm) { return tn == 1 ? 2 : tn == 2 ? (tm == 8 ? 1 : 2) : 1; }
PULPNN_HD constexpr int band_wbytes(int tn, int pf) { return 2 * pf * tn * 1024; }

// Tile shape; bn_bytes: bytes of a batch-norm parameter.  tn, tm: 16-channel and 16-pixel groups per wave; lds: dynamic LDS
// of the launch.  False for a layer the kernel does not take.
inline bool band_shape(const ConvLayer &L, int cus, int bn_bytes, BandGeom *out, int *tn_out, int *tm_out, size_t *lds_out, int *pf_out = nullptr)
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
  auto lds_for = [&](int r, int pc, int t) -> long long {
    const long long iw = (pc - 1) * (long long)L.sx + L.kx, nr = (r - 1) * (long long)L.sy + L.ky;
    const long long tab = nr * iw * g.CP, c = tab + 16ll * ((g.NK + 3) & ~3);  // (whole groups of steps)
    const long long w = (c + 16ll * tn * g.WN * (4 + 2 * bn_bytes) + 1023) & ~1023ll;
    g.R = r;
    g.PC = pc;
    g.IW = (int)iw;
    g.NR = (int)nr;
    g.tab_off = (int)tab;
    g.c_off = (int)c;
    g.w_off = (int)w;
    // (offsets inside a tile's input have to fit an int as well)
    return (nr - 1) * L.W * L.Ci + iw * L.Ci < 0x7ffffff0ll ? w + 4ll * band_wbytes(tn, band_pf(tn, t)) : 1ll << 40;
  };
  constexpr int MOST = 160 * 1024 - 512;
  // The run of pixels of a workgroup: the one with which the busiest compute unit has least to do, a workgroup's set-up counting as
  // three 16-pixel groups of 16 channels a wave, two of 32, one of 64.  (64 channels a wave take 500 registers with eight groups: one wave per SIMD, so up to four there.)
  int tm = 0, r = 1, pc = 1;
  long long least = 0;
  for (int t = tn == 4 ? 4 : 8; t >= 2; t /= 2) {
    const int px = 16 * t * wm;
    int tpc = std::min(px, g.Wo), tr = tpc < g.Wo ? 1 : std::max(1, std::min(px / tpc, g.Ho));
    while (tr > 1 && lds_for(tr, tpc, t) > 80 * 1024) tr--;
    while (t == 2 && tpc > 1 && lds_for(tr, tpc, t) > MOST) tpc = (tpc + 1) / 2;
    if (t > 2 && lds_for(tr, tpc, t) > 80 * 1024) continue;
    auto count = [&](int n) { return (long long)B * ((g.Ho + tr - 1) / tr) * ((g.Wo + n - 1) / n) * ((g.N + 16 * tn * g.WN - 1) / (16 * tn * g.WN)); };
    // A row of which LDS holds one workgroup, however few weights are in flight, in halves where the busiest compute unit then has less than a whole
    // one's rounds to do (whole rows / halves, 64 bits: 28x13x53 256 -> 32 5x5 43.6 / 31.7 us, 109x15x51 256 -> 32 5x5 stride 2 86.3 / 78.5; where the rounds
    // come out even halves lose: 125x8x57 224 -> 48 5x5 stride 2 40.5 / 48.2).
    const int half = (tpc + 1) / 2;
    if (tn == 1 && t == 2 && tr == 1 && count(tpc) > cus && lds_for(tr, tpc, t) - 4 * band_wbytes(1, 1) > MOST / 2 && lds_for(tr, half, t) <= MOST / 2 &&
        (count(half) + cus - 1) / cus < 2 * ((count(tpc) + cus - 1) / cus))
      tpc = half;
    const long long wgs = count(tpc);
    if (t > 2 && wgs < cus) continue;
    const long long work = (wgs + cus - 1) / cus * ((tn == 4 ? 1 : 4 - tn) + (tr * tpc + 16 * wm - 1) / (16 * wm));
    if (tm && work >= least) continue;
    least = work;
    tm = t;
    r = tr;
    pc = tpc;
  }
  g.xtiles = (g.Wo + pc - 1) / pc;
  // a row split evenly, rows spread evenly over the bands
  if (g.xtiles > 1) pc = (int)(((long long)g.Wo + g.xtiles - 1) / g.xtiles);
  g.bands = (g.Ho + r - 1) / r;
  r = (g.Ho + g.bands - 1) / g.bands;
  // (no more pixels a wave than the tile has: all waves take part where LDS holds few rows)
  while (tm > 2 && r * pc <= 16 * (tm / 2) * wm && lds_for(r, pc, tm / 2) <= MOST) tm /= 2;
  long long lds = lds_for(r, pc, tm);
  if (lds > MOST) return false;
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
  g.cpp = std::min(g.CG, 256);
  g.ppp = 256 / g.cpp;
  g.srow = g.ppp / g.IW;
  g.scol = g.ppp % g.IW;
  g.wtap = 4 / g.CG;
  g.wc = 4 % g.CG;
  g.in_bytes = (long long)L.B * L.H * L.W * L.Ci;
  g.d_cpp = fastdiv_make((unsigned)g.cpp);
  g.d_ppp = fastdiv_make((unsigned)g.ppp);
  *tn_out = tn;
  *tm_out = tm;
  // Groups of weights: four steps for long filters in launches of few workgroups, which wait for their weights; one where that lets another
  // workgroup share a compute unit (call times, two / four steps: 8x38x9 240 -> 32 stride 2 11.4 / 11.0; 57x43 24 -> 40 stride 2 batch 32
  // 8.0 / 8.5, 19x33 85 -> 8 batch 123 11.1 / 13.7; two / one: 27x39 pointwise 320 -> 8 batch 215 25.7 / 20.7; in
  // no more than two workgroups a compute unit 16x55x64 178 -> 64 5x5 stride 2 38.7 / 24.2, 12x41x28 250 -> 32 7x7 81.8 / 50.6, 73x14x54 224 -> 32 5x5 stride 2
  // 39.8 / 26.9).  (Without weights in LDS there was room for a second one in some where now there is none: 125x8x57 224 -> 48 5x5 stride 2 23.7 / 40.5,
  // 109x15x51 256 -> 32 59.9 / 78.3.)
  int pf = band_pf(tn, tm);
  if (tn == 1 && tm == 2) {
    const auto with = [&](int n) { return lds + 4 * (band_wbytes(1, n) - band_wbytes(1, pf)); };
    const int to = g.NK > 8 && total <= 2ll * cus && with(4) <= (total <= cus ? MOST : 80 * 1024) ? 4
                   : total > MOST / with(2) * cus && MOST / with(1) > MOST / with(2) && MOST / with(2) < 3 ? 1
                                                                                                   : 2;
    lds = with(to);
    pf = to;
  }
  if (pf_out) *pf_out = pf;
  *lds_out = (size_t)lds;
  return true;
}

// Whether a layer of 33 to 64 output channels on a channel count of whole 16-byte chunks but no multiple of 64 takes this kernel, not the tiled one: it
// does, over 60 layers in 0.73 of the time, but for
// - eight groups of pixels a wave, of which a compute unit holds two workgroups and gets more (tiled / band: 144x41x32 144 -> 48 stride 2 18.7 / 26.3 us,
//   183x36x44 160 -> 39 28.1 / 38.2, 81x15x60 224 -> 41 31.8 / 31.6; four or two groups, or room for a third, are mixed: 94x48x39 144 -> 63 23.0 / 20.9);
// - halves of rows, with larger filters, in more than four workgroups a compute unit (144x12x61 224 -> 48 5x5 stride 2 51.2 / 70.6; 48x11x50 224 -> 40 7x7
//   stride 2 86.1 / 63.8).
inline bool band_for_up_to_64(const ConvLayer &L, int cus, int bn_bytes)
{
  BandGeom g;
  int tn, tm;
  size_t lds;
  if (!band_shape(L, cus, bn_bytes, &g, &tn, &tm, &lds)) return false;
  if (L.kx * L.ky <= 9) return L.kx * L.ky == 1 || !(tm == 8 && lds > 53 * 1024 && g.total > 2 * cus);
  return !(g.xtiles > 1 && 2 * g.R * g.PC <= 16 * tm * (4 / g.WN) && g.total > 4 * cus);
}

// Whether a layer of 65 to 128 output channels on a channel count of whole 16-byte chunks but no multiple of 64 takes this kernel, not the tiled one, which
// gathers such inputs chunk by chunk in tiles of 128 pixels x 64 channels.  Whole calls, tiled / band: 12x12 112 -> 71 batch 146 16.5 / 10.3 us, 27x8
// 176 -> 120 batch 177 19.7 / 11.7, 48x18 96 -> 100 stride 2 batch 101 9.7 / 6.2.  Not
// - up to five K slices, which the tiled kernel fetches at once (2x2 on 41x54 48 -> 72 batch 9 5.8 / 7.0);
// - where LDS holds one workgroup (20x53 176 -> 112 stride 2 batch 119 19.9 / 36.5), or from stride 2 on, where a pixel's input is four pixels, in more than
//   two a compute unit or in tiles of eight groups of pixels or a third empty (24x48 176 -> 96 stride 2 batch 182 26.3 / 36.9);
// - where the tiled kernel's tiles are one for almost every compute unit, which is what it does best, and these are more (63x21 96 -> 96 stride 2 batch 39
//   8.7 / 10.5, 10x17 96 -> 120 batch 92 8.8 / 10.3);
// - where two workgroups of eight groups of pixels, which is what a compute unit holds, are not all it gets (16x28 176 -> 128 batch 133 24.7 / 32.6, 33x15
//   48 -> 128 batch 119 9.3 / 14.2);
// - on more than some 60000 pixels in all (42x31 48 -> 96 batch 54 14.4 / 18.3), nor, with large filters, on more than 96 channels.
// Over 300 layers drawn for it the mean is 0.857 of the tiled kernel's time; of the 231 that it takes fourteen are more than 3 % slower, the worst 18x51 112 -> 80
// batch 34 13.1 / 16.2, 48x34 208 -> 128 batch 13 1.23.
inline bool band_for_odd_channels(const ConvLayer &L, int cus, int bn_bytes)
{
  const long long m = (long long)L.B * L.Ho * L.Wo, tiled = (m + 127) / 128 * ((L.N + 63) / 64);
  const int taps = L.kx * L.ky;
  if (L.N > 128 || L.Ci % 64 == 0 || taps == 1 || (taps > 9 && L.Ci > 96) || taps * L.Ci <= 320 || m > 60000) return false;
  BandGeom g;
  int tn, tm;
  size_t lds;
  if (!band_shape(L, cus, bn_bytes, &g, &tn, &tm, &lds) || lds > 80 * 1024) return false;
  if (tm > 2 && g.total > cus && tiled <= cus && 5 * tiled >= 4 * cus) return false;
  if (tm == 8 && g.total > 2 * cus) return false;
  if (L.sx == 1 && L.sy == 1) return true;
  return g.total <= 2 * cus && (tm == 2 || (tm == 4 && 10 * g.R * g.PC >= 7 * 16 * tm * (4 / g.WN)));
}
