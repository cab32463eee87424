// Tile shape of dwpw_kernel (dwpw.h) and the arithmetic that says which bytes a thread reads and writes.  Plain C++: the kernel and
// its launcher use it, and a host program can walk the same numbers.
#pragma once
#include <stdint.h>

#include <algorithm>

#include "fastdiv.h"

// A tile: TR output rows of one image, or NI whole images (planes of at most 64 output pixels, and chains).  Its input rows lie in
// LDS with the padding around them; the depthwise output of its pixels is the activation operand of the pointwise layer, in 64-byte
// slices of K (rows of C bytes for C < 64).
struct DwPwTile {
  int B, C, H, Ho, Co;
  int whole, NI, TR;     // whole images, how many; output rows of a tile
  int lpxb;              // log2 of the tile's blocks of 64 pixels
  int R, nrb, nst;       // depthwise stage: rows of a strip, row blocks of a tile, strips (16 columns, or fewer of several row blocks)
  int CS, slabs;         // channels whose input is in LDS at a time
  int XR, pitch;         // rows of input in LDS, bytes per pixel (an odd number of 16-byte chunks)
  int x_off, lds;        // LDS: where the input starts, bytes in all
  int waves, tiles, lsplit, cf_per;  // 2^lsplit workgroups share a tile, with cf_per 16-channel groups of output each
  int par_off, w_off, kp;            // LDS: the depthwise layer's parameters; the weights, kp slices of K for every wave that multiplies (a chain: every wave)
  int bands;             // tiles per image (1: whole images)
  FastDiv d_n, d_hp, d_ho, d_bands;  // divisions by CS / 16, by H + 2, Ho and bands
};

struct DwPwPlace {
  int b0, oy0;   // first image, first output row in it
  int live;      // output pixels the tile really has
};
template <int WO>
PULPNN_HD DwPwPlace dwpw_place(const DwPwTile &g, unsigned tile)
{
  const unsigned t = fastdiv(tile, g.d_bands);
  DwPwPlace p;
  p.b0 = (int)t * g.NI;
  p.oy0 = (int)(tile - t * g.bands) * g.TR;
  const int images = g.NI < g.B - p.b0 ? g.NI : g.B - p.b0, rows = g.TR < g.Ho - p.oy0 ? g.TR : g.Ho - p.oy0;
  p.live = (g.whole ? images * g.Ho : rows) * WO;
  return p;
}

// The first input row that belongs to the tile, in rows of the whole batch (one above the image where the padding is).
template <int S>
PULPNN_HD long long dwpw_first_row(const DwPwTile &g, const DwPwPlace &p) { return (long long)p.b0 * g.H + (g.whole ? 0 : p.oy0 * S - 1); }
// Rows from there on that a tile may fetch.
PULPNN_HD int dwpw_rows_in(const DwPwTile &g) { return g.whole ? g.NI * g.H : g.XR; }
// 16-byte chunk t of the tile's input with its padding: its place in LDS behind x_off, and its offset from the first row (channel 0 of
// the slab); -1: padding
struct DwPwChunk {
  int lds, off;
};
template <int W, int S>
PULPNN_HD DwPwChunk dwpw_chunk(const DwPwTile &g, const DwPwPlace &p, int t)
{
  const int px = (int)fastdiv((unsigned)t, g.d_n), chunk = t - px * (g.CS / 16);
  const int row = px / (W + 2), col = px - row * (W + 2) - 1;
  const int img = g.whole ? (int)fastdiv((unsigned)row, g.d_hp) : 0;
  const int y = g.whole ? row - img * (g.H + 2) - 1 : p.oy0 * S - 1 + row;   // row of the image
  const bool in = (unsigned)y < (unsigned)g.H && (unsigned)col < (unsigned)W && row < g.XR && p.b0 + img < g.B;
  DwPwChunk c;
  c.lds = px * g.pitch + 16 * chunk;
  c.off = in ? ((g.whole ? img * g.H + y : row) * W + col) * g.C + 16 * chunk : -1;
  return c;
}
template <int W>
PULPNN_HD int dwpw_chunks(const DwPwTile &g) { return g.XR * (W + 2) * (g.CS / 16); }

// One lane of strip st: pixel (of the tile) of its first output row, and the place in LDS of filter column kx of that row's first
// input row (channel 0).  live: the lane has a row block.
struct DwPwLane {
  int px, x;
  bool live;
};
template <int W, int S>
PULPNN_HD DwPwLane dwpw_lane(const DwPwTile &g, int st, int l16, int kx)
{
  constexpr int WO = W / S, XS = WO >= 16 ? WO / 16 : 1, RS = WO >= 16 ? 1 : 16 / WO;  // strips along a row, row blocks of a strip
  const int rb = st / XS * RS + (RS == 1 ? 0 : l16 / WO), ox = RS == 1 ? st % XS * 16 + l16 : l16 % WO;
  DwPwLane n;
  n.live = RS == 1 || rb < g.nrb;
  const int row = (n.live ? rb : g.nrb - 1) * g.R;
  const int img = g.whole ? (int)fastdiv((unsigned)row, g.d_ho) : 0;
  n.px = row * WO + ox;
  n.x = ((img * (g.H + 2) + (row - img * g.Ho) * S) * (W + 2) + ox * S + kx) * g.pitch;
  return n;
}

// Activation operand: 16 channels from c on (a multiple of 16) of pixel px.
PULPNN_HD int dwpw_act(const DwPwTile &g, int px, int c)
{
  return g.C < 64 ? px * g.C + c : (((c >> 6) << g.lpxb) << 12) + px * 64 + ((((c >> 4) & 3) ^ ((px >> 1) & 3)) << 4);
}

// Chains: pixel px's place as an input pixel of the next block (whole images, stride 1).
template <int W>
PULPNN_HD int dwpw_next_x(const DwPwTile &g, int px)
{
  const int row = px / W, img = (int)fastdiv((unsigned)row, g.d_ho);
  return ((row + 2 * img + 1) * (W + 2) + px % W + 1) * g.pitch;
}

// One layer's parameters in LDS, for C channels: bias, k, lambda, and with a filter its 9 bytes a channel, each as in memory from a
// multiple of 1 KB on.
struct DwPwPar {
  int k, l, f, bytes;
};
PULPNN_HD DwPwPar dwpw_par(int C, int bn_bytes, bool filter)
{
  DwPwPar p;
  p.k = (C + 1023) & ~1023;
  p.l = p.k + ((C * bn_bytes + 1023) & ~1023);
  p.f = p.l + ((C * bn_bytes + 1023) & ~1023);
  p.bytes = p.f + (filter ? (9 * C + 1023) & ~1023 : 0);
  return p;
}

// What one instruction of 16 bytes a lane fetches of them, to place `to` (a multiple of 1 KB): array (0 bias, 1 k, 2 lambda, 3 filter), first byte in
// it, and bytes from there on that exist: lanes past them are out of range and get zeros.  (By the lane's own offset: what the scalar offset of a
// load adds does not count where the range is checked.)
struct DwPwParPiece {
  int array, first, bytes;
};
PULPNN_HD DwPwParPiece dwpw_par_piece(const DwPwPar &at, int C, int bn_bytes, bool bias, bool bn, int to)
{
  DwPwParPiece p;
  p.array = to < at.k ? 0 : to < at.l ? 1 : to < at.f ? 2 : 3;
  p.first = to - (p.array == 0 ? 0 : p.array == 1 ? at.k : p.array == 2 ? at.l : at.f);
  const int all = p.array == 0 ? (bias ? C : 0) : p.array == 3 ? 9 * C : bn ? C * bn_bytes : 0;
  p.bytes = all > p.first ? all - p.first : 0;
  return p;
}

// The pointwise layer's weights on their way to LDS: 16 rows (channels out) of 64 bytes, slice kt of K; four lanes fetch the 64 contiguous bytes of a
// row.  Offset of the lane's 16 bytes and what the scalar offset adds; bytes and slices that do not exist are out of range by the lane's own offset.
#define DWPW_OOB 0x80000000u
struct DwPwWeight {
  unsigned off;
  int add;
};
// (narrow: C may be less than 64)
PULPNN_HD unsigned dwpw_w_lane(int C, int cf, int lane, bool narrow)
{
  // (which of the four fetches which 16 bytes depends on the row, as in the activation operand)
  const int row = lane >> 2, chunk = (lane & 3) ^ ((row >> 1) & 3);
  return !narrow || 16 * chunk < C ? (unsigned)((16 * cf + row) * C + 16 * chunk) : DWPW_OOB;
}
PULPNN_HD DwPwWeight dwpw_w_slice(int C, unsigned lane_off, int kt)
{
  const bool ok = 64 * kt < C;
  return DwPwWeight{ok ? lane_off : DWPW_OOB, ok ? 64 * kt : 0};
}

// The shapes that pulp_nn_hip_dw_pw_hwc and pulp_nn_hip_dw_pw_chain_hwc (n_blocks > 1) take, by the limits that their declarations state:
// the rows a wave takes at once, 1024 output channels per workgroup, whole images and 64 KB of LDS for a chain.  (dwpw_kernel alone could
// do more; what a caller may rely on is what the declarations say.)  The reason of a refusal, or null.
inline const char *dwpw_refusal(long long B, int C, int W, int Ho, int Wo, int Co, int S, unsigned n_blocks, int cus, int bn_bytes)
{
  static const char *const other = "no fused kernel for this geometry: call the depthwise and the pointwise layer separately";
  int R = 0, waves = 4;
  if (W == 64) R = 2;
  else if (W == 32) R = 4;
  else if (W == 16 || W == 8) {
    R = S == 1 ? 4 : 2;
    waves = 8;
  } else if (W == 4 && S == 1) {
    R = 4;
    waves = 8;
  }
  const bool c_ok = C == 16 || C == 32 || (C % 64 == 0 && C <= 1024);
  const long long M = B * Ho * Wo;
  if (!R || !c_ok) return other;
  const int LG = C >= 64 ? 1 : 64 / C, CGN = C >= 64 ? C / 64 : 1;
  if (Ho % (R * LG) || Co % 16 || M > 0x7fffffffLL || (long long)Co * C >= 0x7fffffffLL) return other;
  const int item = R * LG * Wo;  // pixels of one wave's rows
  auto lds_bytes = [&](int px, int ch) { return (long long)px * C + (long long)ch * (4 + 2 * bn_bytes); };
  int segs = (waves + CGN - 1) / CGN;
  while ((segs * item) % 32) segs++;
  while (segs > 1 && (segs * item * C > 49152 || (M + (long long)segs * item - 1) / (segs * item) < cus)) segs--;
  while ((segs * item) % 32) segs++;
  int px = segs * item, split = 1;
  const long long tiles = (M + px - 1) / px;
  const int groups = (Co + 63) / 64;
  while (tiles * split < cus && split * 2 <= groups) split *= 2;
  const int per = (groups + split - 1) / split * 64;
  if (per > 1024) return "more than 1024 output channels per workgroup: call the depthwise and the pointwise layer separately";
  long long lds = lds_bytes(px, per);
  if (n_blocks > 1) {
    const int img = Ho * Wo;
    int images = (px + img - 1) / img;
    while ((images * img) % 32 || (images * img) % item) images++;
    px = images * img;
    lds = lds_bytes(px, groups * 64) + (long long)px * (Co + 64);
    if (S != 1 || C != Co || B % images != 0)
      return "blocks can only be chained at stride 1 with as many channels out as in, on whole images per tile";
  }
  if (lds > 65536) return other;
  if (n_blocks > 1 && W == 64) return "blocks of this width cannot be chained";
  return nullptr;
}

// Waves of a workgroup for a tile of px pixels: a wave's item is 16 channels of 16 or more pixels.  Measured, call by call at batch 256 with 4 /
// 8 / 16 waves: 64x64x16 in tiles of 256 pixels 31.2 / 39.3 / 68.1 us, 32x32x64 27.4 / 21.9 / 27.9, 16x16x128 22.0 / 14.8 / 12.8, 8x8x256 whole 13.6 /
// 9.9 / 9.0; batch 8, tiles of 64 pixels, 16x16x128 6.8 / 5.7 / 6.3.
inline int dwpw_waves(int C, bool whole, int px) { return C == 16 ? 4 : C <= 64 || (!whole && px * C <= 8192) ? 8 : 16; }

// Tile of NI whole images (whole) or of px output pixels, at most `waves` waves per workgroup, at least `least` slabs of input.  False if it
// does not fit.
inline bool dwpw_tile(DwPwTile &g, int W, int S, bool chain, int cus, int bn_bytes, int NI, int px, int waves, int least)
{
  const int WO = W / S, CF = g.Co / 16, C = g.C;
  g.NI = NI;
  g.TR = g.whole ? NI * g.Ho : std::min(std::max(1, px / WO), g.Ho);
  g.bands = g.whole ? 1 : (g.Ho + g.TR - 1) / g.TR;
  for (g.lpxb = 0; (64 << g.lpxb) < g.TR * WO;) g.lpxb++;
  g.x_off = (64 << g.lpxb) * C;
  // all channels' input at once if that is no more than 56 KB, else equal slabs of them
  long long x = 0;
  for (int parts = 1; parts <= std::max(1, C / 64); parts++) {
    if (parts > 1 && (chain || C / 64 % parts || (parts < least && parts < C / 64))) continue;
    if (least > 1 && parts == 1) continue;
    g.CS = C / parts;
    g.slabs = parts;
    g.pitch = 16 * ((g.CS / 16) | 1);
    g.XR = g.whole ? g.NI * (g.H + 2) : (g.TR - 1) * S + 3;
    x = (long long)(g.XR + 1) * (W + 2) * g.pitch;  // (a walk reads one row past the last one it needs)
    if (x <= 56 * 1024) break;
  }
  const long long tiles = (long long)((g.B + g.NI - 1) / g.NI) * g.bands;
  if (g.x_off + x > 160 * 1024 || tiles > 0x7fffffff / 64) return false;
  g.tiles = (int)tiles;
  // (a tile is shared only as long as that gives no compute unit a second workgroup: each of them computes the depthwise stage)
  for (g.lsplit = 0; !chain && ((long long)g.tiles << (g.lsplit + 1)) <= cus && (2 << g.lsplit) <= CF / 4;) g.lsplit++;
  g.cf_per = (CF + (1 << g.lsplit) - 1) >> g.lsplit;
  // depthwise stage: rows per strip, as many as leave every wave a strip
  const int cgs = g.CS / 16;
  auto strips = [&](int r) { return WO >= 16 ? g.TR / r * (WO / 16) : (g.TR / r + 16 / WO - 1) / (16 / WO); };
  const int want = std::min(waves, dwpw_waves(C, g.whole, g.TR * WO));
  for (g.R = 4; g.R > 1 && (g.TR % g.R || g.Ho % g.R || strips(g.R) * cgs < want);) g.R /= 2;
  g.nrb = g.TR / g.R;
  g.nst = strips(g.R);
  const int most = std::max(g.nst * cgs, g.cf_per << g.lpxb);
  for (g.waves = 4; g.waves < most && g.waves < want;) g.waves *= 2;
  // LDS: activation operand, input, depthwise parameters, weights (all of K at once for up to eight slices, if that fits)
  g.par_off = (int)((g.x_off + x + 1023) & ~1023);
  g.w_off = g.par_off + dwpw_par(C, bn_bytes, true).bytes;
  const int busy = chain ? g.waves : std::min(g.waves, g.cf_per << g.lpxb);
  g.kp = C <= 64 ? 1 : C <= 256 || g.w_off + busy * 8 * 1024 > 150 * 1024 ? 4 : 8;
  g.lds = g.w_off + busy * g.kp * 1024;
  return g.lds <= 160 * 1024;
}

// W = 4 .. 64, a power of two; C = 16, 32 or a multiple of 64; Co a multiple of 16.  chain: whole images and all channels per workgroup.
// Takes everything that dwpw_refusal lets pass.
inline bool dwpw_shape(int B, int C, int H, int W, int Ho, int Co, int S, bool chain, int cus, int bn_bytes, DwPwTile *out)
{
  DwPwTile &g = *out;
  g = DwPwTile{};
  g.B = B;
  g.C = C;
  g.H = H;
  g.Ho = Ho;
  g.Co = Co;
  const int WO = W / S;
  g.whole = chain || Ho * WO <= 64;
  bool ok = false;
  // (more slabs than the input alone asks for only where nothing fits beside it: two output rows of 1024 channels)
  for (int least = 1; least <= std::max(1, chain ? 1 : C / 64) && !ok; least *= 2)
  for (int waves = 16; waves >= 4 && !ok; waves /= 2) {
    if (g.whole) {
      // images until the tile has 64 pixels, as long as their input fits without being cut into slabs
      for (int ni = std::min(B, std::max(1, 64 / (Ho * WO))); ni >= 1 && !ok; ni /= 2)
        ok = dwpw_tile(g, W, S, chain, cus, bn_bytes, ni, 0, waves, least) && (g.slabs == 1 || ni == 1);
    } else {
      // 256, 128 or 64 pixels: the most that leave every compute unit sixteen waves
      int px = 256;
      while (px > 64 && (px < WO || (long long)B * ((Ho + px / WO - 1) / (px / WO)) * dwpw_waves(C, false, px) < 16ll * cus)) px /= 2;
      for (; px >= 64 && !ok; px /= 2) ok = dwpw_tile(g, W, S, chain, cus, bn_bytes, 1, px, waves, least);
    }
  }
  if (!ok) return false;
  g.d_n = fastdiv_make((unsigned)g.CS / 16);
  g.d_hp = fastdiv_make((unsigned)H + 2);
  g.d_ho = fastdiv_make((unsigned)Ho);
  g.d_bands = fastdiv_make((unsigned)g.bands);
  return true;
}
