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
  int act_px;            // pixels of the activation operand (a multiple of 16; of 64 in chains and with more than one block)
  int R, nrb, nst;       // depthwise stage: rows of a strip, row blocks of a tile, strips (16 columns, or fewer of several row blocks)
  int CS, slabs;         // channels whose input is in LDS at a time (the last slab may have fewer)
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

// Activation operand: 16 channels from c on (a multiple of 16) of pixel px; narrow: rows of C bytes (C < 64), step: bytes of a 64-byte slice of
// all pixels.  (A macro: as a function it costs dwpw_kernel eight scalar registers in spills, 32x32x64 batch 1 5.28 -> 5.40 us.)
#define DWPW_ACT_AT(narrow, C, step, px, c) ((narrow) ? (px) * (C) + (c) : ((c) >> 6) * (step) + (px) * 64 + (((((c) >> 4) & 3) ^ (((px) >> 1) & 3)) << 4))
PULPNN_HD int dwpw_act(const DwPwTile &g, int px, int c) { return DWPW_ACT_AT(g.C < 64, g.C, 64 * g.act_px, px, c); }

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

// Planes 16 pixels wide at stride 2 with 128 channels or more go to dwpw16_kernel while there is no more than one tile of 64 output pixels for every
// four compute units, with up to 512 channels out for every two.  dwpw_kernel / dwpw16_kernel: 16x16x256 batch 1 7.9 / 7.2 us, batch 32 8.7 / 8.4, batch 128
// 9.7 / 9.1; 16x16x512 batch 64 17.1 / 15.2, batch 128 18.7 / 16.6; 16x16x128 batch 1 6.1 / 5.8, batch 128 7.2 / 6.2.  Past the lines: 16x16x512 -> 1024 batch
// 96 20.9 / 24.4; 16x16x128 batch 160 7.4 / 8.0, batch 256 7.6 / 8.5.
inline bool dwpw_small16(long long B, int C, int W, int Ho, int Co, int S, int cus)
{
  return W == 16 && S == 2 && C >= 128 && B * Ho * 8 <= (Co <= 512 ? 32ll : 16ll) * cus;
}

// Whether four slices of weights take the kernel that asks for the pointwise constants where they are used and has five waves a SIMD, not four: where LDS
// holds a second workgroup of sixteen waves, and so few of them have a part in the pointwise stage that the next one can begin beside them.
// Constants ahead / lean: 16x16x256 -> 64 batch 268 27.1 / 22.8 us, 16x16x192 -> 64 26.9 / 23.1, 16x16x128 -> 32 batch 500 21.5 / 18.9; elsewhere ahead is the better: 8x8x256 -> 512
// stride 2 batch 64 6.7 / 6.8, 16x16x640 -> 1024 stride 2 batch 128 31.9 / 32.9, 8x8x128 -> 256 stride 2 batch 18 4.7 / 4.9.
inline bool dwpw_lean(const DwPwTile &t, int cus)
{
  return t.waves == 16 && t.cf_per << t.lpxb <= 4 && 2 * t.lds <= 160 * 1024 && (long long)t.tiles << t.lsplit > cus;
}

#define DWPW16_PX 32  // output pixels of a tile of it: four rows, two of them one item of the depthwise stage
// Workgroups that share such a tile, each with a part of the output channels: as many as leave every compute unit one, and no workgroup
// more than 1024 channels.  LDS of one of them: the activation operand, and bias, k and lambda of its channels.
inline int dwpw16_split(int tiles, int Co, int cus)
{
  int split = 1;
  for (const int blocks = (Co + 63) / 64; split * 2 <= blocks && (2ll * tiles * split <= cus || blocks > 16 * split);) split *= 2;
  return split;
}
inline int dwpw16_lds(int C, int Co, int split, int bn_bytes) { return DWPW16_PX * C + ((Co + 63) / 64 + split - 1) / split * 64 * (4 + 2 * bn_bytes); }

// Waves of a workgroup for a tile of px pixels: a wave's item is 16 channels of 16 or more pixels.  Measured, call by call at batch 256 with 4 /
// 8 / 16 waves: 64x64x16 in tiles of 256 pixels 31.2 / 39.3 / 68.1 us, 32x32x64 27.4 / 21.9 / 27.9, 16x16x128 22.0 / 14.8 / 12.8, 8x8x256 whole 13.6 /
// 9.9 / 9.0; batch 8, tiles of 64 pixels, 16x16x128 6.8 / 5.7 / 6.3.  8 / 16 waves at batch 64: 8x8x128 5.8 / 6.7, two images of 4x4x128 5.6 / 5.8,
// but one 5.7 / 5.4.
inline int dwpw_waves(int C, int px) { return C == 16 ? 4 : C <= 64 || (C <= 128 && px >= 32 && px <= 64) ? 8 : 16; }

// Tile of NI whole images (whole) or of px output pixels.  0 if it does not fit, 1 with fewer waves than it should have, else 2.
inline int dwpw_tile(DwPwTile &g, int W, int S, bool chain, int cus, int bn_bytes, int NI, int px)
{
  const int WO = W / S, CF = g.Co / 16, C = g.C, units = C < 64 ? 1 : C / 64;
  g.NI = NI;
  g.TR = g.whole ? NI * g.Ho : std::min(std::max(1, px / WO), g.Ho);
  g.bands = g.whole ? 1 : (g.Ho + g.TR - 1) / g.TR;
  for (g.lpxb = 0; (64 << g.lpxb) < g.TR * WO;) g.lpxb++;
  g.act_px = g.lpxb || chain ? 64 << g.lpxb : (g.TR * WO + 15) & ~15;
  g.x_off = g.act_px * C;
  g.XR = g.whole ? g.NI * (g.H + 2) : (g.TR - 1) * S + 3;
  const long long tiles = (long long)((g.B + g.NI - 1) / g.NI) * g.bands;
  if (g.x_off > 160 * 1024 || tiles > 0x7fffffff / 64) return 0;
  g.tiles = (int)tiles;
  // (a tile is shared only as long as that gives no compute unit a second workgroup: each of them computes the depthwise stage)
  for (g.lsplit = 0; !chain && ((long long)g.tiles << (g.lsplit + 1)) <= cus && (2 << g.lsplit) <= CF / 4;) g.lsplit++;
  g.cf_per = (CF + (1 << g.lsplit) - 1) >> g.lsplit;
  const int want = C > 64 && (chain || (g.whole && W == 16 && S == 2)) ? 16 : dwpw_waves(C, g.TR * WO), par = dwpw_par(C, bn_bytes, true).bytes;
  // LDS: activation operand, input, depthwise parameters, weights.  A slab of the input costs a round trip to memory and two barriers, so
  // there are as few as fit (16x16x256 stride 2, batch 16, two slabs / one: 9.5 / 8.3 us; 8x8x512 10.9 / 9.5).  The weights of a wave are all of
  // K at once for up to eight slices, if that fits, else four (in a chain, where sixteen waves leave no room for eight, always).  More than five
  // slabs of 64 channels only if half as many waves, with room for
  // fewer weights, do not get along with fewer of them (16x16x640 stride 2, batch 128, 16 waves and ten slabs / 8 and four: 36.8 / 28.9; but
  // 64x64x320, five slabs / two: 61.4 / 76.2), and 4 waves (16x16x768 stride 2 26.2 us, 8 waves 18.7) only where nothing else fits.
  DwPwTile best = {};
  int with = 0;
  for (int waves = want; waves >= 4 && !(waves == 4 && best.lds); waves /= 2) {
    for (int parts = 1; parts <= (chain ? 1 : units); parts++) {
      DwPwTile t = g;
      t.CS = C < 64 ? C : 64 * ((units + parts - 1) / parts);
      t.slabs = (C + t.CS - 1) / t.CS;
      if (t.slabs != parts) continue;
      t.pitch = 16 * ((t.CS / 16) | 1);
      const long long x = (long long)(t.XR + 1) * (W + 2) * t.pitch;  // (a walk reads one row past the last one it needs)
      if (t.x_off + x > 160 * 1024) continue;
      // depthwise stage: rows per strip, as many as leave every wave a strip; in a chain no wave a second one (dwpw_chain_kernel)
      const int cgs = t.CS / 16;
      auto strips = [&](int r) { return WO >= 16 ? t.TR / r * (WO / 16) : (t.TR / r + 16 / WO - 1) / (16 / WO); };
      for (t.R = 4; t.R > 1 && (t.TR % t.R || t.Ho % t.R || (strips(t.R) * cgs < waves && !(chain && strips(t.R / 2) * cgs > 16)));) t.R /= 2;
      t.nrb = t.TR / t.R;
      t.nst = strips(t.R);
      const int most = std::max(t.nst * cgs, t.cf_per << t.lpxb);
      for (t.waves = 4; t.waves < most && t.waves < waves;) t.waves *= 2;
      t.par_off = (int)((t.x_off + x + 1023) & ~1023);
      t.w_off = t.par_off + par;
      const int busy = chain ? t.waves : std::min(t.waves, t.cf_per << t.lpxb);
      t.kp = C <= 64 ? 1 : chain || C <= 256 || t.w_off + busy * 8 * 1024 > 150 * 1024 ? 4 : 8;
      t.lds = t.w_off + busy * t.kp * 1024;
      if (t.lds > 160 * 1024) continue;
      if (!best.lds || t.slabs < best.slabs) best = t, with = waves;
      break;
    }
    if (best.lds && (best.slabs <= 5 || best.CS >= 128)) break;
  }
  if (!best.lds) return 0;
  g = best;
  return with < want ? 1 : 2;
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
  const int WO = W / S, img = Ho * WO;
  g.whole = chain || img <= 64;
  bool ok = false;
  // whether a tile half as large than g makes a second workgroup per compute unit, where there are that many tiles (64x64x64 -> 64 stride
  // 2 batch 256, 256 / 128 pixels 41.4 / 34.7 us; 16x16x64 stride 2 batch 1024 four / two images 11.7 / 10.1)
  auto two = [&](int px, int ni, int half) {
    DwPwTile t = g;
    return px > 64 && g.lds > 80 * 1024 && 2ll * g.tiles > cus && dwpw_tile(t, W, S, chain, cus, bn_bytes, ni, half) == 2 && t.lds <= 80 * 1024;
  };
  if (chain) {
    // images until the tile has 64 pixels, as long as they fit with all waves
    for (int ni = std::min(B, std::max(1, 64 / img)); ni >= 1 && !ok; ni /= 2) ok = dwpw_tile(g, W, S, chain, cus, bn_bytes, ni, 0) >= (ni == 1 ? 1 : 2);
  } else if (g.whole) {
    // One image, or as many as leave every compute unit one workgroup (two of 8 waves), up to 128 pixels: its set-up is paid once for all of
    // them.  One / two / four images: 4x4x128 batch 256 5.6 / 6.0 / 6.6 us, batch 1024 11.9 / 10.7 / 7.5; 8x8x64 batch 1024 11.1 / 8.6 / 9.2.  Up to 64
    // pixels with fewer workgroups where one small image leaves most of a block of 64 pixels empty, and reads all weights for that: 4x4x384
    // batch 256 11.3 / 9.7 / 9.3, 4x4x512 -> 1024 batch 128 13.1 / 11.1 / 10.6.  Not where that takes more than 64 KB of input or cuts it in slabs,
    // unless there is more than one round of workgroups (8x8x512 stride 2, two images in two slabs / one in one: batch 128 12.4 / 11.3, batch 512
    // 16.4 / 26.4; four in eight 28.0).
    const int one = img > 16 && C <= 128 ? 2 * cus : cus, few = img > 16 || C < 256 ? one : C < 320 ? cus / 4 : cus / 16;
    auto groups = [&](int ni) { return (B + ni - 1) / ni; };
    int ni = 1;
    while (groups(ni) > (ni * img < 64 ? few : one) && 2 * ni * img <= 128) ni *= 2;
    for (; ni >= 1 && !ok; ni /= 2) {
      const int fits = dwpw_tile(g, W, S, chain, cus, bn_bytes, ni, 0);
      if (ni == 1) ok = fits != 0;
      else if (fits != 2 || two(ni * img, ni / 2, 0)) ok = false;
      else if (ni * img <= 32 ? groups(ni / 2) >= cus : groups(ni / 2) > cus) ok = g.slabs <= (ni * img <= 32 ? 6 : 2);
      else ok = g.slabs == 1 && g.par_off - g.x_off <= 64 * 1024;
    }
  } else {
    // 64 pixels, 128 where that leaves every compute unit a workgroup, 256 where it leaves it sixteen waves
    auto tiles = [&](int px) { return (long long)B * ((Ho + px / WO - 1) / (px / WO)); };
    int px = 256;
    while (px > 64 && (px < WO || tiles(px) < cus || (px == 256 && tiles(px) * dwpw_waves(C, px) < 16ll * cus))) px /= 2;
    // ... but not 256 where the waves would then fetch weights again more than twice (64x64x128 -> 256 batch 64, 256 / 128 pixels 87.3 / 72.6 us)
    if (px == 256 && C > 64 && 4 * (Co / 16) > 3 * dwpw_waves(C, px)) px = 128;
    for (; px >= 64 && !ok; px /= 2) {
      const int fits = dwpw_tile(g, W, S, chain, cus, bn_bytes, 1, px);
      // (with all its waves, and few slabs, while half a tile has four rows: of three rows of input one belongs to a row of output alone)
      ok = px / 2 < std::max(64, WO) ? fits != 0 : (px / 2 < 4 * WO ? fits != 0 : fits == 2 && g.slabs <= 2) && !two(px, 1, px / 2);
    }
  }
  if (!ok) return false;
  g.d_n = fastdiv_make((unsigned)g.CS / 16);
  g.d_hp = fastdiv_make((unsigned)H + 2);
  g.d_ho = fastdiv_make((unsigned)Ho);
  g.d_bands = fastdiv_make((unsigned)g.bands);
  return true;
}
