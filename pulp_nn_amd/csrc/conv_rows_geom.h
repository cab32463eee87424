// Addresses of conv_rows_kernel (conv_rows.h).  Plain C++: the kernel uses them, and a host program can walk the same numbers.
#pragma once
#include <stdint.h>

#include <algorithm>

#include "fastdiv.h"

// Units of 16 consecutive output pixels.  A filter row of a pixel is L = kx * Ci contiguous bytes of the input.
struct RowsGeom {
  const uint8_t *in;
  const int8_t *w;
  const int8_t *bias;   // may be null
  uint8_t *out;
  int M, N, K, L;       // output pixels, channels, bytes of a filter and of one of its rows
  int H, W, Ci, Ho, Wo, kx, ky, pt, pl, sx, sy;
  int total;            // bytes of input
  bool gather;          // a wave has whole pixels, not in whole pieces: worth putting together in LDS before they are stored
  int groups, npass;    // groups of 64 pixels; how many a wave takes, 4 apart
  FastDiv d_wo, d_ho;
};

// The window of a pixel: the offset of its first byte (which may lie outside the input), its first row and column.
struct RowsWindow {
  int at, iy, ix;
};
PULPNN_HD RowsWindow rows_window(const RowsGeom &g, unsigned m)
{
  const unsigned r = fastdiv(m, g.d_wo), b = fastdiv(r, g.d_ho);
  const int ox = (int)(m - r * g.Wo), oy = (int)(r - b * g.Ho);
  RowsWindow w;
  w.iy = oy * g.sy - g.pt;
  w.ix = ox * g.sx - g.pl;
  w.at = (((int)b * g.H + w.iy) * g.W + w.ix) * g.Ci;
  return w;
}
// The 16 bytes that are fetched for a filter row that starts at offset `at`: from the dword below it, inside the input; the row starts
// rows_shift bytes behind.  A row longer than 13 bytes that does not start on a dword needs the dword behind them too.
PULPNN_HD int rows_fetch(const RowsGeom &g, int at)
{
  const int most = (g.total - 16) & ~3;
  return at < 0 ? 0 : at < most ? at & ~3 : most;
}
PULPNN_HD int rows_more(const RowsGeom &g, int at)
{
  const int most = (g.total - 4) & ~3;
  return at < 0 ? 0 : (at & ~3) + 16 < most ? (at & ~3) + 16 : most;
}
PULPNN_HD bool rows_long(const RowsGeom &g) { return g.L > 13 && g.Ci % 4 != 0; }
// ... and near the ends of the tensor, where those would not hold the whole row: 16 bytes at any address, moved by at - rows_exact.
PULPNN_HD int rows_exact(const RowsGeom &g, int at) { return at < 0 ? 0 : at < g.total - 16 ? at : g.total - 16; }
// (Wide enough for all of the fetches here: a row from offset 16 on and up to 40 bytes before the end lies in 16-byte pieces that were not
// clamped.)
PULPNN_HD bool rows_near_end(const RowsGeom &g, int at) { return at < 16 || at > g.total - 40; }
// A unit of 16 pixels of one output row (Wo % 16 == 0), w: the first one's window.  Pixel l16's filter row fy starts rows_lane bytes further.
PULPNN_HD int rows_lane(const RowsGeom &g, int l16, int fy) { return (fy * g.W + l16 * g.sx) * g.Ci; }
// Whether some of a unit's rows do not lie inside the image as a whole, or near the ends of the tensor.
PULPNN_HD bool rows_edge(const RowsGeom &g, const RowsWindow &w)
{
  return w.iy < 0 || w.iy + g.ky > g.H || w.ix < 0 || w.ix + 15 * g.sx + g.kx > g.W || rows_near_end(g, w.at) || rows_near_end(g, w.at + rows_lane(g, 15, g.ky - 1));
}
// A group of 64 pixels of one output row (Wo % 64 == 0) whose input rows go through LDS: filter row fy is fetched from the dword below its first
// byte on, rows_chunks(g) times 16 bytes of it, ROWS_PITCH bytes apart in LDS (so that the four filter rows that a wave's lanes read start in
// different banks).  Row fy of the group's window starts at offset `at`.
#define ROWS_PITCH 608
PULPNN_HD int rows_span(const RowsGeom &g) { return 63 * g.sx * g.Ci + 16 + 3; }  // (as far as any lane reads)
PULPNN_HD int rows_chunks(const RowsGeom &g) { return (rows_span(g) + 15) / 16; }
PULPNN_HD int rows_chunk_at(const RowsGeom &g, int at, int chunk)
{
  const int a = (at & ~3) + 16 * chunk, most = (g.total - 16) & ~3;
  return a < 0 ? 0 : a < most ? a : most;
}
// What is kept of filter row fy of the pixel whose window is w: bytes [lo, hi), if the row exists.
struct RowsKeep {
  bool row;
  int lo, hi;
};
PULPNN_HD RowsKeep rows_keep(const RowsGeom &g, const RowsWindow &w, int fy)
{
  RowsKeep k;
  k.row = fy < g.ky && (unsigned)(w.iy + fy) < (unsigned)g.H;
  k.lo = (w.ix < 0 ? -w.ix : 0) * g.Ci;
  const int right = g.W - w.ix < g.kx ? g.W - w.ix : g.kx;
  k.hi = (right > 0 ? right : 0) * g.Ci;
  return k;
}

// False for a layer the kernel does not take.
inline bool rows_shape(const uint8_t *in, const int8_t *w, const int8_t *bias, uint8_t *out, long long M, int N, int H, int W, int Ci, int Ho, int Wo, int kx, int ky, int pt,
                       int pl, int sx, int sy, int cus, int nt, RowsGeom *o)
{
  const long long batch = M / ((long long)Ho * Wo), total = batch * H * W * Ci;
  // (32-bit offsets, also of rows and columns in the padding and of pixels past the last one)
  const long long reach = ((long long)(Ho + 1) * sy + ky + pt + H) * W * Ci + ((long long)Wo * sx + kx + pl) * Ci;
  if (kx * Ci > 16 || ky > 4 || ((uintptr_t)in & 3) || total < 32 || (long long)N * kx * ky * Ci < 16 || total + reach >= 0x7fffffffLL || M >= 0x7fffffffLL - 4096) return false;
  RowsGeom &g = *o;
  g = RowsGeom{};
  g.in = in;
  g.w = w;
  g.bias = bias;
  g.out = out;
  g.M = (int)M;
  g.N = N;
  g.L = kx * Ci;
  g.K = g.L * ky;
  g.H = H;
  g.W = W;
  g.Ci = Ci;
  g.Ho = Ho;
  g.Wo = Wo;
  g.kx = kx;
  g.ky = ky;
  g.pt = pt;
  g.pl = pl;
  g.sx = sx;
  g.sy = sy;
  g.total = (int)total;
  g.gather = N <= 16 * nt && N % (4 * nt) != 0;
  g.groups = (int)((M + 63) / 64);
  // groups per wave: as many as leave every SIMD eight waves, at most 8 (the filters are set up once for all of them)
  const long long blocks = (N + 16 * nt - 1) / (16 * nt);
  g.npass = (int)std::max<long long>(1, std::min<long long>(8, g.groups * blocks / (32ll * cus)));
  g.d_wo = fastdiv_make((unsigned)Wo);
  g.d_ho = fastdiv_make((unsigned)Ho);
  return true;
}
