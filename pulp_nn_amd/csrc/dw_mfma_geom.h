// Tile shape of dw_mfma_kernel and the arithmetic that says which bytes a tile reads and writes.  Plain C++: the kernel
// and its launcher use it, and a host program can walk the same numbers.
#pragma once
#include <stdint.h>

#include <algorithm>

#include "fastdiv.h"

// LDS bytes of a filter row: 8 zeros and its up to 8 bytes; of one wave's filter rows: those of a quarter of the channels, and 8 zeros.
enum { DWM_WROW = 16 };
PULPNN_HD int dwm_wpart(int channels, int ky) { return channels / 4 * ky * DWM_WROW + 16; }

struct DwLayer {
  const uint8_t *in;
  const int8_t *wt;
  const int8_t *bias;
  uint8_t *out;
  int B, CH, H, W, Ho, Wo, kx, ky, pt, pl, sx, sy;
};

struct DwmGeom {
  const uint8_t *in;
  const int8_t *wt;
  const int8_t *bias;  // may be null
  uint8_t *out;
  int B, CH, H, W, Ho, Wo;
  int kx, ky, pt, pl, sx, sy;
  long long in_bytes;   // bytes of the whole input tensor
  long long edge_bytes; // a tile whose last plane ends behind this byte may load behind the tensor
  int wt_bytes;         // bytes of all filters
  int ND, rND;          // dwords of an input row behind 16 output columns; 65536 / ND + 1
  int RB, NR;           // output rows per tile, input rows behind them
  int XT;               // groups of 16 output columns per tile
  int pitch, CS;        // LDS bytes per staged row and per channel
  int Q;                // 16-byte chunks staged per row
  int w_off, o_off;     // LDS offsets: filter rows (DWM_WROW bytes each), output tile
  int nper, cpar;       // staging: slots (row, chunk) a pass covers, channels side by side
  // tile index -> (channels, columns, rows, image); thread -> channel; slot -> row; unit -> row; pixel -> row (of a tile
  // of full width)
  FastDiv d_cb, d_xt, d_band, d_nper, d_q, d_xg, d_wt;
  int cblocks, xtiles, bands, total;  // (one aligned scalar load: what a workgroup asks for first)
  FastDiv d_wt_last;  // pixel -> row of the last tile along a row
};

// One tile: CB channels from c0 on (ncb of them exist), output rows oy0 .. oy0 + rows - 1 of image b, output columns
// 16 * xg0 .. 16 * xg0 + wt - 1.
struct DwmTile {
  int c0, ncb, xt, xg0, oy0, rows, wt;
  unsigned b;
};
template <int CB>
PULPNN_HD DwmTile dwm_tile(const DwmGeom &g, unsigned id)
{
  // channels vary fastest: the pieces of a pixel's line that different workgroups write meet in one L2
  const unsigned t1 = fastdiv(id, g.d_cb), t2 = fastdiv(t1, g.d_xt), b = fastdiv(t2, g.d_band);
  DwmTile t;
  t.b = b;
  t.c0 = (int)(id - t1 * g.cblocks) * CB;
  t.xt = (int)(t1 - t2 * g.xtiles);
  t.xg0 = t.xt * g.XT;
  t.oy0 = (int)(t2 - b * g.bands) * g.RB;
  t.ncb = CB < g.CH - t.c0 ? CB : g.CH - t.c0;
  t.rows = g.RB < g.Ho - t.oy0 ? g.RB : g.Ho - t.oy0;
  t.wt = 16 * g.XT < g.Wo - 16 * t.xg0 ? 16 * g.XT : g.Wo - 16 * t.xg0;
  return t;
}

// Whether a layer of this tile shape, with 64 channels a workgroup, takes that rather than 16.
// A workgroup's set-up is most of its work on planes of up to 64 output pixels, and with 64 channels it is paid once instead of four times, as long as
// enough workgroups remain and LDS holds whole planes: cut in bands, the planes' rows are staged again and the set-up is paid again.  Whole calls, 16 /
// 64 channels: 7x7x512 batch 256 28.1 / 19.7 us, 5x5x512 26.9 / 17.9, 4x4x130 batch 700 21.4 / 16.8, 5x5 filters on 7x7x256 20.9 / 17.9; in bands stride 2 on
// 13x13x256 22.0 / 25.6, 7x7 filters on 7x7x256 25.0 / 34.2.
inline bool dwm_wide(const DwLayer &L, const DwmGeom &g64, int cus)
{
  return L.Ho * L.Wo <= 64 && (long long)L.B * ((L.CH + 63) / 64) >= 4ll * cus && g64.bands == 1;
}

// Whether a 16-byte load of the tile may leave the tensor (before: bytes of the tensor in front of the tile's first plane).
PULPNN_HD bool dwm_edge(const DwmGeom &g, const DwmTile &t, long long before)
{
  return before < g.pl || before + t.ncb * (g.H * g.W) > g.edge_bytes;
}

// Bytes from the tile's first plane to the load of chunk column x in row iy of channel c (a row outside the image: the
// start of the plane, masked off).
PULPNN_HD int dwm_load_base(const DwmGeom &g, int iy, int x) { return (unsigned)iy < (unsigned)g.H ? iy * g.W + x : 0; }

// 16-byte loads that a thread has in flight.  (Eight with 64 channels a workgroup: 50 registers more, three waves a SIMD and, from two MFMAs a
// unit on, two.  Eight / four: 7x7x512 batch 256 24.0 / 19.7 us, 64 bits 28.0 / 24.0, 5x5x512 22.8 / 17.6; 5x5 filters on 7x7x256 20.6 / 17.9.)
enum { DWM_LOADS = 4 };

// First channel of the thread whose first one is cpi: out of reach of every channel where its pass has no slot for it.
PULPNN_HD int dwm_thread_channel(int cb, int cpi, bool slot) { return slot ? cpi : cb + 64; }

// Lane's offset of a buffer load of a tile that is no edge, from 64 bytes in front of the tile's first plane, where a row's left padding may
// begin: chunk `at` of the c-th channel behind the thread's first one, or of the last channel that exists.  The lane's offset says it
// all and none of it is left to the scalar one, which is not documented to take part in the range check: asked for with the scalar one, the
// channels past a short last block lay up to 80 KB behind the tensor.  A thread without a slot is out of range.
// (One addition and one minimum a load.  Out of range by a comparison with the channel, 2 % slower over 114 layers.)
PULPNN_HD unsigned dwm_buffer_first(int plane, int ch, int cpi, int at) { return ch == cpi ? (unsigned)(64 + cpi * plane + at) : 0xf0000000u; }
PULPNN_HD unsigned dwm_buffer_last(int plane, int ncb, int ch, int cpi, int at) { return ch == cpi ? (unsigned)(64 + (ncb - 1) * plane + at) : 0xf0000000u; }
PULPNN_HD unsigned dwm_buffer_off(unsigned first, unsigned last, int plane, int c)
{
  const unsigned at = first + (unsigned)(c * plane);
  return at < last ? at : last;
}

// First byte of row t of the filters of channel c0 + cw and those behind it; rows of channels that do not exist: the last one.
PULPNN_HD int dwm_filter_at(const DwmGeom &g, const DwmTile &t, int cw, int row)
{
  const int at = (t.c0 + cw) * g.ky + row, last = (t.c0 + t.ncb) * g.ky - 1;
  return (at < last ? at : last) * g.kx;
}

// Row of the tile's pixel p, counted row by row.
PULPNN_HD int dwm_out_row(const DwmGeom &g, const DwmTile &t, int p)
{
  if (g.xtiles == 1) return 0;  // (one column tile: a single run of pixels)
  return (int)fastdiv((unsigned)p, t.xt + 1 == g.xtiles ? g.d_wt_last : g.d_wt);
}

// Tile shape for CB channels per workgroup.  nm: MFMAs per (channel, 16 units);
// lds: dynamic LDS of the launch.  False for a layer the kernel does not take.
template <int CB>
bool dwm_shape(const DwLayer &L, int cus, DwmGeom *out, int *nm_out, size_t *lds_out)
{
  const long long plane = (long long)L.H * L.W;
  if (L.kx > 8 || L.kx * L.ky > 256 || L.sx > 4 || L.pl > 64 || plane * CB > (1 << 29) || (long long)L.B * L.CH * plane < 16) return false;
  DwmGeom &g = *out;
  g = DwmGeom{};
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
  g.in_bytes = (long long)L.B * L.CH * plane;
  g.wt_bytes = L.CH * L.kx * L.ky;
  g.ND = (15 * L.sx + L.kx + 3) / 4;
  g.rND = 65536 / g.ND + 1;
  const int nm = (L.ky * g.ND + 15) / 16;
  if (nm > 5) return false;
  g.cblocks = (L.CH + CB - 1) / CB;
  const int xg = (L.Wo + 15) / 16;
  const int fixed = 4 * dwm_wpart(CB, L.ky);
  // LDS of a tile, in 64 bits: a tall output at a large row stride would reach over more input rows than an int counts
  // (the fields are what they should be for tiles that fit)
  auto shape = [&](int xt, int rb) -> long long {
    const long long nr = (rb - 1) * (long long)L.sy + L.ky;
    g.XT = xt;
    g.RB = rb;
    g.NR = (int)nr;
    g.Q = ((xt - 1) * 16 * L.sx + 4 * g.ND + 15) / 16;
    g.pitch = 16 * (g.Q | 1);  // an odd number of 16-byte chunks: the rows of a tile start in different banks
    g.CS = (int)(nr * g.pitch);
    g.xtiles = (xg + xt - 1) / xt;
    g.bands = (L.Ho + rb - 1) / rb;
    return CB * nr * g.pitch + fixed + (long long)rb * std::min(16 * xt, L.Wo) * (CB + 4);
  };
  // Rows of the full width, all rows of the plane, unless that takes more than 32 KB of LDS (four workgroups of a
  // compute unit cover each other's load, multiply and store phases) ...
  constexpr int LDS = CB == 16 ? 32 * 1024 : 48 * 1024;
  int xt = xg, rb = std::min(L.Ho, LDS / (CB + 4));
  while (xt > 1 && shape(xt, 1) > LDS) xt = (xt + 1) / 2;
  if (shape(xt, 1) > 64 * 1024) return false;
  while (rb > 1 && shape(xt, rb) > LDS) rb--;
  // ... and fewer rows while that leaves compute units without a workgroup and a tile still fills an MFMA
  auto count = [&] { return (long long)L.B * g.cblocks * ((xg + xt - 1) / xt) * ((L.Ho + rb - 1) / rb); };
  while (rb * xt > 16 && rb > 1 && count() < 2ll * cus) rb = (rb + 1) / 2;
  rb = (L.Ho + (L.Ho + rb - 1) / rb - 1) / ((L.Ho + rb - 1) / rb);  // rows spread evenly over the bands
  const long long lds_bytes = shape(xt, rb);
  const long long total = (long long)L.B * g.cblocks * g.xtiles * g.bands;
  if (total > 0x7fffffffLL) return false;
  g.total = (int)total;
  g.w_off = CB * g.CS;
  g.o_off = g.w_off + fixed;
  // The last chunk of a row may reach over the end of its plane, by less than `over`.  Where a row outside the image, which loads
  // from the start of its plane, may do so too (planes of fewer than 16 bytes), and where the channels of a pass are too far apart
  // for 32-bit offsets, every tile counts as one that may leave the tensor: each of its loads is held inside.
  const long long over = std::max(0ll, 16ll * g.XT * g.sx * (g.xtiles - 1) - g.pl + 16ll * g.Q - g.W);
  g.edge_bytes = plane < 16 || plane * CB > (1 << 27) ? -(1ll << 62) : g.in_bytes - over;
  g.d_cb = fastdiv_make((unsigned)g.cblocks);
  g.d_xt = fastdiv_make((unsigned)g.xtiles);
  g.d_band = fastdiv_make((unsigned)g.bands);
  g.nper = std::min(g.NR * g.Q, 256);
  g.cpar = std::min(256 / g.nper, CB);
  g.d_nper = fastdiv_make((unsigned)g.nper);
  g.d_q = fastdiv_make((unsigned)g.Q);
  g.d_xg = fastdiv_make((unsigned)g.XT);
  g.d_wt = fastdiv_make((unsigned)std::min(16 * xt, L.Wo));
  g.d_wt_last = fastdiv_make((unsigned)(L.Wo - 16 * xt * (g.xtiles - 1)));
  *nm_out = nm;
  *lds_out = (size_t)lds_bytes + 32;
  return true;
}
