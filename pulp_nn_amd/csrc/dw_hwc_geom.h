// Work split of the HWC depthwise kernel on the matrix cores (dw_hwc.h) and the arithmetic that says which bytes a lane
// reads and writes.  Plain C++: the kernel and its launcher use it, and a host program can walk the same numbers.
#pragma once
#include <stdint.h>

#include "dw_mfma_geom.h"
#include "fastdiv.h"

// One wave: R output rows of full width of one image times 16 * NT channels, where an input row of them is 64 chunks of 16
// bytes, one per lane (64 pixels of 16 channels, 32 of 32, 16 of 64).
struct DwhGeom {
  const uint8_t *in;
  const int8_t *wt;
  const int8_t *bias;  // may be null
  uint8_t *out;
  int C, H, Ho;
  int R;               // output rows per wave
  int cblocks, bands, total;
  unsigned lead, size, out_size;  // the input buffer starts `lead` bytes in front of the input, so that offsets are not negative
  FastDiv d_cb, d_band;
};

#define DWH_OOB 0x80000000u  // an offset past the end of either buffer, whatever is added for rows and chunks

struct DwhItem {
  int c0, oy0, rows;  // first channel, first output row, output rows there are
  unsigned b;
};
template <int NT>
PULPNN_HD DwhItem dwh_item(const DwhGeom &g, unsigned id)
{
  // channels vary fastest: the pieces of a pixel's line that different waves read and write meet in one cache
  const unsigned t1 = fastdiv(id, g.d_cb), b = fastdiv(t1, g.d_band);
  DwhItem it;
  it.c0 = (int)(id - t1 * g.cblocks) * 16 * NT;
  it.oy0 = (int)(t1 - b * g.bands) * g.R;
  it.rows = g.R < g.Ho - it.oy0 ? g.R : g.Ho - it.oy0;
  it.b = b;
  return it;
}

// Input rows behind the rows of an item; row ir of them is image row oy0 * S - 1 + ir, and one outside the image is not fetched.
template <int S>
PULPNN_HD int dwh_rows_in(const DwhItem &it) { return (it.rows - 1) * S + 3; }
template <int S>
PULPNN_HD bool dwh_row_ok(const DwhGeom &g, const DwhItem &it, int ir) { return (unsigned)(it.oy0 * S - 1 + ir) < (unsigned)g.H && ir < dwh_rows_in<S>(it); }
// Offset in the input buffer of the lane's chunk of input row 0; row ir is ir * W * C further.
template <int W, int S>
PULPNN_HD unsigned dwh_in_offset(const DwhGeom &g, const DwhItem &it, int lane)
{
  constexpr int NT = 64 / W;
  return ((it.b * (unsigned)g.H + (unsigned)(it.oy0 * S)) * W + (unsigned)(lane / NT)) * (unsigned)g.C + (unsigned)(it.c0 + 16 * (lane % NT));
}
// Output rows.  With one tile of 16 channels (W = 64) a lane writes one pixel of a row, with stride 2 of the two rows from r on; otherwise a lane writes the 4 * NT channels of pixel l16 of strip x.  Offset in the output of
// what a lane writes of output row 0 (strip 0); row r is r * Wo * C further, strip x is 16 * x * C.
template <int W, int S>
PULPNN_HD unsigned dwh_out_offset(const DwhGeom &g, const DwhItem &it, int lane)
{
  constexpr int NT = 64 / W, WO = W / S;
  const unsigned row0 = (it.b * (unsigned)g.Ho + (unsigned)it.oy0) * WO * (unsigned)g.C + (unsigned)it.c0;
  return NT == 1 ? row0 + (unsigned)lane * (unsigned)g.C : row0 + (unsigned)(lane & 15) * (unsigned)g.C + 4u * NT * (unsigned)(lane >> 4);
}
// ... and whether output row r, or the part of rows r and r + 1 that the lane writes, exists
template <int W, int S>
PULPNN_HD bool dwh_out_ok(const DwhItem &it, int r, int lane) { return r + (W == 64 ? lane / (64 / S) : 0) < it.rows; }

// A row in LDS: W + 2 pixels of 16 * NT bytes, columns -1 .. W.  The chunks of a pixel change places with its column, so that
// the lanes that read one chunk of 8 neighbouring pixels meet 8 different places of the 128 bytes (stride 2: 4).
template <int W>
PULPNN_HD int dwh_lds(int col, int chunk)
{
  constexpr int NT = 64 / W;
  const int swz = NT == 1 ? 0 : NT == 2 ? (col >> 2) & 1 : (col >> 1) & 3;
  return (col * NT + (chunk ^ swz)) * 16;
}
template <int W>
PULPNN_HD constexpr int dwh_row_bytes() { return (W + 2) * (64 / W) * 16; }

// False for a layer the kernel does not take.
template <int W, int S>
bool dwh_shape(const DwLayer &L, int cus, DwhGeom *out)
{
  constexpr int NT = 64 / W;
  DwhGeom &g = *out;
  g = DwhGeom{};
  if (L.W != W || L.sx != S || L.CH % (16 * NT) || L.Wo != W / S || L.Ho > (L.H - 1) / S + 1) return false;
  const long long lead = (long long)W * L.CH, size = (long long)L.B * L.H * W * L.CH + lead;
  if (size >= 0x7fffffffLL) return false;
  g.in = L.in;
  g.wt = L.wt;
  g.bias = L.bias;
  g.out = L.out;
  g.C = L.CH;
  g.H = L.H;
  g.Ho = L.Ho;
  g.cblocks = L.CH / (16 * NT);
  // As many rows per wave as leave every SIMD one wave, at most 16: a wave reads two (stride 2: one) rows more than it needs by
  // itself, and sets up its channels' operands, some 100 instructions, for all of its rows.  Call by call, rows per wave 2 / 4 / 8 /
  // 16 at batch 256: 64x64x16 12.9 / 9.4 / 9.3 / 9.1 us, 32x32x64 14.0 / 10.0 / 9.5 / 8.7; batch 64 4.8 / 4.3 / 5.0 / 6.7 and 5.3 / 4.5 / 5.4 / 7.0.
  g.R = 16;
  while (g.R > 1 && (long long)L.B * ((L.Ho + g.R - 1) / g.R) * g.cblocks < 4ll * cus) g.R /= 2;
  g.bands = (L.Ho + g.R - 1) / g.R;
  const long long total = (long long)L.B * g.bands * g.cblocks;
  if (total > 0x7fffffffLL - 4) return false;
  g.total = (int)total;
  g.lead = (unsigned)lead;
  g.size = (unsigned)size;
  g.out_size = (unsigned)((long long)L.B * L.Ho * (W / S) * L.CH);
  g.d_cb = fastdiv_make((unsigned)g.cblocks);
  g.d_band = fastdiv_make((unsigned)g.bands);
  return true;
}
