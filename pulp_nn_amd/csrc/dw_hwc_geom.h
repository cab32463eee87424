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

#define DWH_LARGE (64ll << 20)  // input and output, bytes
inline long long dwh_bytes(const DwLayer &L) { return (long long)L.B * L.CH * ((long long)L.H * L.W + (long long)L.Ho * L.Wo); }
// Large layers of rows of 64 pixels and 128 channels or more, where dw3x3_rows_kernel, which reads 64 channels of a pixel at a time, is
// the faster one; here / there: stride 1 64x64x128 batch 45 (47 MB in and out) 16.8 / 16.1 us, 91 37.1 / 33.4, 64x64x512 batch 22 36.9 / 33.6, 45 67.8 /
// 60.8, 35x64x128 batch 167 36.7 / 35.9, but 7x64x256 batch 418 36.3 / 38.8; stride 2 64x64x192 batch 61 (59 MB) 17.0 / 18.8, 122 42.7 / 35.7, 35x64x512
// batch 83 43.6 / 39.2, 7x64x256 batch 837 43.4 / 35.8.
inline bool dwh_wide(const DwLayer &L) { return L.W == 64 && L.CH >= 128 && (L.sx == 2 || L.Ho >= 16) && dwh_bytes(L) > DWH_LARGE; }

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
  // Rows per wave, 16 or a fraction of it: a wave walks down its rows one after the other and reads up to two more than it needs by
  // itself, and a SIMD whose waves are all resident takes about as long as that for each of them.  So the least product of rows and
  // rounds, in bands of one height (35 rows are 12 + 12 + 11, not 16 + 16 + 3), and the more rows where two are equal.  Rows per wave 2 / 4 /
  // 8 / 16 at batch 64 (1024 waves at 4 rows) 64x64x16 4.8 / 4.3 / 5.0 / 6.7 us, at batch 256 12.9 / 9.4 / 9.3 / 9.1; 16x16x128 batch 244 (976 waves at 8 rows)
  // 4 / 8 rows 7.8 / 6.9, 35x32x128 batch 55 (1980, 1100) 7.2 / 9.0; 35x64x32 batch 334 16 + 16 + 3 rows 11.3, 12 + 12 + 11 10.3.
  // At most 8 in large layers where a wave's 16 or 32 bytes of a pixel are a small part of it: the waves that read the rest of its lines
  // run apart from each other, the further the more rows they walk, and the lines are gone when they come.  8 / 16 rows: 64x64x64 batch 256
  // 40.9 / 43.4 us, 32x32x1024 batch 45 35.7 / 40.2, stride 2 64x64x512 batch 22 19.5 / 23.7, but 64x64x64 batch 256 24.8 / 21.8.
  const int least = S == 1 ? 4 : 2;  // rows that the kernel's loop does at a time
  long long cost = 0;
  for (int R = dwh_bytes(L) > DWH_LARGE && NT < 4 && g.cblocks > 2 * S ? 8 : 16; R >= 1; R /= 2) {
    const int even = (L.Ho + (L.Ho + R - 1) / R - 1) / ((L.Ho + R - 1) / R), rows = even > least ? (even + least - 1) / least * least : even;
    const int bands = (L.Ho + rows - 1) / rows;
    const long long waves = (long long)L.B * bands * g.cblocks, c = (waves + 4 * cus - 1) / (4 * cus) * (S * even + 2);
    if (cost && c >= cost) continue;
    cost = c;
    g.R = rows;
    g.bands = bands;
  }
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
