// Addresses of igemm_kernel's range-checked activation loads.  Plain C++: the kernel uses it, and a host program can walk the
// same numbers.
#pragma once
#include "fastdiv.h"

PULPNN_HD int igemm_clamp(int n, int most) { return n < 0 ? 0 : n > most ? most : n; }

// What a lane keeps for one pixel row of the tile: the byte offset of its chunk at tap (0, 0), from a buffer that starts
// (pt * W + pl) * Ci bytes in front of the input, and one bit per tap that lies outside the image.  SUB: several taps per K
// slice (16 or 32 input channels); ck: the lane's 16-byte chunk of the slice.  G: ConvGeom.
template <bool SUB, class G>
PULPNN_HD void igemm_row_gather(const G &g, int m, int ck, unsigned *poff, unsigned *pinv)
{
  // (a row past the last pixel: with SUB the tap's offset is added to poff before the range check, so 0xffffffff
  // alone would wrap to an address in front of the input; every tap of such a row is out of range)
  *poff = 0xffffffffu;
  *pinv = SUB ? ~0u : 0u;
  if (m < g.M) {
    const int b = (int)fastdiv((unsigned)m, g.d_howo), rem = m - b * g.HoWo;
    const int oy = (int)fastdiv((unsigned)rem, g.d_wo), ox = rem - oy * g.Wo;
    *poff = (unsigned)b * (unsigned)g.in_img + (unsigned)((oy * g.sy * g.W + ox * g.sx) * g.Ci) +
            (SUB ? (16u * ck) & (unsigned)(g.Ci - 1) : 16u * ck);
    // taps inside the image: columns fx_lo .. fx_hi - 1 of rows fy_lo .. fy_hi - 1, a bit pattern of columns times one bit per row
    const int iy = oy * g.sy - g.pt, ix = ox * g.sx - g.pl;
    if (g.kx * g.ky == 1) {
      *pinv = (unsigned)iy < (unsigned)g.H && (unsigned)ix < (unsigned)g.W ? ~1u : ~0u;
      return;
    }
    const int fy_hi = igemm_clamp(g.H - iy, g.ky), fy_lo = igemm_clamp(-iy, fy_hi), fx_hi = igemm_clamp(g.W - ix, g.kx), fx_lo = igemm_clamp(-ix, fx_hi);
    unsigned rows = 0;
    for (int fy_ = 0; fy_ < g.ky; fy_++) rows |= 1u << (fy_ * g.kx);
    const unsigned in_rows = rows & (unsigned)((1ull << (fy_hi * g.kx)) - (1ull << (fy_lo * g.kx)));
    *pinv = ~((unsigned)((1ull << fx_hi) - (1ull << fx_lo)) * in_rows);  // (SUB: the tail of the last K slice past the filter too)
  }
}

// SUB: the offset of a chunk at tap t, all ones (out of range) for a tap outside the image
template <class G>
PULPNN_HD unsigned igemm_sub_offset(const G &g, unsigned poff, unsigned pinv, int t)
{
  const int tfy = (t * g.rkx) >> 16, tfx = t - tfy * g.kx;
  const unsigned toff = (unsigned)((tfy * g.W + tfx) * g.Ci);
#ifdef __HIP_DEVICE_COMPILE__
  const unsigned oob = (unsigned)__builtin_amdgcn_sbfe((int)pinv, t, 1);
#else
  const unsigned oob = 0u - (pinv >> t & 1u);
#endif
  return (poff + toff) | oob;
}
