// Addresses of igemm_kernel's range-checked activation loads.  Plain C++: the kernel uses it, and a host program can walk the
// same numbers.
#pragma once
#include "fastdiv.h"

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
    if (SUB) *pinv = ~0u << (g.kx * g.ky);  // taps past the filter (the tail of the last K slice)
    for (int fy_ = 0, t = 0; fy_ < g.ky; fy_++)
      for (int fx_ = 0; fx_ < g.kx; fx_++, t++) {
        const int iy = oy * g.sy - g.pt + fy_, ix = ox * g.sx - g.pl + fx_;
        if ((unsigned)iy >= (unsigned)g.H || (unsigned)ix >= (unsigned)g.W) *pinv |= 1u << t;
      }
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
