// Division of a 32-bit unsigned number by a divisor fixed for the launch, as a multiply-high, an add and
// two shifts (Granlund & Montgomery); the host computes the constants.  The compiler's expansion of a
// 32-bit division is some 40 instructions, and a tile's set-up divides several times per lane.
// Also compiled by itself on the host (the tile arithmetic that is walked there).
#pragma once

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define PULPNN_HD __host__ __device__ __forceinline__
#else
#define PULPNN_HD inline
#endif

struct FastDiv {
  unsigned mul, sh1, sh2;
};
static inline FastDiv fastdiv_make(unsigned d)
{
  FastDiv f;
  unsigned l = 0;
  while ((1ull << l) < d) l++;  // ceil(log2(d))
  f.mul = (unsigned)(((1ull << 32) * ((1ull << l) - d)) / d + 1);
  f.sh1 = l < 1 ? l : 1;
  f.sh2 = l > 1 ? l - 1 : 0;
  return f;
}
PULPNN_HD unsigned fastdiv(unsigned n, const FastDiv &f)
{
#ifdef __HIP_DEVICE_COMPILE__
  const unsigned t = __umulhi(n, f.mul);
#else
  const unsigned t = (unsigned)(((unsigned long long)n * f.mul) >> 32);
#endif
  return (t + ((n - t) >> f.sh1)) >> f.sh2;
}
