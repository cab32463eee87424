// Convolution, pointwise and linear layers: which kernel a shape takes, and its launch.
#include "host.h"

#include <algorithm>

#include "igemm.h"
#include "igemm_patch.h"
#include "igemm_ring.h"
#include "linear_skinny.h"
#include "pw_any_geom.h"
#include "pw_packed.h"
#include "pw_stream.h"
#include "smallk.h"

namespace {

// ---- implicit GEMM dispatch -------------------------------------------------

// launch-constant divisions of the tiled kernels (call after tiles_n is known)
void conv_geom_divs(ConvGeom &g)
{
  g.d_howo = fastdiv_make((unsigned)g.HoWo);
  g.d_wo = fastdiv_make((unsigned)g.Wo);
  g.d_tiles_n = fastdiv_make((unsigned)g.tiles_n);
  g.batch = (g.M + g.HoWo - 1) / g.HoWo;
  g.ci_shift = 0;
  while ((1 << (g.ci_shift + 1)) <= g.Ci) g.ci_shift++;
  g.rkx = 65536 / g.kx + 1;
}

template <int TN, int WM_, int WN_, int GATHER, int TM = 4, int ONEPASS = 0>
void launch_igemm_mode(int mode, ConvGeom &g, const EpiArgs &e, hipStream_t s)
{
  constexpr int BM = 16 * TM * WM_, BN = 16 * TN * WN_;
  const int tiles_m = (g.M + BM - 1) / BM;
  g.tiles_n = (g.N + BN - 1) / BN;
  g.tiles_total = tiles_m * g.tiles_n;
  conv_geom_divs(g);
  g.vec_store = (g.N % (4 * TN) == 0) && aligned(g.out, 4 * TN);
  // default store policy: the tiled kernel is not bound by HBM, its 16-byte pieces would reach HBM
  // uncombined with the streaming policy (1.36 x the bytes), and the next layer finds the output in cache
  g.nt = 0;
  dim3 grid(g.tiles_total), block(64 * WM_ * WN_);
  switch (mode) {
    case EPI_BN: hipLaunchKernelGGL((igemm_kernel<TN, WM_, WN_, GATHER, EPI_BN, TM, ONEPASS>), grid, block, 0, s, g, e); break;
    case EPI_MULT: hipLaunchKernelGGL((igemm_kernel<TN, WM_, WN_, GATHER, EPI_MULT, TM, ONEPASS>), grid, block, 0, s, g, e); break;
    case EPI_RAW: hipLaunchKernelGGL((igemm_kernel<TN, WM_, WN_, GATHER, EPI_RAW, TM, ONEPASS>), grid, block, 0, s, g, e); break;
    default: hipLaunchKernelGGL((igemm_kernel<TN, WM_, WN_, GATHER, EPI_OUT32, TM, ONEPASS>), grid, block, 0, s, g, e); break;
  }
}

// 256 x 256 tiles of persistent workgroups fed by LDS-direct loads (igemm_ring.h).  Returns false if the shape
// does not qualify or the kernel cannot be launched (the caller then uses the tiled kernel).
bool launch_igemm_ring(int mode, ConvGeom &g, const EpiArgs &e, hipStream_t s)
{
  typedef IgrShape<4> S;
  // K: at least as many sub-slices as ring stages; below 2^16, so that accumulator and correction term each
  // fit 32 bits (the epilogue adds them in 64-bit arithmetic in the 64-bit build)
  if (g.Ci % 64 || g.K < 64 * S::NS || g.K >= 65536 || g.N % 16 || !aligned(g.out, 16) || mode == EPI_OUT32) return false;
  g.tiles_n = (g.N + S::BN - 1) / S::BN;
  g.tiles_total = ((g.M + IGR_BM - 1) / IGR_BM) * g.tiles_n;
  // the grid: a multiple of 8 * tiles_n workgroups (a workgroup keeps its channel range, an XCD gets whole
  // pixel tiles), at most one per compute unit and no more than there are tiles
  const int unit = 8 * g.tiles_n;
  const int grid_n = (int)(std::min<long long>(num_cus(), g.tiles_total) / unit) * unit;
  if (grid_n <= 0) return false;
  conv_geom_divs(g);
  g.cpt = g.Ci / 64;
  g.d_cpt = fastdiv_make((unsigned)g.cpt);
  g.d_kx = fastdiv_make((unsigned)g.kx);
  g.vec_store = 1;
  g.nt = (long long)g.M * g.N >= PULPNN_NT_BYTES;
  const size_t lds = (size_t)S::lds_bytes();
  const dim3 grid(grid_n), block(S::THREADS);
  switch (mode) {
    case EPI_BN:
      if (!raise_lds_limit<igemm_ring_kernel<EPI_BN, 4>>(lds)) return false;
      hipLaunchKernelGGL((igemm_ring_kernel<EPI_BN, 4>), grid, block, lds, s, g, e);
      break;
    case EPI_MULT:
      if (!raise_lds_limit<igemm_ring_kernel<EPI_MULT, 4>>(lds)) return false;
      hipLaunchKernelGGL((igemm_ring_kernel<EPI_MULT, 4>), grid, block, lds, s, g, e);
      break;
    default:
      if (!raise_lds_limit<igemm_ring_kernel<EPI_RAW, 4>>(lds)) return false;
      hipLaunchKernelGGL((igemm_ring_kernel<EPI_RAW, 4>), grid, block, lds, s, g, e);
      break;
  }
  return true;
}

// 4-row x 64-column output patches whose input rows are staged once per filter row (igemm_patch.h): 3-wide
// stride-1 filters on images of 57 to 64 output columns.  Returns false if the shape does not qualify.
bool launch_igemm_patch(int mode, ConvGeom &g, const EpiArgs &e, hipStream_t s)
{
  if (g.kx != 3 || g.sx != 1 || g.sy != 1 || g.pl > 1 || g.Wo > 64 || g.ky > 31) return false;
  if (g.Ci % 64 || g.ky * (g.Ci / 64) < 2 || g.K >= 65536 || g.N % 16 || !aligned(g.out, 16) || mode == EPI_OUT32) return false;
  if (g.M % g.HoWo) return false;  // whole images
  // pixels wanted against pixels computed (whole patches): at least nine tenths
  const int rgroups = (g.Ho + 3) / 4;
  if ((long long)g.Ho * g.Wo * 10 < (long long)rgroups * 4 * 64 * 9) return false;
  g.tiles_n = (g.N + IGP_BN - 1) / IGP_BN;
  conv_geom_divs(g);
  g.rgroups = rgroups;
  g.d_rg = fastdiv_make((unsigned)rgroups);
  const long long tiles = (long long)g.batch * rgroups * g.tiles_n;
  if (tiles > 0x7fffffffLL) return false;
  g.tiles_total = (int)tiles;
  const int unit = 8 * g.tiles_n;
  const int grid_n = (int)(std::min<long long>(num_cus(), g.tiles_total) / unit) * unit;
  if (grid_n <= 0) return false;
  g.cpt = g.Ci / 64;
  g.d_cpt = fastdiv_make((unsigned)g.cpt);
  g.d_kx = fastdiv_make((unsigned)g.kx);
  g.vec_store = 1;
  g.nt = (long long)g.M * g.N >= PULPNN_NT_BYTES;
  const size_t lds = (size_t)igp_lds_bytes();
  const dim3 grid(grid_n), block(IGP_THREADS);
  switch (mode) {
    case EPI_BN:
      if (!raise_lds_limit<igemm_patch_kernel<EPI_BN>>(lds)) return false;
      hipLaunchKernelGGL((igemm_patch_kernel<EPI_BN>), grid, block, lds, s, g, e);
      break;
    case EPI_MULT:
      if (!raise_lds_limit<igemm_patch_kernel<EPI_MULT>>(lds)) return false;
      hipLaunchKernelGGL((igemm_patch_kernel<EPI_MULT>), grid, block, lds, s, g, e);
      break;
    default:
      if (!raise_lds_limit<igemm_patch_kernel<EPI_RAW>>(lds)) return false;
      hipLaunchKernelGGL((igemm_patch_kernel<EPI_RAW>), grid, block, lds, s, g, e);
      break;
  }
  return true;
}

// 128 px x 64 ch tiles, for layers too small to fill the machine with larger ones.  With at most five
// K slices (K <= 320) a tile's whole K extent fits in LDS and is fetched in one go.  Eight waves of 32 x 32 per tile
// rather than four of 64 x 32: these layers are a chain of latencies (gather, stage, multiply, store), and with twice
// the waves every link is issued in half the time (config 0: 7.0 -> 6.6 us).  Longer ones nine slices at a time in 110 KB where
// every tile has a compute unit to itself (16x16 64 -> 64 batch 64 6.4 -> 5.6 us, 14x14 128 -> 128 batch 60 9.9 -> 8.8, 12x12 256 -> 200 batch 5
// 14.4 -> 13.3; but 316 tiles, 10x10 256 -> 256 batch 100, 19.5 -> 26.5).
template <int GATHER>
void launch_igemm_small(int mode, ConvGeom &g, const EpiArgs &e, hipStream_t s)
{
  if (GATHER != GATHER_BYTES && g.K <= 5 * IGEMM_BK) launch_igemm_mode<2, 4, 2, GATHER, 2, 5>(mode, g, e, s);
  else if (GATHER == GATHER_UNIFORM && (long long)((g.M + 127) / 128) * ((g.N + 63) / 64) <= num_cus())
    launch_igemm_mode<2, 4, 2, GATHER, 2, GATHER == GATHER_UNIFORM ? 9 : 0>(mode, g, e, s);
  else launch_igemm_mode<2, 4, 2, GATHER, 2>(mode, g, e, s);
}

template <int GATHER>
void launch_igemm_tile(int mode, ConvGeom &g, const EpiArgs &e, hipStream_t s)
{
  // 256 px x 256 ch with 16 waves when there are at least two such tiles per CU: half the
  // L2 -> LDS bytes per multiply of the 128 x 128 tile
  const long long big_tiles = (long long)((g.M + 255) / 256) * ((g.N + 255) / 256);
  if (GATHER == GATHER_UNIFORM && g.N > 128 && big_tiles >= 2 * num_cus()) {
    // operands go HBM/L2 -> LDS without passing through registers, persistent workgroups
    if (launch_igemm_patch(mode, g, e, s)) return;
    if (launch_igemm_ring(mode, g, e, s)) return;
    launch_igemm_mode<4, 4, 4, GATHER>(mode, g, e, s);
  } else
  // 128 px x 64 ch while 128 x 128 tiles would give a CU at most one workgroup: twice the workgroups to
  // hide each other's latency (such layers are a few K slices long)
  if (g.N > 64 && (long long)((g.M + 127) / 128) * ((g.N + 127) / 128) <= num_cus()) launch_igemm_small<GATHER>(mode, g, e, s);
  else
  if (g.N > 64) launch_igemm_mode<4, 2, 2, GATHER>(mode, g, e, s);       // 128 px x 128 ch
  else if (g.N > 32 && (g.M + 255) / 256 < 2 * num_cus()) launch_igemm_small<GATHER>(mode, g, e, s);  // 128 px x 64 ch: more workgroups
  else if (g.N > 32) launch_igemm_mode<4, 4, 1, GATHER>(mode, g, e, s);  // 256 px x 64 ch
  else if (g.N > 16) launch_igemm_mode<2, 4, 1, GATHER>(mode, g, e, s);  // 256 px x 32 ch
  else launch_igemm_mode<1, 4, 1, GATHER>(mode, g, e, s);                // 256 px x 16 ch
}

void launch_igemm(int mode, ConvGeom &g, const EpiArgs &e, hipStream_t s)
{
  const bool chunk16 = (g.Ci % 16 == 0) && aligned(g.in, 16) && aligned(g.w, 16);
  // scalar tap walk + range-checked buffer loads: whole K slices inside one tap, one bit
  // per tap in a 32-bit mask, 32-bit byte offsets
  const long long batch = (g.M + g.HoWo - 1) / g.HoWo;
  const bool uniform = chunk16 && (g.Ci % 64 == 0) && g.kx * g.ky <= 32 &&
                       batch * g.in_img + (long long)(g.pt * g.W + g.pl) * g.Ci < 0x7fffffffLL &&
                       (long long)g.N * g.K < 0x7fffffffLL;
  // 16 or 32 input channels: two or four whole taps per K slice, same buffer loads (one bit per tap up to
  // the end of the last slice must fit the 32-bit mask)
  const bool subtap = chunk16 && (g.Ci == 16 || g.Ci == 32) && g.kx * g.ky + 64 / g.Ci <= 32 && g.kx <= 32 &&
                      batch * g.in_img + (long long)(g.pt * g.W + g.pl) * g.Ci + (long long)(g.ky * g.W + g.kx) * g.Ci < 0x7fffffffLL &&
                      (long long)g.N * g.K + 64 < 0x7fffffffLL;
  if (uniform) launch_igemm_tile<GATHER_UNIFORM>(mode, g, e, s);
  else if (subtap) launch_igemm_tile<GATHER_SUBTAP>(mode, g, e, s);
  else if (chunk16) launch_igemm_tile<GATHER_CHUNK16>(mode, g, e, s);
  else launch_igemm_tile<GATHER_BYTES>(mode, g, e, s);
}

// Direct (vector ALU) convolution for filters of at most 32 bytes and at most 32 channels, gathered byte by byte.
template <int NCH>
void launch_smallk(int mode, ConvGeom &g, const EpiArgs &e, hipStream_t s)
{
  g.vec_store = (g.N == NCH) && aligned(g.out, 16);
  g.nt = (long long)g.M * g.N >= PULPNN_NT_BYTES;
  dim3 grid((unsigned)((g.M + 255) / 256)), block(256);
  switch (mode) {
    case EPI_BN: hipLaunchKernelGGL((smallk_conv_kernel<NCH, EPI_BN>), grid, block, 0, s, g, e); break;
    case EPI_MULT: hipLaunchKernelGGL((smallk_conv_kernel<NCH, EPI_MULT>), grid, block, 0, s, g, e); break;
    default: hipLaunchKernelGGL((smallk_conv_kernel<NCH, EPI_RAW>), grid, block, 0, s, g, e); break;
  }
}

template <auto KERN>
bool launch_skinny_kernel(const SkinnyGeom &g, const EpiArgs &e, dim3 grid, hipStream_t s)
{
  if (!raise_lds_limit<KERN>(SKINNY_LDS)) return false;
  hipLaunchKernelGGL(KERN, grid, dim3(256), SKINNY_LDS, s, g, e);
  return true;
}
template <int MODE, bool ANY>
bool launch_skinny_mode(const SkinnyGeom &g, const EpiArgs &e, dim3 grid, hipStream_t s)
{
  if constexpr (ANY) return launch_skinny_kernel<linear_skinny_any_kernel<MODE>>(g, e, grid, s);
  else return launch_skinny_kernel<linear_skinny_kernel<MODE>>(g, e, grid, s);
}
template <bool ANY>
bool launch_skinny(int mode, const SkinnyGeom &g, const EpiArgs &e, dim3 grid, hipStream_t s)
{
  switch (mode) {
    case EPI_BN: return launch_skinny_mode<EPI_BN, ANY>(g, e, grid, s);
    case EPI_MULT: return launch_skinny_mode<EPI_MULT, ANY>(g, e, grid, s);
    case EPI_RAW: return launch_skinny_mode<EPI_RAW, ANY>(g, e, grid, s);
    default: return launch_skinny_mode<EPI_OUT32, ANY>(g, e, grid, s);
  }
}

// Launches one instantiation; raises its dynamic-LDS limit above the default 64 KB as needed.
template <auto KERN>
bool launch_pw(const PwGeom &g, const EpiArgs &e, dim3 grid, dim3 block, size_t lds, hipStream_t s)
{
  if (!raise_lds_limit<KERN>(lds)) return false;
  hipLaunchKernelGGL(KERN, grid, block, lds, s, g, e);
  return true;
}

// Two shapes of the streaming kernel: 16 waves taking 16 pixels per step for launches
// with at least three steps for every wave of every CU (more waves in flight hide the
// arithmetic of a step behind the memory traffic of the others), 8 waves taking 32 pixels
// per step otherwise (half the LDS reads per pixel, and the 128-register budget of the
// 16-wave shape is too small for K = 256).
template <int TN, int NP, int KS, int TM, int NW>
bool launch_pw_stream_mode(int mode, const PwGeom &g, const EpiArgs &e, dim3 grid, size_t lds, hipStream_t s)
{
  dim3 block(64 * NW);
  switch (mode) {
    case EPI_BN: return launch_pw<pw_stream_kernel<TN, KS, NP, EPI_BN, false, TM, NW>>(g, e, grid, block, lds, s);
    case EPI_MULT:
      if (e.shift >= 16) return launch_pw<pw_stream_kernel<TN, KS, NP, EPI_MULT, true, TM, NW>>(g, e, grid, block, lds, s);
      return launch_pw<pw_stream_kernel<TN, KS, NP, EPI_MULT, false, TM, NW>>(g, e, grid, block, lds, s);
    default: return launch_pw<pw_stream_kernel<TN, KS, NP, EPI_RAW, false, TM, NW>>(g, e, grid, block, lds, s);
  }
}

template <int TN, int NP>
bool launch_pw_stream_ks(int mode, int ks, bool wide, const PwGeom &g, const EpiArgs &e, dim3 grid, size_t lds,
                         hipStream_t s)
{
  if (ks == 1) {
    if (wide) return launch_pw_stream_mode<TN, NP, 1, 1, 16>(mode, g, e, grid, lds, s);
    return launch_pw_stream_mode<TN, NP, 1, 2, 8>(mode, g, e, grid, lds, s);
  } else if (ks == 2) {
    if (wide) return launch_pw_stream_mode<TN, NP, 2, 1, 16>(mode, g, e, grid, lds, s);
    return launch_pw_stream_mode<TN, NP, 2, 2, 8>(mode, g, e, grid, lds, s);
  } else {
    return launch_pw_stream_mode<TN, NP, 4, 2, 8>(mode, g, e, grid, lds, s);
  }
}

template <int K16, int Q>
void launch_pw_packed(int mode, PwGeom &g, const EpiArgs &e, hipStream_t s)
{
  constexpr int PX = 64 / K16;
  g.units = (g.M + PX - 1) / PX;
  const dim3 grid(std::min((g.units + 3) / 4, 4 * num_cus())), block(256);
  if (g.nt) hipLaunchKernelGGL((pw_packed_kernel<K16, Q, true>), grid, block, 0, s, g, e, mode);
  else hipLaunchKernelGGL((pw_packed_kernel<K16, Q, false>), grid, block, 0, s, g, e, mode);
}

// Weights-stationary streaming path: a GEMM whose rows are contiguous K-byte pixels,
// whose weight matrix (at most 256 x 256) fits in LDS and whose channel count is one
// of 16, 32, 64, 128, 192, 256 (every lane then owns real channels and stores whole
// vectors).  Returns false if the shape does not qualify (the caller then uses the
// tiled kernel).
bool try_pw_stream(int mode, const uint8_t *in, const int8_t *w, const int8_t *bias, void *out, long long M, int N,
                   int K, const EpiArgs &e, hipStream_t s)
{
  if (K > 256 || (K % 16) || !aligned(in, 16) || !aligned(w, 16) || !aligned(out, 16) || M < 2048 || M > PW_MOST_PIXELS) return false;
  if (!(N == 16 || N == 32 || N == 64 || N == 128 || N == 192 || N == 256)) return false;
  if (mode == EPI_OUT32) return false;
  const int tn = N == 16 ? 1 : (N == 32 ? 2 : 4);
  const int np = N / (16 * tn);
  const int ks = K <= 64 ? 1 : (K <= 128 ? 2 : 4);
  PwGeom g;
  g.in = in;
  g.w = w;
  g.bias = bias;
  g.out = out;
  g.M = (int)M;
  g.N = N;
  g.K = K;
  g.units = (int)((M + 15) / 16);
  g.nt = M * N >= PULPNN_NT_BYTES;
  const bool wide = ks <= 2 && g.units >= 3 * 16 * num_cus();
  const int nw = wide ? 16 : 8, tm = wide ? 1 : 2;
  const int lds = pw_lds_bytes(tn, ks, np, mode == EPI_BN, nw, tm);
  if (lds > 160 * 1024 - 512) return false;  // 512: static LDS of the kernel
  // Persistent grid: one workgroup per CU (the weights are staged once per CU), fewer
  // when there are not two 16-pixel units for every wave.
  int blocks = num_cus();
  const int need = (g.units + 2 * nw - 1) / (2 * nw);
  if (blocks > need) blocks = need;
  // a launch that would leave more than half of the CUs without a workgroup is better off tiled:
  // every CU takes part there, and staging the weights per workgroup no longer pays
  if (2 * need < num_cus()) return false;
  // Several pixels of 16 or 32 channels in a column of the matrix cores, from a load of 16 channels for every wave on (of 32 that is two loads a wave).  One pixel a
  // column / so, kernel times, batches of 64x64: batch 64 16 -> 16 5.3 / 4.1 us, 16 -> 32 6.0 / 5.4, 32 -> 64 7.4 / 6.7; batch 128 7.2 / 5.1, 8.2 / 6.6, 10.2 / 8.4; below
  // the line batch 56 5.0 / 4.0, 5.6 / 5.2, 7.3 / 6.5; batch 48 4.8 / 3.7, 5.4 / 4.7, 7.0 / 6.2; batch 32 3.7 / 3.2, 4.1 / 3.9, 5.2 / 5.4; with 64 bits 16 -> 16 batch 64 5.4 / 5.1,
  // 56 5.0 / 5.0, 32 3.7 / 3.9: with 32 bits a line at three quarters of it, for 16 channels lower still, that this rule does not draw.  Not where its
  // registers leave too few waves: 16 -> 64 7.6 / 8.0, 32 -> 32 3.9 / 4.5 and 6.8 / 6.9; with constants of 64 bits 16 -> 32 6.0 / 7.8, 32 -> 64 8.2 / 10.3.
  if (M >= 64ll * 16 * num_cus()) {
    if (K == 16 && N == 16) return launch_pw_packed<1, 1>(mode, g, e, s), true;
    if constexpr (sizeof(bn_t) == 4) {
      if (K == 16 && N == 32) return launch_pw_packed<1, 2>(mode, g, e, s), true;
      if (K == 32 && N == 64) return launch_pw_packed<2, 4>(mode, g, e, s), true;
    }
  }
  dim3 grid(blocks);
  // (false also if the kernel's LDS limit cannot be raised: the caller then uses the tiled kernel)
  if (tn == 1) return launch_pw_stream_ks<1, 1>(mode, ks, wide, g, e, grid, lds, s);
  if (tn == 2) return launch_pw_stream_ks<2, 1>(mode, ks, wide, g, e, grid, lds, s);
  if (np == 1) return launch_pw_stream_ks<4, 1>(mode, ks, wide, g, e, grid, lds, s);
  if (np == 2) return launch_pw_stream_ks<4, 2>(mode, ks, wide, g, e, grid, lds, s);
  if (np == 3) return launch_pw_stream_ks<4, 3>(mode, ks, wide, g, e, grid, lds, s);
  return launch_pw_stream_ks<4, 4>(mode, ks, wide, g, e, grid, lds, s);
}

}  // namespace

// Shared body of the six convolution entry points.
void conv_common(const char *fn, bool pointwise, const uint8_t *in, const int8_t *bias, uint8_t *out,
                 const int8_t *w, bn_t *k, bn_t *lambda, uint16_t out_mult, uint16_t out_shift,
                 uint16_t dim_in_x, uint16_t dim_in_y, uint16_t ch_in, uint16_t dim_out_x, uint16_t dim_out_y,
                 uint16_t ch_out, uint16_t kx, uint16_t ky, uint16_t pt, uint16_t pl, uint16_t sx, uint16_t sy,
                 int flag_relu, int flag_batch_norm)
{
  if (!in || !out || !w) return set_error(PULP_NN_HIP_ERR_ARGUMENT, fn, "null activation or weight pointer");
  if (!dim_in_x || !dim_in_y || !ch_in || !dim_out_x || !dim_out_y || !ch_out)
    return set_error(PULP_NN_HIP_ERR_ARGUMENT, fn, "zero dimension");
  if (pointwise) {
    // pulp_nn_pointwise_HoWo_parallel.c:103 reads pixel (y, x) of the input for output (y, x)
    kx = ky = 1;
    pt = pl = 0;
    sx = sy = 1;
    if (dim_out_x > dim_in_x || dim_out_y > dim_in_y)
      return set_error(PULP_NN_HIP_ERR_ARGUMENT, fn, "pointwise output larger than input");
  } else if (!kx || !ky || !sx || !sy) {
    return set_error(PULP_NN_HIP_ERR_ARGUMENT, fn, "zero kernel size or stride");
  }
  const int mode = epi_mode(flag_relu, flag_batch_norm);
  EpiArgs e;
  if (!epi_args(mode, k, lambda, out_mult, out_shift, &e))
    return set_error(PULP_NN_HIP_ERR_ARGUMENT, fn, "out_shift out of range or null k/lambda");
  const long long M = (long long)g_batch * dim_out_x * dim_out_y;
  if (M > 0x7fffffffLL) return set_error(PULP_NN_HIP_ERR_ARGUMENT, fn, "batch too large");
  if (kx == 1 && ky == 1 && sx == 1 && sy == 1 && pt == 0 && pl == 0 && dim_out_x == dim_in_x && dim_out_y == dim_in_y &&
      (try_pw_stream(mode, in, w, bias, out, M, ch_out, ch_in, e, g_stream) ||
       launch_pw_any(mode, in, w, bias, out, M, ch_out, ch_in, e, num_cus(), g_stream)))
    return check_launch(fn);
  ConvGeom g;
  g.in = in;
  g.w = w;
  g.bias = bias;
  g.out = out;
  g.M = (int)M;
  g.N = ch_out;
  g.K = (int)kx * ky * ch_in;
  g.H = dim_in_y;
  g.W = dim_in_x;
  g.Ci = ch_in;
  g.Ho = dim_out_y;
  g.Wo = dim_out_x;
  g.HoWo = (int)dim_out_x * dim_out_y;
  g.kx = kx;
  g.ky = ky;
  g.pt = pt;
  g.pl = pl;
  g.sx = sx;
  g.sy = sy;
  g.in_img = (long long)dim_in_x * dim_in_y * ch_in;
  // Filters of up to four rows of up to 16 bytes: a row is one 16-byte slot of K on the matrix cores, whatever the geometry.  Small pointwise
  // layers of 16 channels leave three slots of four empty; up to 32 output channels that is still the faster one (64x64 16 -> 32 batch 1
  // 6.9 us a pixel per lane, 3.6 here), beyond them the tiled kernel is (20x20 16 -> 256 batch 3 3.9 us, 4.4 here; batch 20 4.1 / 5.0).
  const ConvLayer L = {in, w, bias, out, (int)g_batch, dim_in_y, dim_in_x, ch_in, dim_out_y, dim_out_x, ch_out, kx, ky, pt, pl, sx, sy};
  const bool tiled16 = kx == 1 && ky == 1 && ch_in == 16 && ch_out > 32 && aligned(in, 16) && aligned(w, 16);
  if (!tiled16 && launch_conv_rows(mode, L, e, num_cus(), g_stream)) return check_launch(fn);
  if (g.K <= 4 * SMALLK_KD && g.N <= 32) {
    if (g.N <= 16) launch_smallk<16>(mode, g, e, g_stream);
    else launch_smallk<32>(mode, g, e, g_stream);
  } else {
    // Channel counts that are not whole 16-byte chunks: from a band of the input in LDS (conv_band.h).  So are layers of
    // few output channels, which leave most of the tiled kernel's 128 x 64 tile empty and its many waves waiting for each
    // other (kernel times, tiled / band: 8x38x9 240 -> 32 s2 21.9 / 10.8 us; 2x8x13 48 -> 16 5x5 14.2 / 6.6; 31x19 80 -> 16
    // 9.8 / 5.6; 23x14 144 -> 35 11.2 / 7.2, batch 23 11.4 / 8.3; 37x19 48 -> 20 batch 22 8.7 / 5.8; but 252x12x29 64 -> 40 s2 5.9 / 7.3).
    // 16 and 32 input channels stay with the tiled kernel, which takes two or four taps per K slice there.  It is the faster one
    // from 40 output channels on (tiled / band, 32 -> 64 at batch 256 16x16 6.1 / 8.0, batch 133 28x28 9.9 / 13.0, batch 64 64x64
    // 16.2 / 22.6; 8x57x43 32 -> 40 4.8 / 6.2) and the slower one below on small layers (16x16 32 -> 24 batch 1 6.7 / 4.6, 32x32 32 -> 32 batch 16
    // 6.3 / 5.0, 8x57x43 16 -> 24 6.4 / 5.0, 256x16x16 32 -> 16 5.8 / 5.6; but 256x16x16 32 -> 32 6.4 / 7.0, 133x28x28 16 -> 32 6.6 / 7.7, 64x64x64
    // 32 -> 32 10.6 / 14.2): a line by output channels and size that this rule does not draw.
    const bool whole16 = ch_in % 16 == 0 && aligned(in, 16) && aligned(w, 16);
    // Up to 128 output channels it is also the faster one for many layers whose channel count is no multiple of 64, which the tiled kernel gathers
    // chunk by chunk (band_for_odd_channels; up to 64 band_for_up_to_64).
    auto odd64 = [&] { return g.N > 64 ? band_for_odd_channels(L, num_cus(), (int)sizeof(bn_t)) : band_for_up_to_64(L, num_cus(), (int)sizeof(bn_t)); };
    const bool few = ch_in == 16 || ch_in == 32 ? false : g.N <= 32 || (ch_in % 64 && odd64());
    if (!whole16 || few) {
      if (launch_conv_band(mode, L, e, num_cus(), g_stream)) return check_launch(fn);
    }
    launch_igemm(mode, g, e, g_stream);
  }
  check_launch(fn);
}

void linear_common(const char *fn, int mode, const uint8_t *in, const int8_t *bias, void *out, const int8_t *w,
                   const EpiArgs &e, uint16_t dim_vec, uint16_t num_o_neurons, int rows)
{
  if (!in || !out || !w) return set_error(PULP_NN_HIP_ERR_ARGUMENT, fn, "null pointer");
  if (!dim_vec || !num_o_neurons) return set_error(PULP_NN_HIP_ERR_ARGUMENT, fn, "zero dimension");
  // few rows: a workgroup per 16 neurons streams their weights once, no staging and no K-slice barriers; rows that are
  // not whole aligned 16-byte chunks by unaligned loads (shorter than one chunk: the tiled kernel)
  if (rows <= 256 && dim_vec >= 16) {
    const int rblocks = (rows + 63) / 64, ngroups = (num_o_neurons + 15) / 16;
    // K in four parts and a workgroup per block of rows while that still leaves CUs without work
    const bool spread = ngroups * rblocks <= 2 * num_cus();
    const int kparts = spread ? 4 : (rblocks == 1 ? 4 : (rblocks == 2 ? 2 : 1));
    const SkinnyGeom sg = {in, w, bias, out, rows, (int)num_o_neurons, (int)dim_vec, kparts, kparts == 4 ? 2 : kparts == 2 ? 1 : 0,
                           num_o_neurons % 4 == 0 && aligned(out, 4)};
    const dim3 grid(ngroups, spread ? rblocks : 1);
    const bool whole = dim_vec % 16 == 0 && aligned(in, 16) && aligned(w, 16);
    if (whole ? launch_skinny<false>(mode, sg, e, grid, g_stream) : launch_skinny<true>(mode, sg, e, grid, g_stream)) return check_launch(fn);
  }
  ConvGeom g;
  g.in = in;
  g.w = w;
  g.bias = bias;
  g.out = out;
  g.M = rows;
  g.N = num_o_neurons;
  g.K = dim_vec;
  g.H = g.W = 1;
  g.Ci = dim_vec;
  g.Ho = g.Wo = g.HoWo = 1;
  g.kx = g.ky = 1;
  g.pt = g.pl = 0;
  g.sx = g.sy = 1;
  g.in_img = dim_vec;
  launch_igemm(mode, g, e, g_stream);
  check_launch(fn);
}

