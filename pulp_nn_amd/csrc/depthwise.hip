// Depthwise layers: which kernel a shape takes, and its launch.
#include "host.h"

#include <algorithm>

#include "depthwise.h"
#include "depthwise_stream.h"

// ---- depthwise dispatch -------------------------------------------------------

void depthwise_common(const char *fn, const uint8_t *in, const int8_t *bias, uint8_t *out, const int8_t *wt,
                      bn_t *k, bn_t *lambda, uint16_t out_mult, int out_shift, int W, int H, int Wo, int Ho, int CH,
                      int kx, int ky, int pt, int pl, int sx, int sy, int mode, bool hwc_in)
{
  if (!in || !out || !wt) return set_error(PULP_NN_HIP_ERR_ARGUMENT, fn, "null activation or weight pointer");
  if (W <= 0 || H <= 0 || Wo <= 0 || Ho <= 0 || CH <= 0 || kx <= 0 || ky <= 0 || sx <= 0 || sy <= 0)
    return set_error(PULP_NN_HIP_ERR_ARGUMENT, fn, "zero dimension");
  EpiArgs e;
  if (!epi_args(mode, k, lambda, out_mult, out_shift, &e))
    return set_error(PULP_NN_HIP_ERR_ARGUMENT, fn, "out_shift out of range or null k/lambda");
  // the accumulators of these kernels fit easily; guard the i32 sum anyway
  if ((long long)kx * ky > 4096) return set_error(PULP_NN_HIP_ERR_UNSUPPORTED, fn, "kernel too large");

  DwGeom g;
  g.in = in;
  g.wt = wt;
  g.bias = bias;
  g.out = out;
  g.B = (int)g_batch;
  g.CH = CH;
  g.H = H;
  g.W = W;
  g.Ho = Ho;
  g.Wo = Wo;
  g.kx = kx;
  g.ky = ky;
  g.pt = pt;
  g.pl = pl;
  g.sx = sx;
  g.sy = sy;
  g.planes = (long long)g.B * CH;
  g.cgroups = (CH + DW_CG - 1) / DW_CG;
  const bool fast = kx == 3 && ky == 3 && sx == sy && (sx == 1 || sx == 2) && (pl == 0 || pl == 1);
  // small square planes, padding 1: one plane per lane, in registers
  const int ho_plane = (H - 1) / sx + 1;
  const bool plane = fast && W == H && pt == 1 && pl == 1 && ((H == 8) || (H == 4 && sx == 1)) && Ho == ho_plane &&
                     Wo == ho_plane && CH % DW_CG == 0 && aligned(in, hwc_in ? 4 : 16) && aligned(out, 4) &&
                     (long long)g.B * g.cgroups <= 0x7fffffffLL;
  // rows of 16, 32 or 64 bytes, padding 1, any height: a few rows of a plane per lane, in registers
  // (Batch x channels of whole groups of 64: dw3x3_rows_kernel needs it.  The HWC kernel on the matrix cores does not, but HWC layers
  // have no other kernel, and which calls are refused does not depend on how a buffer is aligned.)
  const bool rowsk = !plane && fast && pt == 1 && pl == 1 && (W == 16 || W == 32 || W == 64) && Wo == (W - 1) / sx + 1 &&
                     Ho <= (H - 1) / sy + 1 && CH % 4 == 0 && ((long long)g_batch * CH) % DW_CG == 0 && aligned(in, hwc_in ? 4 : 16) &&
                     aligned(out, 4) && (long long)g_batch * CH / DW_CG * Ho < 0x7fffffffLL;
  // Whole 64-channel groups on rows of whole dwords: bands staged by LDS-direct loads (dw3x3_lin_kernel).  Bands are
  // kept under 40 KiB, so that four workgroups share a compute unit and the loads of one are covered by the arithmetic
  // of the others; not when that would leave fewer than 6 (stride 2: 4) output rows per band (ky - sy more input rows
  // are staged per band than it consumes alone).
  bool lin = !plane && !rowsk && !hwc_in && fast && W % 4 == 0 && W / 4 * 3 <= 255 && aligned(in, 16) && CH % DW_CG == 0 &&
             Wo % 4 == 0 && aligned(out, 4) && (long long)g_batch * CH * H * W < 0x7fffffffLL;
  size_t lin_lds = 0;
  if (lin) {
    g.LP = 0;
    g.LWD = W / 4;
    int max_csd = 255;  // 64 channels x 255 dwords = 63.75 KiB of LDS
    if ((156 / g.LWD - ky) / sy + 1 >= (sx == 1 ? 6 : 4)) max_csd = 156;
    const int rb_max = std::min((max_csd / g.LWD - ky) / sy + 1, Ho);
    g.bands = (Ho + rb_max - 1) / rb_max;
    g.RB = (Ho + g.bands - 1) / g.bands;
    g.bands = (Ho + g.RB - 1) / g.RB;
    g.NR = (g.RB - 1) * sy + ky;
    g.CSD = ((g.NR * g.LWD + 3) & ~3) | 1;  // room for the last 16-byte piece of a band
    lin_lds = DW_CG * (size_t)g.CSD * 4 + 16;
    lin = lin_lds <= 64 * 1024 && (long long)g.B * g.bands * g.cgroups <= 0x7fffffffLL;
  }
  // Layers that fill the machine with one workgroup per image and 64 channels (two per compute unit): the plane
  // streamed through LDS, 8 rows of it per request.  Up to 14 groups of 4 output columns, 64 KiB of LDS.  A chunk
  // costs a barrier and a round trip to memory however few rows it holds, so at stride 1 only planes of whole chunks
  // take this kernel: 56 rows do, the 58 pre-padded rows of pulp_nn_depthwise_3x3_s1 run faster in bands (57 / 51 us).
  // Kernel times streamed / in bands, stride 1: 56x56x128 batch 256 52.1 / 54.2 us, 48x48x256 batch 128 36.2 / 40.1, 40x52x64
  // batch 512 34.4 / 36.1; but 64 images of 56x56x512 54.6 / 54.3, and 24x40x128 batch 256 (three chunks) 21.0 / 16.2: a line
  // at more chunks that this rule does not draw.
  const int stream_csd = (2 * DWS_ROWS * (W / 4)) | 1;
  const size_t stream_lds = 4 * ((size_t)DW_CG * stream_csd + 8 * (size_t)(Wo / 4));
  const bool stream = lin && Wo / 4 <= 16 - DWS_LOADERS && stream_lds <= 64 * 1024 && DWS_ROWS * W <= 1024 &&
                      (sx == 2 || H % DWS_ROWS == 0) &&
                      (long long)g_batch * (CH / DW_CG) >= 2ll * num_cus();
  if (hwc_in && !plane && !rowsk)
    return set_error(PULP_NN_HIP_ERR_UNSUPPORTED, fn, "no fused kernel for this geometry: use pulp_nn_hip_hwc_to_chw and the CHW entry point");
  // HWC rows of 16, 32 or 64 pixels: on the matrix cores where the channels are whole tiles, the maps 16-byte aligned and the layer not one
  // of the large ones that dwh_wide names.  (16-pixel rows at stride 2 and 8 x 8 and 4 x 4 planes stay in registers: 4.4 and 3.1-3.9 us
  // at batch 256, of which 3 are the launch.)
  if (hwc_in && rowsk) {
    const DwLayer L = {in, wt, bias, out, (int)g_batch, CH, H, W, Ho, Wo, kx, ky, pt, pl, sx, sy};
    if (launch_dw_hwc(mode, L, e, num_cus(), g_stream)) return check_launch(fn);
  }
  // Small layers on the matrix cores: up to 2 MB of input and 64 units of an image's 64 channels, where dw3x3_lin_kernel has a long chain of
  // rows on few workgroups and dw_mfma_kernel splits them (bands / matrix cores: 63x8x64 batch 2 15.1 / 4.5 us, 11x40x64 batch 2 6.7 / 4.3, 51x12x512
  // batch 5 10.8 / 5.5, 18x28x64 batch 56 6.5 / 4.9; past the line 9x8x64 stride 2 batch 248 5.0 / 8.0, 9x36x64 batch 195 6.3 / 7.5, 23x8x384 batch 73
  // 8.8 / 11.4; stride 2 on rows of 40 pixels and more 12x40x64 batch 4 4.8 / 5.3, 61x40x64 batch 14 5.4 / 5.9).
  if (lin && !stream && (long long)g_batch * CH * H * W <= 2 << 20 && (long long)g_batch * (CH / DW_CG) <= 64 && !(sx == 2 && W >= 40)) {
    const DwLayer L = {in, wt, bias, out, (int)g_batch, CH, H, W, Ho, Wo, kx, ky, pt, pl, sx, sy};
    if (launch_dw_mfma(mode, L, e, num_cus(), g_stream)) return check_launch(fn);
  }
  if (plane) {
    const dim3 pgrid((unsigned)(((long long)g.B * g.cgroups + DW_REG_WAVES - 1) / DW_REG_WAVES)), pblock(64 * DW_REG_WAVES);
#define DWP_LAYOUT(HW, S, HWC)                                                                                            \
  switch (mode) {                                                                                                         \
    case EPI_BN: hipLaunchKernelGGL((dw3x3_plane_kernel<HW, S, EPI_BN, HWC>), pgrid, pblock, 0, g_stream, g, e); break;     \
    case EPI_MULT: hipLaunchKernelGGL((dw3x3_plane_kernel<HW, S, EPI_MULT, HWC>), pgrid, pblock, 0, g_stream, g, e); break; \
    default: hipLaunchKernelGGL((dw3x3_plane_kernel<HW, S, EPI_RAW, HWC>), pgrid, pblock, 0, g_stream, g, e); break;        \
  }
#define DWP_MODE(HW, S)                      \
  if (hwc_in) { DWP_LAYOUT(HW, S, true) }    \
  else { DWP_LAYOUT(HW, S, false) }
    if (H == 8 && sx == 1) { DWP_MODE(8, 1) }
    else if (H == 8) { DWP_MODE(8, 2) }
    else { DWP_MODE(4, 1) }
#undef DWP_MODE
#undef DWP_LAYOUT
  } else if (rowsk) {
    const long long groups = (long long)g_batch * CH / DW_CG;
#define DWR_LAYOUT(WB, R, S, HWC)                                                                                                \
  {                                                                                                                              \
    const dim3 rgrid((unsigned)((groups * ((Ho + R - 1) / R) + DW_REG_WAVES - 1) / DW_REG_WAVES)), rblock(64 * DW_REG_WAVES);    \
    switch (mode) {                                                                                                              \
      case EPI_BN: hipLaunchKernelGGL((dw3x3_rows_kernel<WB, R, S, EPI_BN, HWC>), rgrid, rblock, 0, g_stream, g, e); break;      \
      case EPI_MULT: hipLaunchKernelGGL((dw3x3_rows_kernel<WB, R, S, EPI_MULT, HWC>), rgrid, rblock, 0, g_stream, g, e); break;  \
      default: hipLaunchKernelGGL((dw3x3_rows_kernel<WB, R, S, EPI_RAW, HWC>), rgrid, rblock, 0, g_stream, g, e); break;         \
    }                                                                                                                            \
  }
#define DWR_MODE(WB, R, S)                       \
  {                                              \
    if (hwc_in) DWR_LAYOUT(WB, R, S, true)       \
    else DWR_LAYOUT(WB, R, S, false)             \
  }
    if (W == 16 && sx == 1) DWR_MODE(16, 8, 1)
    else if (W == 16) DWR_MODE(16, 4, 2)
    else if (W == 32 && sx == 1) DWR_MODE(32, 4, 1)
    else if (W == 32) DWR_MODE(32, 4, 2)
    else if (sx == 1) DWR_MODE(64, 2, 1)
    else DWR_MODE(64, 2, 2)
#undef DWR_MODE
#undef DWR_LAYOUT
  } else if (stream) {
    // whole planes streamed through LDS by loader waves, one workgroup per image and 64 channels
    g.NR = DWS_ROWS;
    g.RB = 2;
    g.CSD = stream_csd;
    g.bands = 1;
    g.total = (int)((long long)g.B * g.cgroups);
    const dim3 sgrid(g.total), sblock(64 * (Wo / 4 + DWS_LOADERS));
#define DWS_MODE(S, PL)                                                                                                  \
  switch (mode) {                                                                                                        \
    case EPI_BN: hipLaunchKernelGGL((dw3x3_stream_kernel<S, PL, EPI_BN>), sgrid, sblock, stream_lds, g_stream, g, e); break;     \
    case EPI_MULT: hipLaunchKernelGGL((dw3x3_stream_kernel<S, PL, EPI_MULT>), sgrid, sblock, stream_lds, g_stream, g, e); break; \
    default: hipLaunchKernelGGL((dw3x3_stream_kernel<S, PL, EPI_RAW>), sgrid, sblock, stream_lds, g_stream, g, e); break;        \
  }
    if (sx == 1 && pl == 1) { DWS_MODE(1, 1) }
    else if (sx == 1) { DWS_MODE(1, 0) }
    else if (pl == 1) { DWS_MODE(2, 1) }
    else { DWS_MODE(2, 0) }
#undef DWS_MODE
  } else if (lin) {
    g.total = (int)((long long)g.B * g.bands * g.cgroups);
    const dim3 grid(g.total), block(64 * DW_WAVES);
#define DW3L(S, PL)                                                                                                           \
  switch (mode) {                                                                                                             \
    case EPI_BN: hipLaunchKernelGGL((dw3x3_lin_kernel<S, PL, EPI_BN>), grid, block, lin_lds, g_stream, g, e); break;     \
    case EPI_MULT: hipLaunchKernelGGL((dw3x3_lin_kernel<S, PL, EPI_MULT>), grid, block, lin_lds, g_stream, g, e); break; \
    default: hipLaunchKernelGGL((dw3x3_lin_kernel<S, PL, EPI_RAW>), grid, block, lin_lds, g_stream, g, e); break;        \
  }
    if (sx == 1 && pl == 1) { DW3L(1, 1) }
    else if (sx == 1) { DW3L(1, 0) }
    else if (pl == 1) { DW3L(2, 1) }
    else { DW3L(2, 0) }
#undef DW3L
  } else {
    // any other shape: on the matrix cores (filters up to 8 columns wide), or a byte loop
    g.LP = pl > 4 ? ((pl + 3) & ~3) : 4;
    // The widths this entry point takes: ky rows of 64 channels in 64 KiB, rows as windows of dwords read them.
    // (dw_mfma_kernel alone could do more; callers see one limit, whichever kernel a shape takes.)
    const int window = fast ? 4 * (g.LP / 4 - 1 + ((Wo + 3) / 4 - 1) * sx + (6 - pl + 3 * sx) / 4 + 1) : g.LP - pl + (Wo - 1) * sx + kx;
    const bool dword_rows = fast && W % 4 == 0 && W / 4 * 3 <= 255 && aligned(in, 16);
    if (!dword_rows && 255 / ((std::max(window, g.LP + W + 1) + 3) / 4) < ky)
      return set_error(PULP_NN_HIP_ERR_UNSUPPORTED, fn, "image too wide for the LDS tile");
    const DwLayer L = {in, wt, bias, out, (int)g_batch, CH, H, W, Ho, Wo, kx, ky, pt, pl, sx, sy};
    if (launch_dw_mfma(mode, L, e, num_cus(), g_stream)) return check_launch(fn);
    g.LWD = (std::max(g.LP - pl + (Wo - 1) * sx + kx, g.LP + W + 1) + 3) / 4;
    const int nr_max = 255 / g.LWD;  // 64 channels x 255 dwords = 63.75 KiB of LDS
    if (nr_max < ky) return set_error(PULP_NN_HIP_ERR_UNSUPPORTED, fn, "image too wide for the LDS tile");
    const int rb_max = std::min((nr_max - ky) / sy + 1, Ho);
    g.bands = (Ho + rb_max - 1) / rb_max;
    g.RB = (Ho + g.bands - 1) / g.bands;
    g.bands = (Ho + g.RB - 1) / g.RB;
    g.NR = (g.RB - 1) * sy + ky;
    g.CSD = (g.NR * g.LWD) | 1;
    const long long total = (long long)g.B * g.bands * g.cgroups;
    if (total > 0x7fffffffLL) return set_error(PULP_NN_HIP_ERR_ARGUMENT, fn, "batch too large");
    g.total = (int)total;
    g.inc_dw = 256 % g.LWD;
    const int carry = 256 / g.LWD;
    g.inc_row = carry % g.NR;
    g.inc_c = carry / g.NR;
    g.in_align4 = aligned(in, 4) && (W % 4 == 0);
    const size_t lds = (size_t)DW_CG * g.CSD * 4;
    const dim3 grid(g.total), block(256);
    switch (mode) {
      case EPI_BN: hipLaunchKernelGGL(dw_generic_kernel<EPI_BN>, grid, block, lds, g_stream, g, e); break;
      case EPI_MULT: hipLaunchKernelGGL(dw_generic_kernel<EPI_MULT>, grid, block, lds, g_stream, g, e); break;
      default: hipLaunchKernelGGL(dw_generic_kernel<EPI_RAW>, grid, block, lds, g_stream, g, e); break;
    }
  }
  check_launch(fn);
}
