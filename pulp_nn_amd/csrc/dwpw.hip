// Depthwise + pointwise blocks as one launch: tile shape and launch of dwpw_fused.h.
#include "host.h"

#include "dwpw_fused.h"

// Common part of pulp_nn_hip_dw_pw_hwc (one block) and pulp_nn_hip_dw_pw_chain_hwc (several).
void dwpw_common(const char *fn, const unsigned char *Im_in, unsigned char *Im_out, int W, int H, int C, int Wo_arg,
                        int Ho_arg, int Co, int S, unsigned n_blocks, const pulp_nn_hip_block *blocks)
{
  REQUIRE(Im_in && Im_out && blocks && n_blocks >= 1, PULP_NN_HIP_ERR_ARGUMENT, "null activation pointer or no block");
  REQUIRE(n_blocks <= DWPW_MAX_BLOCKS, PULP_NN_HIP_ERR_ARGUMENT, "too many blocks for one launch");
  REQUIRE(W && H && C && Co && (S == 1 || S == 2), PULP_NN_HIP_ERR_ARGUMENT, "zero dimension or stride other than 1 or 2");
  const int Wo = (W - 1) / S + 1, Ho = (H - 1) / S + 1;
  REQUIRE(Wo_arg == Wo && Ho_arg == Ho, PULP_NN_HIP_ERR_ARGUMENT, "output size is not that of a 3x3 window with padding 1");
  DwPwGeom g;
  g.nblocks = (int)n_blocks;
  bool w_aligned = true;
  for (unsigned j = 0; j < n_blocks; j++) {
    const pulp_nn_hip_block &b = blocks[j];
    REQUIRE(b.dw_wt && b.pw_weight, PULP_NN_HIP_ERR_ARGUMENT, "null weight pointer");
    DwPwBlock &P = g.blk[j];
    P.dw_wt = (const int8_t *)b.dw_wt;
    P.dw_bias = (const int8_t *)b.dw_bias;
    P.pw_w = (const int8_t *)b.pw_weight;
    P.pw_bias = (const int8_t *)b.pw_bias;
    P.mode_dw = epi_mode(b.dw_flag_relu, b.dw_flag_batch_norm, true);  // pulp_nn_depthwise_generic.c:167-178 tests FLAG_RELU for truth
    P.mode_pw = epi_mode(b.pw_flag_relu, b.pw_flag_batch_norm);
    REQUIRE(epi_args(P.mode_dw, (bn_t *)b.dw_k, (bn_t *)b.dw_lambda, b.dw_out_mult, b.dw_out_shift, &P.e_dw) &&
                epi_args(P.mode_pw, (bn_t *)b.pw_k, (bn_t *)b.pw_lambda, b.pw_out_mult, b.pw_out_shift, &P.e_pw),
            PULP_NN_HIP_ERR_ARGUMENT, "out_shift out of range or null k/lambda");
    w_aligned = w_aligned && aligned(b.pw_weight, 16);
  }
  // per input width and stride: output rows of a stage-1 item, waves per workgroup, pixels / 16 of a stage-2 block
  int R = 0, NWV = 4, TMB = 2;
  if (W == 64) R = 2;
  else if (W == 32) R = 4;
  else if (W == 16) { R = S == 1 ? 4 : 2; NWV = 8; TMB = 2; }
  else if (W == 8) { R = S == 1 ? 4 : 2; NWV = 8; TMB = 2; }
  else if (W == 4 && S == 1) { R = 4; NWV = 8; TMB = 2; }
  const bool c_ok = (C == 16 || C == 32 || (C % 64 == 0 && C <= 1024));
  const int LG = C >= 64 ? 1 : 64 / C, CGN = C >= 64 ? C / 64 : 1;
  const long long M = (long long)g_batch * Ho * Wo;
  const bool ok = R > 0 && c_ok && Ho % (R * LG) == 0 && Co % 16 == 0 && aligned(Im_in, 4) && aligned(Im_out, 16) &&
                  w_aligned && M <= 0x7fffffffLL && (long long)Co * C < 0x7fffffffLL;
  if (!ok)
    return set_error(PULP_NN_HIP_ERR_UNSUPPORTED, fn, "no fused kernel for this geometry: call the depthwise and the pointwise layer separately");
  g.in = Im_in;
  g.out = Im_out;
  g.B = (int)g_batch;
  g.C = C;
  g.H = H;
  g.Ho = Ho;
  g.Co = Co;
  g.M = (int)M;
  g.KT = (C + 63) / 64;
  g.d_howo = fastdiv_make((unsigned)(Ho * Wo));
  // a tile: enough stage-1 items (item_px pixels x 64 channels each) to give every wave one, in whole stage-2 blocks
  const int item_px = R * LG * Wo, bp = 16 * TMB;
  int segs = (NWV + CGN - 1) / CGN;                       // items along the pixels
  while ((segs * item_px) % bp) segs++;
  while (segs > 1 && (dwpw_lds_bytes(segs * item_px, C) > 49152 || (M + (long long)segs * item_px - 1) / (segs * item_px) < num_cus()))
    segs--;
  while ((segs * item_px) % bp) segs++;
  g.BM = segs * item_px;
  int tiles = (int)((M + g.BM - 1) / g.BM);
  const int nbt = (Co + 63) / 64;
  // few pixel tiles: several workgroups share one, each with a part of the output channels (and its own copy of stage 1)
  g.nsplit = 1;
  while (tiles * g.nsplit < num_cus() && g.nsplit * 2 <= nbt) g.nsplit *= 2;
  // (the kernel stages the pointwise constants of at most 1024 channels per workgroup)
  if (((nbt + g.nsplit - 1) / g.nsplit) * 64 > 1024)
    return set_error(PULP_NN_HIP_ERR_UNSUPPORTED, fn, "more than 1024 output channels per workgroup: call the depthwise and the pointwise layer separately");
  size_t lds = (size_t)dwpw_lds_bytes(g.BM, C) + (size_t)dwpw_const_bytes(((nbt + g.nsplit - 1) / g.nsplit) * 64);
  if (n_blocks > 1) {
    // Several blocks: the output of one is the next one's input and stays in LDS, so a tile has to be whole images
    // (the 3x3 window of a pixel then never leaves the tile), the blocks have to keep the shape (stride 1, as many
    // channels out as in), and a workgroup computes all channels.
    const int img_px = Ho * Wo;
    int per_tile = (g.BM + img_px - 1) / img_px;  // images per tile
    while ((per_tile * img_px) % bp || (per_tile * img_px) % item_px) per_tile++;
    g.BM = per_tile * img_px;
    tiles = (int)((M + g.BM - 1) / g.BM);
    g.nsplit = 1;
    lds = (size_t)dwpw_lds_bytes(g.BM, C) + (size_t)dwpw_const_bytes(nbt * 64) + (size_t)g.BM * (Co + DWPW_YPAD);
    if (S != 1 || C != Co || g_batch % (unsigned)per_tile != 0)
      return set_error(PULP_NN_HIP_ERR_UNSUPPORTED, fn, "blocks can only be chained at stride 1 with as many channels out as in, on whole images per tile");
  }
  if (lds > 65536)
    return set_error(PULP_NN_HIP_ERR_UNSUPPORTED, fn, "no fused kernel for this geometry: call the depthwise and the pointwise layer separately");
  const dim3 grid((unsigned)(tiles * g.nsplit)), block(64 * NWV);
#define DWPW_KP(WB, RR, SS, NW, TM)                                                                    \
  if (g.KT == 1) hipLaunchKernelGGL((dwpw_fused_kernel<WB, RR, SS, NW, TM, 1>), grid, block, lds, g_stream, g);      \
  else if (g.KT == 2) hipLaunchKernelGGL((dwpw_fused_kernel<WB, RR, SS, NW, TM, 2>), grid, block, lds, g_stream, g); \
  else hipLaunchKernelGGL((dwpw_fused_kernel<WB, RR, SS, NW, TM, 4>), grid, block, lds, g_stream, g);
#define DWPW_CHAIN_KP(WB, RR, NW, TM, NT)                                                                                     \
  if (g.KT == 1) hipLaunchKernelGGL((dwpw_fused_kernel<WB, RR, 1, NW, TM, 1, true, NT>), grid, block, lds, g_stream, g);      \
  else if (g.KT == 2) hipLaunchKernelGGL((dwpw_fused_kernel<WB, RR, 1, NW, TM, 2, true, NT>), grid, block, lds, g_stream, g); \
  else hipLaunchKernelGGL((dwpw_fused_kernel<WB, RR, 1, NW, TM, 4, true, NT>), grid, block, lds, g_stream, g);
  // Stage-2 blocks of 64 pixels x 32 channels instead of 32 x 64: each weight fragment then goes to one wave of the tile,
  // not to two.  Chains of width 8 take it (part of what brought five blocks of 8x8x256 from 48 to 36 us, see
  // dwpw_fused.h).  Width 4 makes no difference (five blocks of 4x4x256 28.3 / 28.3 us, two of
  // 4x4x64 8.6 / 8.6).  Single blocks, which do not take it, would gain at widths 8 and 16 where a tile is 64 pixels (32 x 64 /
  // 64 x 32, batch 256: 16x16x256 33.3 / 23.2 us, 16x16x128 14.3 / 12.6, 8x8x256 11.0 / 9.3, 16x16x128 -> 256 stride 2 8.8 / 8.0)
  // and lose nowhere measured.
  const bool wide_px = g.BM % 64 == 0 && C >= 64;
  if (n_blocks > 1) {
    // (stride 1 only; the widest planes never fit the LDS of a chained launch)
    if (W == 32) { DWPW_CHAIN_KP(32, 4, 4, 2, 4) }
    else if (W == 16) { DWPW_CHAIN_KP(16, 4, 8, 2, 4) }
    else if (W == 8 && wide_px) { DWPW_CHAIN_KP(8, 4, 8, 4, 2) }
    else if (W == 8) { DWPW_CHAIN_KP(8, 4, 8, 2, 4) }
    else if (W == 4) { DWPW_CHAIN_KP(4, 4, 8, 2, 4) }
    else return set_error(PULP_NN_HIP_ERR_UNSUPPORTED, fn, "blocks of this width cannot be chained");
    check_launch(fn);
    return;
  }
  if (W == 64 && S == 1) { DWPW_KP(64, 2, 1, 4, 2) }
  else if (W == 64) { DWPW_KP(64, 2, 2, 4, 2) }
  else if (W == 32 && S == 1) { DWPW_KP(32, 4, 1, 4, 2) }
  else if (W == 32) { DWPW_KP(32, 4, 2, 4, 2) }
  else if (W == 16 && S == 1) { DWPW_KP(16, 4, 1, 8, 2) }
  else if (W == 16) { DWPW_KP(16, 2, 2, 8, 2) }
  else if (W == 8 && S == 1) { DWPW_KP(8, 4, 1, 8, 2) }
  else if (W == 8) { DWPW_KP(8, 2, 2, 8, 2) }
  else { DWPW_KP(4, 4, 1, 8, 2) }
#undef DWPW_KP
#undef DWPW_CHAIN_KP
  check_launch(fn);
}

