// Depthwise + pointwise blocks as one launch: which shapes, and the launch (the tile's shape: dwpw_geom.h).
#include "host.h"

#include "dwpw16.h"
#include "dwpw_chain.h"

namespace {

template <int W, int S, int KP, bool CHAIN, bool LEAN = false>
bool launch_kp(const DwPwGeom &g)
{
  if (!raise_lds_limit<dwpw_kernel<W, S, KP, CHAIN, LEAN>>((size_t)g.t.lds)) return false;
  hipLaunchKernelGGL((dwpw_kernel<W, S, KP, CHAIN, LEAN>), dim3((unsigned)g.t.tiles << g.t.lsplit), dim3(64 * g.t.waves), (size_t)g.t.lds, g_stream, g);
  return true;
}
template <int W>
bool launch_chain(const DwPwGeom &g)
{
  const int lds = dwpw_chain_lds(g.t.lds, g.t.C);
  if (lds > 160 * 1024) return false;
  for (int j = 0; j < g.nblocks; j++)
    if (!aligned(g.blk[j].dw_wt, 4) || !aligned(g.blk[j].dw_bias, 4) || !aligned(g.blk[j].pw_bias, 4)) return false;
  if (!raise_lds_limit<dwpw_chain_kernel<W>>((size_t)lds)) return false;
  hipLaunchKernelGGL((dwpw_chain_kernel<W>), dim3((unsigned)g.t.tiles), dim3(1024), (size_t)lds, g_stream, g);
  return true;
}
template <int W, int S, bool CHAIN>
bool launch(const DwPwGeom &g)
{
  if constexpr (CHAIN && W <= 16) {
    // every wave of sixteen at most one item of either stage (up to 256 channels, so the four slices of K that the kernel has in LDS; tiles of 64
    // channels or fewer have fewer waves)
    if (g.t.waves == 16 && g.t.kp == DWPW_CHAIN_KP && g.t.C / 16 * g.t.nst <= 16 && g.t.C / 16 << g.t.lpxb <= 16 && launch_chain<W>(g)) return true;
  }
  if constexpr (!CHAIN)  // (a chain has no eight slices: dwpw_tile)
    if (g.t.kp == 8) return launch_kp<W, S, 8, CHAIN>(g);
  if constexpr (!CHAIN && sizeof(bn_t) == 4)  // (with 64 bits every kernel of a single block is as lean)
    if (g.t.kp == 4 && dwpw_lean(g.t, num_cus())) return launch_kp<W, S, 4, CHAIN, true>(g);
  return g.t.kp == 1 ? launch_kp<W, S, 1, CHAIN>(g) : launch_kp<W, S, 4, CHAIN>(g);
}
template <bool CHAIN>
bool launch_s1(int W, const DwPwGeom &g)
{
  if constexpr (!CHAIN)
    if (W == 64) return launch<64, 1, CHAIN>(g);
  return W == 32 ? launch<32, 1, CHAIN>(g) : W == 16 ? launch<16, 1, CHAIN>(g) : W == 8 ? launch<8, 1, CHAIN>(g) : launch<4, 1, CHAIN>(g);
}
bool launch_s2(int W, const DwPwGeom &g)
{
  return W == 64 ? launch<64, 2, false>(g) : W == 32 ? launch<32, 2, false>(g) : W == 16 ? launch<16, 2, false>(g) : launch<8, 2, false>(g);
}

// Few planes 16 pixels wide at stride 2 (the rule, and what it measured: dwpw_small16)
void launch16(const DwPwGeom &g, int B, int C, int H, int Ho, int Co, int cus)
{
  const int M = B * Ho * 8, tiles = (M + DWPW16_PX - 1) / DWPW16_PX, split = dwpw16_split(tiles, Co, cus);
  const DwPw16Geom t = {g.in, g.out, M, C, H, Ho, Co, split, fastdiv_make((unsigned)Ho), g.blk[0]};
  const size_t lds = (size_t)dwpw16_lds(C, Co, split, (int)sizeof(bn_t));
  const dim3 grid((unsigned)(tiles * split)), block(64 * DWPW16_WAVES);
  if (C == 128) hipLaunchKernelGGL(dwpw16_kernel<2>, grid, block, lds, g_stream, t);
  else hipLaunchKernelGGL(dwpw16_kernel<4>, grid, block, lds, g_stream, t);
}

}  // namespace

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
  const char *refusal = dwpw_refusal(g_batch, C, W, Ho, Wo, Co, S, n_blocks, num_cus(), (int)sizeof(bn_t));
  if (!refusal && !(aligned(Im_in, 4) && aligned(Im_out, 16) && w_aligned))
    refusal = "no fused kernel for this geometry: call the depthwise and the pointwise layer separately";
  if (refusal) return set_error(PULP_NN_HIP_ERR_UNSUPPORTED, fn, refusal);
  g.in = Im_in;
  g.out = Im_out;
  if (n_blocks == 1 && dwpw_small16(g_batch, C, W, Ho, Co, S, num_cus())) launch16(g, (int)g_batch, C, H, Ho, Co, num_cus());
  else if (!dwpw_shape((int)g_batch, C, H, W, Ho, Co, S, n_blocks > 1, num_cus(), (int)sizeof(bn_t), &g.t) ||
      !(n_blocks > 1 ? launch_s1<true>(W, g) : S == 1 ? launch_s1<false>(W, g) : launch_s2(W, g)))
    return set_error(PULP_NN_HIP_ERR_UNSUPPORTED, fn, "no fused kernel for this geometry: call the depthwise and the pointwise layer separately");
  check_launch(fn);
}
