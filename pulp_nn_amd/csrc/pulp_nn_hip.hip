// C-ABI host layer: the PULP-NN layer functions on MI355X.
//
// Built twice: -DPULPNN_BN_BITS=32 -> libpulpnn_hip32.so, =64 -> libpulpnn_hip64.so,
// mirroring the reference's 32bit/ and 64bit/ trees (same symbol names, k / lambda
// typed int32_t or int64_t).  Each function validates its arguments, picks a
// kernel variant and queues it; nothing is allocated and no state is kept
// besides the per-thread batch count, stream and last error.
#include "host.h"

#include <stdio.h>

#include "calib.h"
#include "layout.h"
#include "pool.h"

__thread unsigned g_batch = 1;
__thread hipStream_t g_stream = nullptr;
static __thread int g_err = PULP_NN_HIP_OK;
static __thread char g_errmsg[256] = "";

void set_error(int code, const char *fn, const char *msg)
{
  g_err = code;
  snprintf(g_errmsg, sizeof g_errmsg, "%s: %s", fn, msg);
}

void check_launch(const char *fn)
{
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) set_error(PULP_NN_HIP_ERR_RUNTIME, fn, hipGetErrorString(e));
}

bool epi_args(int mode, const bn_t *k, const bn_t *lambda, uint16_t out_mult, int out_shift_param, EpiArgs *e)
{
  e->k = k;
  e->lambda = lambda;
  e->mult = (int)(int16_t)out_mult;
  if (mode == EPI_RAW) {
    e->shift = out_shift_param;  // used as written: sum >> out_shift
    return e->shift >= 0 && e->shift < 32;
  }
  e->shift = (int)(int8_t)out_shift_param;  // the quantiser functions take int8_t
  const int lim = (mode == EPI_BN) ? PULPNN_BN_BITS : 32;
  if (mode == EPI_BN && (!k || !lambda)) return false;
  return e->shift >= 0 && e->shift < lim;
}

// Cached per process; concurrent first calls compute the same value, so a relaxed atomic is enough.
int num_cus()
{
  static std::atomic<int> cached{0};
  int n = cached.load(std::memory_order_relaxed);
  if (!n) {
    int dev = 0;
    hipDeviceProp_t p;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&p, dev) == hipSuccess) n = p.multiProcessorCount;
    if (n <= 0) n = 256;
    cached.store(n, std::memory_order_relaxed);
  }
  return n;
}

namespace {

template <int BW, int BH>
void launch_maxpool16(const PoolGeom &g, bool nt, bool lnt)
{
  const dim3 grid((unsigned)((g.total + 255) / 256)), block(256);
  if (nt && lnt) hipLaunchKernelGGL((maxpool16_kernel<true, true, BW, BH>), grid, block, 0, g_stream, g);
  else if (nt) hipLaunchKernelGGL((maxpool16_kernel<true, false, BW, BH>), grid, block, 0, g_stream, g);
  else if (lnt) hipLaunchKernelGGL((maxpool16_kernel<false, true, BW, BH>), grid, block, 0, g_stream, g);
  else hipLaunchKernelGGL((maxpool16_kernel<false, false, BW, BH>), grid, block, 0, g_stream, g);
}
template <int BW, int BH>
void launch_avgpool(const PoolGeom &g, const AvgArgs &a)
{
  hipLaunchKernelGGL((avgpool_kernel<BW, BH>), dim3((unsigned)((g.total + 255) / 256)), dim3(256), 0, g_stream, g, a);
}

bool pool_geom(const char *fn, PoolGeom *g, uint8_t *in, uint8_t *out, uint16_t W, uint16_t H, uint16_t C,
               uint16_t Wo, uint16_t Ho, uint16_t kx, uint16_t ky, uint16_t pt, uint16_t pb, uint16_t pl,
               uint16_t pr, uint16_t sx, uint16_t sy)
{
  if (!in || !out) { set_error(PULP_NN_HIP_ERR_ARGUMENT, fn, "null pointer"); return false; }
  if (!W || !H || !C || !Wo || !Ho || !kx || !ky || !sx || !sy) {
    set_error(PULP_NN_HIP_ERR_ARGUMENT, fn, "zero dimension");
    return false;
  }
  g->in = in;
  g->out = out;
  g->B = (int)g_batch;
  g->H = H;
  g->W = W;
  g->C = C;
  g->Ho = Ho;
  g->Wo = Wo;
  g->kx = kx;
  g->ky = ky;
  g->sx = sx;
  g->sy = sy;
  g->pt = pt;
  g->pb = pb;
  g->pl = pl;
  g->pr = pr;
  g->cgroups = (C + 3) / 4;
  g->vec4 = (C % 4 == 0) && aligned(in, 4) && aligned(out, 4);
  pool_threads(g);
  if ((g->total + 255) / 256 > 0x7fffffffLL) {
    set_error(PULP_NN_HIP_ERR_ARGUMENT, fn, "batch too large");
    return false;
  }
  return true;
}

// ---- calibration ---------------------------------------------------------------------

// Device memory of the allocation-free calibration entry point: one partial maximum per
// workgroup.  In host code the array's name only stands for the symbol; its device address
// comes from hipGetSymbolAddress, once per device (every GPU holds its own copy).
#define CALIB_STATIC_SLOTS 8192
static __device__ __align__(256) unsigned long long scratch[CALIB_STATIC_SLOTS];

unsigned long long *static_scratch(const char *fn)
{
  constexpr int MAX_DEV = 64;
  static std::mutex mu;
  static unsigned long long *ptr[MAX_DEV] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEV) {
    set_error(PULP_NN_HIP_ERR_RUNTIME, fn, "cannot identify the current device");
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(mu);
  if (!ptr[dev]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      set_error(PULP_NN_HIP_ERR_RUNTIME, fn, hipGetErrorString(e));
      return nullptr;
    }
    ptr[dev] = (unsigned long long *)p;
  }
  return ptr[dev];
}

// Shared body of the calibration entry points.  partial: device memory for `slots_avail` partial maxima.
void calib_common(const char *fn, CalibGeom &g, unsigned long long *partial, unsigned long long slots_avail,
                  unsigned long long *result)
{
  if (!g.in || !g.w || !g.k || !result) return set_error(PULP_NN_HIP_ERR_ARGUMENT, fn, "null pointer");
  if (g.W <= 0 || g.H <= 0 || g.Ci <= 0 || g.Wo <= 0 || g.Ho <= 0 || g.Co <= 0 || g.kx <= 0 || g.ky <= 0 || g.sx <= 0 ||
      g.sy <= 0)
    return set_error(PULP_NN_HIP_ERR_ARGUMENT, fn, "zero dimension");
  // batch * Ho * Wo * Co can pass 2^63 (batch up to 2^31, the dimensions up to 2^16 each): bound it before it is formed
  const unsigned long long per_image = (unsigned long long)g.Ho * g.Wo * g.Co;  // < 2^48
  if ((unsigned long long)g_batch > (1ull << 47) / per_image) return set_error(PULP_NN_HIP_ERR_ARGUMENT, fn, "batch too large");
  g.total = (long long)((unsigned long long)g_batch * per_image);
  g.in_img = (long long)g.H * g.W * g.Ci;
  const unsigned long long slots = ((unsigned long long)g.total + CALIB_CHUNK - 1) / CALIB_CHUNK;
  if (slots > 0x7fffffffull) return set_error(PULP_NN_HIP_ERR_ARGUMENT, fn, "batch too large");
  if (!partial || slots > slots_avail)
    return set_error(PULP_NN_HIP_ERR_ARGUMENT, fn,
                     "layer too large for the partial-maximum buffer (one 8-byte slot per 65536 outputs)");
  hipLaunchKernelGGL(calib_absmax_kernel, dim3((unsigned)slots), dim3(256), 0, g_stream, g, partial);
  hipLaunchKernelGGL(calib_final_kernel, dim3(1), dim3(256), 0, g_stream, partial, (int)slots, result);
  check_launch(fn);
}

CalibGeom calib_conv_geom(const unsigned char *in, const signed char *bias, const signed char *w, const void *k,
                          unsigned short dim_in_x, unsigned short dim_in_y, unsigned short ch_in,
                          unsigned short dim_out_x, unsigned short dim_out_y, unsigned short ch_out,
                          unsigned short kx, unsigned short ky, unsigned short pt, unsigned short pl,
                          unsigned short sx, unsigned short sy)
{
  CalibGeom g = {};
  g.in = in;
  g.w = (const int8_t *)w;
  g.bias = (const int8_t *)bias;
  g.k = (const bn_t *)k;
  g.H = dim_in_y;
  g.W = dim_in_x;
  g.Ci = ch_in;
  g.Ho = dim_out_y;
  g.Wo = dim_out_x;
  g.Co = ch_out;
  g.kx = kx;
  g.ky = ky;
  g.pt = pt;
  g.pl = pl;
  g.sx = sx;
  g.sy = sy;
  return g;
}

}  // namespace

// ---- added entry points -----------------------------------------------------------

// Shader clock right now: cycles of the shader counter against ticks of the 100 MHz wall clock, over 20 us of one
// wave (pulp_nn_hip_clock_probe).
__global__ void clock_probe_kernel(long long *out)
{
  const long long t0 = wall_clock64(), c0 = __builtin_readcyclecounter();
  long long t1 = t0;
  while (t1 - t0 < 2000) t1 = wall_clock64();
  const long long c1 = __builtin_readcyclecounter();
  if (threadIdx.x == 0) {
    out[0] = t1 - t0;
    out[1] = c1 - c0;
  }
}

extern "C" {

void pulp_nn_hip_set_batch(unsigned n_images)
{
  if (n_images > 0x7fffffffu) return set_error(PULP_NN_HIP_ERR_ARGUMENT, __func__, "batch too large");
  g_batch = n_images ? n_images : 1;
}
unsigned pulp_nn_hip_get_batch(void) { return g_batch; }
void pulp_nn_hip_set_stream(void *hip_stream) { g_stream = (hipStream_t)hip_stream; }
void *pulp_nn_hip_get_stream(void) { return (void *)g_stream; }

int pulp_nn_hip_sync(void)
{
  hipError_t e = hipStreamSynchronize(g_stream);
  if (e != hipSuccess) {
    set_error(PULP_NN_HIP_ERR_RUNTIME, __func__, hipGetErrorString(e));
    return PULP_NN_HIP_ERR_RUNTIME;
  }
  return PULP_NN_HIP_OK;
}

void pulp_nn_hip_clock_probe(long long *out)
{
  REQUIRE(out && aligned(out, 8), PULP_NN_HIP_ERR_ARGUMENT, "null or misaligned pointer");
  hipLaunchKernelGGL(clock_probe_kernel, dim3(1), dim3(64), 0, g_stream, out);
  check_launch(__func__);
}

int pulp_nn_hip_last_error(void) { return g_err; }
const char *pulp_nn_hip_last_error_string(void) { return g_errmsg; }
void pulp_nn_hip_clear_error(void)
{
  g_err = PULP_NN_HIP_OK;
  g_errmsg[0] = 0;
}
int pulp_nn_hip_bn_bits(void) { return PULPNN_BN_BITS; }

void pulp_nn_hip_hwc_to_chw(const unsigned char *in_hwc, unsigned char *out_chw, unsigned dim_x, unsigned dim_y,
                            unsigned ch, unsigned pad_top, unsigned pad_bottom)
{
  REQUIRE(in_hwc && out_chw, PULP_NN_HIP_ERR_ARGUMENT, "null pointer");
  REQUIRE(dim_x && dim_y && ch, PULP_NN_HIP_ERR_ARGUMENT, "zero dimension");
  const unsigned hw = dim_x * dim_y, plane = (pad_top + dim_y + pad_bottom) * dim_x;
  if (ch % 16 == 0 && hw % 4 == 0 && plane % 4 == 0 && (pad_top * dim_x) % 4 == 0 && aligned(in_hwc, 16) &&
      aligned(out_chw, 4)) {
    const int tiles_p = (int)((hw + 255) / 256), tiles_c = (int)((ch + 63) / 64);
    const long long total = (long long)g_batch * tiles_p * tiles_c;
    REQUIRE(total <= 0x7fffffffLL, PULP_NN_HIP_ERR_ARGUMENT, "batch too large");
    if ((long long)g_batch * hw * ch >= PULPNN_NT_BYTES)
      hipLaunchKernelGGL(hwc_to_chw_fast_kernel<true>, dim3((unsigned)total), dim3(256), 0, g_stream, in_hwc, out_chw,
                         (int)dim_y, (int)dim_x, (int)ch, (int)pad_top, (int)pad_bottom, tiles_p, tiles_c);
    else
      hipLaunchKernelGGL(hwc_to_chw_fast_kernel<false>, dim3((unsigned)total), dim3(256), 0, g_stream, in_hwc, out_chw,
                         (int)dim_y, (int)dim_x, (int)ch, (int)pad_top, (int)pad_bottom, tiles_p, tiles_c);
    check_launch(__func__);
    return;
  }
  const int tiles_p = (int)((dim_x * dim_y + 63) / 64), tiles_c = (int)((ch + 63) / 64);
  const long long total = (long long)g_batch * tiles_p * tiles_c;
  REQUIRE(total <= 0x7fffffffLL, PULP_NN_HIP_ERR_ARGUMENT, "batch too large");
  hipLaunchKernelGGL(hwc_to_chw_kernel, dim3((unsigned)total), dim3(256), 0, g_stream, in_hwc, out_chw, (int)dim_y,
                     (int)dim_x, (int)ch, (int)pad_top, (int)pad_bottom, tiles_p, tiles_c);
  check_launch(__func__);
}

unsigned long long pulp_nn_hip_calib_workspace_bytes(unsigned long long n_outputs)
{
  return ((n_outputs + CALIB_CHUNK - 1) / CALIB_CHUNK) * sizeof(unsigned long long);
}

void pulp_nn_hip_calib_conv(const unsigned char *pInBuffer, const signed char *bias, const signed char *pWeight,
                            const void *k, unsigned short dim_in_x, unsigned short dim_in_y, unsigned short ch_in,
                            unsigned short dim_out_x, unsigned short dim_out_y, unsigned short ch_out,
                            unsigned short dim_kernel_x, unsigned short dim_kernel_y, unsigned short padding_y_top,
                            unsigned short padding_x_left, unsigned short stride_x, unsigned short stride_y,
                            void *workspace, unsigned long long workspace_bytes, unsigned long long *result)
{
  CalibGeom g = calib_conv_geom(pInBuffer, bias, pWeight, k, dim_in_x, dim_in_y, ch_in, dim_out_x, dim_out_y, ch_out,
                                dim_kernel_x, dim_kernel_y, padding_y_top, padding_x_left, stride_x, stride_y);
  REQUIRE(aligned(workspace, 8) && aligned(result, 8), PULP_NN_HIP_ERR_ARGUMENT, "workspace and result must be 8-byte aligned");
  calib_common(__func__, g, (unsigned long long *)workspace, workspace_bytes / sizeof(unsigned long long), result);
}

void pulp_nn_hip_calib_conv_static(const unsigned char *pInBuffer, const signed char *bias, const signed char *pWeight,
                                   const void *k, unsigned short dim_in_x, unsigned short dim_in_y,
                                   unsigned short ch_in, unsigned short dim_out_x, unsigned short dim_out_y,
                                   unsigned short ch_out, unsigned short dim_kernel_x, unsigned short dim_kernel_y,
                                   unsigned short padding_y_top, unsigned short padding_x_left,
                                   unsigned short stride_x, unsigned short stride_y, unsigned long long *result)
{
  CalibGeom g = calib_conv_geom(pInBuffer, bias, pWeight, k, dim_in_x, dim_in_y, ch_in, dim_out_x, dim_out_y, ch_out,
                                dim_kernel_x, dim_kernel_y, padding_y_top, padding_x_left, stride_x, stride_y);
  REQUIRE(aligned(result, 8), PULP_NN_HIP_ERR_ARGUMENT, "result must be 8-byte aligned");
  unsigned long long *partial = static_scratch(__func__);
  if (!partial) return;
  calib_common(__func__, g, partial, CALIB_STATIC_SLOTS, result);
}

void pulp_nn_hip_calib_depthwise(const unsigned char *Im_in, const signed char *bias, const signed char *wt,
                                 const void *k, unsigned short dim_im_in_x, unsigned short dim_im_in_y,
                                 unsigned short ch, unsigned short dim_im_out_x, unsigned short dim_im_out_y,
                                 unsigned short dim_kernel_x, unsigned short dim_kernel_y, unsigned short padding_y_top,
                                 unsigned short padding_x_left, unsigned short stride_x, unsigned short stride_y,
                                 int input_is_hwc, void *workspace, unsigned long long workspace_bytes,
                                 unsigned long long *result)
{
  CalibGeom g = calib_conv_geom(Im_in, bias, wt, k, dim_im_in_x, dim_im_in_y, ch, dim_im_out_x, dim_im_out_y, ch,
                                dim_kernel_x, dim_kernel_y, padding_y_top, padding_x_left, stride_x, stride_y);
  g.depthwise = 1;
  g.chw_in = !input_is_hwc;
  REQUIRE(aligned(workspace, 8) && aligned(result, 8), PULP_NN_HIP_ERR_ARGUMENT, "workspace and result must be 8-byte aligned");
  calib_common(__func__, g, (unsigned long long *)workspace, workspace_bytes / sizeof(unsigned long long), result);
}

// ---- the reference API ------------------------------------------------------------

#define CONV_FORWARD(NAME, POINTWISE)                                                                   \
  void NAME(PULP_NN_CONV_ARGS)                                                                          \
  {                                                                                                     \
    (void)pIm2ColBuffer;                                                                                \
    (void)padding_y_bottom;                                                                             \
    (void)padding_x_right;                                                                              \
    conv_common(#NAME, POINTWISE, pInBuffer, bias, pOutBuffer, pWeight, k, lambda, out_mult, out_shift, \
                dim_in_x, dim_in_y, ch_in, dim_out_x, dim_out_y, ch_out, dim_kernel_x, dim_kernel_y,    \
                padding_y_top, padding_x_left, stride_x, stride_y, flag_relu, flag_batch_norm);         \
  }

CONV_FORWARD(pulp_nn_conv_Ho_parallel, false)
CONV_FORWARD(pulp_nn_conv_Co_parallel, false)
CONV_FORWARD(pulp_nn_conv_HoWo_parallel, false)
CONV_FORWARD(pulp_nn_pointwise_HoWo_parallel, true)
CONV_FORWARD(pulp_nn_pointwise_Ho_parallel, true)
CONV_FORWARD(pulp_nn_pointwise_Co_parallel, true)

void pulp_nn_linear(uint8_t *pInBuffer, int8_t *bias, uint8_t *pOutBuffer, int8_t *pWeights, bn_t *k, bn_t *lambda,
                    uint16_t out_mult, int8_t out_shift, uint16_t dim_vec, uint16_t num_o_neurons, int flag_relu,
                    int flag_batch_norm)
{
  const int mode = epi_mode(flag_relu, flag_batch_norm);
  EpiArgs e;
  REQUIRE(epi_args(mode, k, lambda, out_mult, out_shift, &e), PULP_NN_HIP_ERR_ARGUMENT,
          "out_shift out of range or null k/lambda");
  linear_common(__func__, mode, pInBuffer, bias, pOutBuffer, pWeights, e, dim_vec, num_o_neurons, (int)g_batch);
}

void pulp_nn_linear_out_32(uint8_t *pInBuffer, int8_t *bias, int32_t *pOutBuffer, int8_t *pWeights, uint16_t dim_vec,
                           uint16_t num_o_neurons)
{
  REQUIRE(!bias || aligned(bias, 4), PULP_NN_HIP_ERR_ARGUMENT, "bias must be 4-byte aligned (it holds int32 values)");
  REQUIRE(aligned(pOutBuffer, 4), PULP_NN_HIP_ERR_ARGUMENT, "output must be 4-byte aligned");
  EpiArgs e = {nullptr, nullptr, 0, 0};
  linear_common(__func__, EPI_OUT32, pInBuffer, bias, pOutBuffer, pWeights, e, dim_vec, num_o_neurons, (int)g_batch);
}

uint8_t *pulp_nn_matmul(const int8_t *pWeight, uint8_t *pInBuffer, uint16_t ch_out, uint16_t num_col_im2col,
                        uint16_t out_shift, uint16_t out_mult, bn_t *k, bn_t *lambda, const int8_t *bias, uint8_t *pOut,
                        uint8_t *pOut2, int flag_relu, int flag_batch_norm)
{
  const int mode = epi_mode(flag_relu, flag_batch_norm);
  EpiArgs e;
  if (!epi_args(mode, k, lambda, out_mult, out_shift, &e)) {
    set_error(PULP_NN_HIP_ERR_ARGUMENT, __func__, "out_shift out of range or null k/lambda");
    return pOut;
  }
  if (!pOut || !pOut2) {
    set_error(PULP_NN_HIP_ERR_ARGUMENT, __func__, "null pointer");
    return pOut;
  }
  if (pOut2 == pOut + ch_out) {
    linear_common(__func__, mode, pInBuffer, bias, pOut, pWeight, e, num_col_im2col, ch_out, 2);
  } else {
    linear_common(__func__, mode, pInBuffer, bias, pOut, pWeight, e, num_col_im2col, ch_out, 1);
    linear_common(__func__, mode, pInBuffer + num_col_im2col, bias, pOut2, pWeight, e, num_col_im2col, ch_out, 1);
  }
  return pOut + 2 * (size_t)ch_out;
}

void pulp_nn_maxpool(uint8_t *Im_in, uint8_t *Im_out, uint16_t dim_im_in_x, uint16_t dim_im_in_y, uint16_t ch_im_in,
                     uint16_t dim_im_out_x, uint16_t dim_im_out_y, uint16_t dim_kernel_x, uint16_t dim_kernel_y,
                     uint16_t padding_t, uint16_t padding_b, uint16_t padding_l, uint16_t padding_r, uint16_t stride_x,
                     uint16_t stride_y)
{
  PoolGeom g;
  if (!pool_geom(__func__, &g, Im_in, Im_out, dim_im_in_x, dim_im_in_y, ch_im_in, dim_im_out_x, dim_im_out_y,
                 dim_kernel_x, dim_kernel_y, padding_t, padding_b, padding_l, padding_r, stride_x, stride_y))
    return;
  // The reference's in-place x pass re-reads columns it has already overwritten
  // when a window starts left of the column it is stored to, i.e. for some
  // i_x >= 1 with i_x*stride_x - padding_l < i_x (pulp_nn_maxpool.c:58-94).
  REQUIRE(padding_l == 0 || (int)stride_x - 1 >= (int)padding_l, PULP_NN_HIP_ERR_UNSUPPORTED,
          "left padding this large makes the reference's in-place x pass order dependent");
  if (ch_im_in % 16 == 0 && aligned(Im_in, 16) && aligned(Im_out, 16)) {
    g.cgroups = ch_im_in / 16;
    pool_threads(&g);
    // non-temporal loads: windows that do not overlap, on an input too large to find again in a cache
    const bool lnt = stride_x >= dim_kernel_x && stride_y >= dim_kernel_y &&
                     (long long)g.B * g.H * g.W * g.C >= PULPNN_NT_BYTES;
    const bool snt = g.total * 16 >= PULPNN_NT_BYTES;
    switch (pool_max_block(g.kx, g.ky)) {
      case PB_2x2: launch_maxpool16<2, 2>(g, snt, lnt); break;
      case PB_3x3: launch_maxpool16<3, 3>(g, snt, lnt); break;
      case PB_3x1: launch_maxpool16<3, 1>(g, snt, lnt); break;
      case PB_1x3: launch_maxpool16<1, 3>(g, snt, lnt); break;
      case PB_4x1: launch_maxpool16<4, 1>(g, snt, lnt); break;
      case PB_1x4: launch_maxpool16<1, 4>(g, snt, lnt); break;
      case PB_5x1: launch_maxpool16<5, 1>(g, snt, lnt); break;
    }
  } else {
    hipLaunchKernelGGL(maxpool_kernel, dim3((unsigned)((g.total + 255) / 256)), dim3(256), 0, g_stream, g);
  }
  check_launch(__func__);
}

void pulp_nn_avgpool(uint8_t *Im_in, uint8_t *Im_out, bn_t lambda, uint16_t out_shift, bn_t out_add,
                     uint16_t dim_im_in_x, uint16_t dim_im_in_y, uint16_t ch_im_in, uint16_t dim_im_out_x,
                     uint16_t dim_im_out_y, uint16_t dim_kernel_x, uint16_t dim_kernel_y, uint16_t padding_t,
                     uint16_t padding_b, uint16_t padding_l, uint16_t padding_r, uint16_t stride_x, uint16_t stride_y,
                     int flag_requant)
{
  PoolGeom g;
  if (!pool_geom(__func__, &g, Im_in, Im_out, dim_im_in_x, dim_im_in_y, ch_im_in, dim_im_out_x, dim_im_out_y,
                 dim_kernel_x, dim_kernel_y, padding_t, padding_b, padding_l, padding_r, stride_x, stride_y))
    return;
  REQUIRE(!flag_requant || out_shift < PULPNN_BN_BITS, PULP_NN_HIP_ERR_ARGUMENT, "out_shift out of range");
  REQUIRE((long long)dim_kernel_x * dim_kernel_y * 255 < 0xffffffffLL, PULP_NN_HIP_ERR_UNSUPPORTED, "window too large");
  AvgArgs a = {(long long)lambda, (long long)out_add, (int)out_shift, flag_requant, fastdiv_make((unsigned)dim_kernel_x * dim_kernel_y)};
  switch (pool_avg_block(g.kx, g.ky)) {
    case PB_1x1: launch_avgpool<1, 1>(g, a); break;
    case PB_2x1: launch_avgpool<2, 1>(g, a); break;
    case PB_1x2: launch_avgpool<1, 2>(g, a); break;
    case PB_2x2: launch_avgpool<2, 2>(g, a); break;
    case PB_3x1: launch_avgpool<3, 1>(g, a); break;
    case PB_1x3: launch_avgpool<1, 3>(g, a); break;
    case PB_3x3: launch_avgpool<3, 3>(g, a); break;
    case PB_4x1: launch_avgpool<4, 1>(g, a); break;
    case PB_1x4: launch_avgpool<1, 4>(g, a); break;
    case PB_5x1: launch_avgpool<5, 1>(g, a); break;
    case PB_5x3: launch_avgpool<5, 3>(g, a); break;
    case PB_4x4: launch_avgpool<4, 4>(g, a); break;
  }
  check_launch(__func__);
}

void pulp_nn_add(uint8_t *Im_in_1, uint8_t *Im_in_2, uint8_t *Im_out, uint16_t out_mult1, uint16_t out_mult2,
                 uint16_t out_shift, uint16_t dim_im_in_h, uint16_t dim_im_in_w, uint16_t ch_im_in)
{
  REQUIRE(Im_in_1 && Im_in_2 && Im_out, PULP_NN_HIP_ERR_ARGUMENT, "null pointer");
  REQUIRE(dim_im_in_h && dim_im_in_w && ch_im_in, PULP_NN_HIP_ERR_ARGUMENT, "zero dimension");
  const int d = (int)(int8_t)out_shift;  // pulp_nn_add_quant_u8 takes the shift as int8_t
  REQUIRE(d >= 0 && d < 32, PULP_NN_HIP_ERR_ARGUMENT, "out_shift out of range");
  const long long n = (long long)g_batch * dim_im_in_h * dim_im_in_w * ch_im_in;
  const long long threads = (n + 15) / 16;
  REQUIRE((threads + 255) / 256 <= 0x7fffffffLL, PULP_NN_HIP_ERR_ARGUMENT, "batch too large");
  const int vec16 = aligned(Im_in_1, 16) && aligned(Im_in_2, 16) && aligned(Im_out, 16);
  hipLaunchKernelGGL(add_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, g_stream, Im_in_1, Im_in_2,
                     Im_out, n, (int)(int16_t)out_mult1, (int)(int16_t)out_mult2, d, vec16);
  check_launch(__func__);
}

#define DW_FORWARD(NAME)                                                                                       \
  void NAME(PULP_NN_DW_ARGS)                                                                                   \
  {                                                                                                            \
    (void)bufferC;                                                                                             \
    (void)bufferB;                                                                                             \
    (void)ch_im_in;                                                                                            \
    (void)padding_y_bottom;                                                                                    \
    (void)padding_x_right;                                                                                     \
    depthwise_common(#NAME, Im_in, bias, Im_out, wt, k, lambda, out_mult, out_shift, dim_im_in_x, dim_im_in_y, \
                     dim_im_out_x, dim_im_out_y, ch_im_out, dim_kernel_x, dim_kernel_y, padding_y_top,         \
                     padding_x_left, stride_x, stride_y, epi_mode(FLAG_RELU, FLAG_BATCH_NORM, true));          \
  }

DW_FORWARD(pulp_nn_depthwise_generic)
DW_FORWARD(pulp_nn_depthwise_generic_less_4_weights)

void pulp_nn_hip_depthwise_hwc(const unsigned char *Im_in, const signed char *bias, unsigned char *Im_out,
                               const signed char *wt, void *k, void *lambda, unsigned short out_mult,
                               unsigned short out_shift, unsigned short dim_im_in_x, unsigned short dim_im_in_y,
                               unsigned short ch, unsigned short dim_im_out_x, unsigned short dim_im_out_y,
                               unsigned short stride, signed char flag_relu, signed char flag_batch_norm)
{
  depthwise_common(__func__, Im_in, (const int8_t *)bias, Im_out, (const int8_t *)wt, (bn_t *)k, (bn_t *)lambda, out_mult,
                   out_shift, dim_im_in_x, dim_im_in_y, dim_im_out_x, dim_im_out_y, ch, 3, 3, 1, 1, stride, stride,
                   epi_mode(flag_relu, flag_batch_norm, true), true);
}

void pulp_nn_hip_dw_pw_hwc(const unsigned char *Im_in, unsigned char *Im_out, unsigned short dim_im_in_x,
                           unsigned short dim_im_in_y, unsigned short ch, unsigned short dim_im_out_x,
                           unsigned short dim_im_out_y, unsigned short ch_out, unsigned short stride,
                           const signed char *dw_wt, const signed char *dw_bias, void *dw_k, void *dw_lambda,
                           unsigned short dw_out_mult, unsigned short dw_out_shift, signed char dw_flag_relu,
                           signed char dw_flag_batch_norm, const signed char *pw_weight, const signed char *pw_bias,
                           void *pw_k, void *pw_lambda, unsigned short pw_out_mult, unsigned short pw_out_shift,
                           signed char pw_flag_relu, signed char pw_flag_batch_norm)
{
  const pulp_nn_hip_block b = {dw_wt,     dw_bias,   dw_k,        dw_lambda,    dw_out_mult,  dw_out_shift, dw_flag_relu, dw_flag_batch_norm,
                               pw_weight, pw_bias,   pw_k,        pw_lambda,    pw_out_mult,  pw_out_shift, pw_flag_relu, pw_flag_batch_norm};
  dwpw_common(__func__, Im_in, Im_out, dim_im_in_x, dim_im_in_y, ch, dim_im_out_x, dim_im_out_y, ch_out, stride, 1, &b);
}

void pulp_nn_hip_dw_pw_chain_hwc(const unsigned char *Im_in, unsigned char *Im_out, unsigned short dim_im_x,
                                 unsigned short dim_im_y, unsigned short ch, unsigned n_blocks,
                                 const pulp_nn_hip_block *blocks)
{
  dwpw_common(__func__, Im_in, Im_out, dim_im_x, dim_im_y, ch, dim_im_x, dim_im_y, ch, 1, n_blocks, blocks);
}

void pulp_nn_depthwise_3x3_s1(uint8_t *In_Img, uint8_t *Out_Img, int R, int C, int CH, int p_l, int p_r,
                              int8_t *Kernel, int8_t out_shift, uint16_t out_mult, bn_t *kappa, bn_t *lambda,
                              int flag_relu, int flag_batch_norm, unsigned int *memory_chan)
{
  (void)memory_chan;
  REQUIRE(R >= 3 && C >= 2 && CH >= 1, PULP_NN_HIP_ERR_ARGUMENT, "plane too small");
  REQUIRE(R <= 65535 + 2 && C <= 65535 && CH <= 65535, PULP_NN_HIP_ERR_ARGUMENT, "dimension too large");
  // Only for p_l = p_r = 1 and even C do the reference's three row pointers land on
  // the start of the next row after each output row (pulp_nn_depthwise_3x3_s1.c:141-223).
  REQUIRE(p_l == 1 && p_r == 1 && (C % 2) == 0, PULP_NN_HIP_ERR_UNSUPPORTED,
          "only p_l = p_r = 1 with even C is well defined in the reference");
  depthwise_common(__func__, In_Img, nullptr, Out_Img, Kernel, kappa, lambda, out_mult, out_shift, C, R, C, R - 2, CH,
                   3, 3, 0, 1, 1, 1, epi_mode(flag_relu, flag_batch_norm));
}

}  // extern "C"
