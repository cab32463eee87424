// Host-side state and helpers shared by the library's translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#if PULPNN_BN_BITS == 64
#include "../../include/64bit/pulp_nn_kernels.h"
#else
#include "../../include/32bit/pulp_nn_kernels.h"
#endif

#include <atomic>
#include <mutex>

#include "conv_band_geom.h"
#include "dw_hwc_geom.h"
#include "dw_mfma_geom.h"
#include "requant.h"

#pragma GCC visibility push(hidden)

// per host thread: images per call, stream, last error
extern __thread unsigned g_batch;
extern __thread hipStream_t g_stream;

void set_error(int code, const char *fn, const char *msg);
void check_launch(const char *fn);
// Compute units of the current device.
int num_cus();
// Shift as the reference's quantisers see it, plus range validation.
// Returns false if the shift would be undefined behaviour in the reference.
bool epi_args(int mode, const bn_t *k, const bn_t *lambda, uint16_t out_mult, int out_shift_param, EpiArgs *e);

#define REQUIRE(cond, code, msg)        \
  do {                                  \
    if (!(cond)) {                      \
      set_error((code), __func__, msg); \
      return;                           \
    }                                   \
  } while (0)

static inline bool aligned(const void *p, unsigned a) { return ((uintptr_t)p & (a - 1)) == 0; }

// Raises a kernel's dynamic-LDS limit above the default 64 KB, once per process and kernel.
template <auto KERN>
bool raise_lds_limit(size_t lds)
{
  static std::mutex mu;
  static std::atomic<size_t> limit{65536};
  if (lds > limit.load(std::memory_order_acquire)) {
    std::lock_guard<std::mutex> lock(mu);
    if (lds > limit.load(std::memory_order_relaxed)) {
      if (hipFuncSetAttribute((const void *)KERN, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
        (void)hipGetLastError();
        return false;
      }
      limit.store(lds, std::memory_order_release);
    }
  }
  return true;
}

// ---- layers, one family per translation unit (fn: the entry point's name, for error messages) -------------------

void depthwise_common(const char *fn, const uint8_t *in, const int8_t *bias, uint8_t *out, const int8_t *wt,
                      bn_t *k, bn_t *lambda, uint16_t out_mult, int out_shift, int W, int H, int Wo, int Ho, int CH,
                      int kx, int ky, int pt, int pl, int sx, int sy, int mode, bool hwc_in = false);
void dwpw_common(const char *fn, const unsigned char *Im_in, unsigned char *Im_out, int W, int H, int C, int Wo_arg,
                 int Ho_arg, int Co, int S, unsigned n_blocks, const pulp_nn_hip_block *blocks);
void conv_common(const char *fn, bool pointwise, const uint8_t *in, const int8_t *bias, uint8_t *out,
                 const int8_t *w, bn_t *k, bn_t *lambda, uint16_t out_mult, uint16_t out_shift,
                 uint16_t dim_in_x, uint16_t dim_in_y, uint16_t ch_in, uint16_t dim_out_x, uint16_t dim_out_y,
                 uint16_t ch_out, uint16_t kx, uint16_t ky, uint16_t pt, uint16_t pl, uint16_t sx, uint16_t sy,
                 int flag_relu, int flag_batch_norm);
void linear_common(const char *fn, int mode, const uint8_t *in, const int8_t *bias, void *out, const int8_t *w,
                   const EpiArgs &e, uint16_t dim_vec, uint16_t num_o_neurons, int rows);

// ---- kernels with a launcher of their own: false, with nothing queued, for a geometry the kernel does not take ---

bool launch_conv_rows(int mode, const ConvLayer &L, const EpiArgs &e, int cus, hipStream_t s);
bool launch_conv_band(int mode, const ConvLayer &L, const EpiArgs &e, int cus, hipStream_t s);
bool launch_pw_any(int mode, const uint8_t *in, const int8_t *w, const int8_t *bias, uint8_t *out, long long M, int N, int K,
                   const EpiArgs &e, int cus, hipStream_t s);
bool launch_dw_hwc(int mode, const DwLayer &L, const EpiArgs &e, int cus, hipStream_t s);
bool launch_dw_mfma(int mode, const DwLayer &L, const EpiArgs &e, int cus, hipStream_t s);

#pragma GCC visibility pop
