// tq_qjl.h -- the QJL product kernels of tq_qjl.hip, for tq_mse.hip.
#pragma once

#include "tq_common.h"

namespace tq {

// residual scale of the quantize's operand halves (a power of two: exact)
constexpr float kQjlScale = 4096.0f;

typedef _Float16 qjl_half2_t __attribute__((ext_vector_type(2)));

// four int8 as fp16 (exact: 1024 + (z + 128) - 1152)
__device__ __forceinline__ void z_to_half(uint32_t w, uint32_t& lo, uint32_t& hi) {
  const uint32_t u = w ^ 0x80808080u;
  const qjl_half2_t b = {(_Float16)1152.0f, (_Float16)1152.0f};
  lo = __builtin_bit_cast(uint32_t, (qjl_half2_t)(__builtin_bit_cast(qjl_half2_t, __builtin_amdgcn_perm(
                                        0x64646464u, u, 0x04010400u)) - b));
  hi = __builtin_bit_cast(uint32_t, (qjl_half2_t)(__builtin_bit_cast(qjl_half2_t, __builtin_amdgcn_perm(
                                        0x64646464u, u, 0x04030402u)) - b));
}

// quant: zout = sign(X S^T) from X's halves [n][ldk] and S's halves
// [ldk][ldk]; else term = z S (fp32 [n][dim]) from S^T's halves, column j
// times wscale[j] (null: 1).  ldk is a multiple of 128 and >= dim, columns and
// rows past dim zero.
hipError_t launch_qjl(bool quant, const _Float16* xh, const _Float16* xl, const int8_t* z,
                      const _Float16* wh, const _Float16* wl, const float* wscale, int8_t* zout,
                      float* term, int64_t n, int dim, int ldk, hipStream_t st);

}  // namespace tq
