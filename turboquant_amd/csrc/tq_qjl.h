// tq_qjl.h -- the QJL product kernels of tq_qjl.hip, for tq_mse.hip.
#pragma once

#include "tq_common.h"

namespace tq {

// residual scale of the quantize's operand halves (a power of two: exact)
constexpr float kQjlScale = 4096.0f;

// quant: zout = sign(X S^T) from X's halves [n][ldk] and S's halves
// [ldk][ldk]; else term = z S (fp32 [n][dim]) from S^T's halves.  ldk is a
// multiple of 128 and >= dim, columns and rows past dim zero.
hipError_t launch_qjl(bool quant, const _Float16* xh, const _Float16* xl, const int8_t* z,
                      const _Float16* wh, const _Float16* wl, int8_t* zout, float* term, int64_t n,
                      int dim, int ldk, hipStream_t st);

}  // namespace tq
