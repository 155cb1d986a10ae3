// fp32 matrix products (gemm_f32.hip).
#pragma once

#include "iter.h"

namespace mi {

// out[b] = alpha * a[b] @ b[b] + beta * bias[b], any strides of a and b, unit
// column stride of c.
struct GemmF32Args {
  const float* a;
  const float* b;
  float* c;
  const void* bias;
  int bias_dtype;
  int64_t bias_sm, bias_sn, bias_sb;
  int64_t M, N, K;
  int64_t a_sm, a_sk, b_sk, b_sn, ldc;
  int64_t sa, sb, sc;
  float alpha, beta;
};

mi_status_t launch_gemm_f32(const GemmF32Args& q, int64_t batch, bool has_bias, hipStream_t s,
                            const char* what);

}  // namespace mi
