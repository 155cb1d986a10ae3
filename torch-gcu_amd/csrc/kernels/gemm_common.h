// Types that the matrix-product kernels share: MFMA operand vectors, the
// argument block and the per-column epilogue loads.
#pragma once

#include "iter.h"

namespace mi {

struct GemmArgs {
  const uint16_t* a;  // [batch][M][lda], K contiguous
  const void* b;      // [batch][N][ldb], K contiguous (16-bit or int8)
  uint16_t* c;        // [batch][M][ldc], N contiguous
  const void* bias;   // element (m, n) at bias + b*bias_sb + m*bias_sm + n*bias_sn
  const float* scale; // int8 path: per-N fp32 scale
  int bias_dtype;
  int64_t bias_sm, bias_sn, bias_sb;
  int64_t M, N, K;
  int64_t lda, ldb, ldc;
  int64_t sa, sb, sc;  // batch strides (elements)
  float alpha, beta;
  int tiles_m, tiles_n;
  // fused epilogues of the large-tile kernel (EPI_SILU, EPI_RESID below)
  const void* b2;       // EPI_SILU: the up weight, rows laid out like b's (the gate weight)
  const uint16_t* res;  // EPI_RESID: residual, element (m, n) at res[m * ldr + n]
  int64_t ldr;
};

// Few-row products (gemm_rows.hip): out = alpha * a b^T + beta * bias with
// M <= kRowsMax, one batch, K-contiguous operands of any alignment; b 16-bit, or
// int8 when q.scale is set.
constexpr int64_t kRowsMax = 64;
bool gemm_rows_eligible(const GemmArgs& q);
mi_status_t launch_gemm_rows(const GemmArgs& q, bool f16, bool has_bias, hipStream_t s,
                             const char* what);

// 16-bit products of any size by tile shape and K slices (gemm_mid.hip), for
// operands with 16-byte aligned rows, K contiguous, and byte offsets below 4 GB.
bool gemm_mid_eligible(const GemmArgs& q);
mi_status_t launch_gemm_mid(const GemmArgs& q, int64_t batch, bool f16, bool has_bias,
                            hipStream_t s, const char* what);
// linear_residual / linear_silu_mul in one kernel (K a multiple of 64); returns
// whether the call was taken, *st is its status then.
bool launch_gemm_fused(const GemmArgs& q, bool silu, bool f16, hipStream_t s, const char* what,
                       mi_status_t* st);
// out = alpha * scale[n] * sum_s part[s] + beta * bias over S slices of raw
// sums [M][ldp] (gemm.hip).
mi_status_t launch_splitk_combine(const GemmArgs& q, bool f16, bool has_bias, const float* part,
                                  int S, int64_t ldp, hipStream_t s, const char* what);

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

template <typename T>
struct MfmaOp;
template <>
struct MfmaOp<BF16> {
  typedef bf16x8 vec;
  static __device__ __forceinline__ f32x16 mma(vec a, vec b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint16_t store(float v) { return f32_to_bf16(v); }
  static __device__ __forceinline__ float load(uint16_t v) { return bf16_to_f32(v); }
};
template <>
struct MfmaOp<F16> {
  typedef f16x8 vec;
  static __device__ __forceinline__ f32x16 mma(vec a, vec b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint16_t store(float v) { return f32_to_f16(v); }
  static __device__ __forceinline__ float load(uint16_t v) { return f16_to_f32(v); }
};

typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

// 8 int8 (two words) -> 8 x bf16 / f16, exact. One sign-extending byte
// convert per value (v_cvt_f32_i32 with a byte select), then two values per
// word: the upper halves of the two floats for bf16 (exact, an int8 has at
// most 8 significant bits), a round-toward-zero pack for f16 (exact too).
// 12 VALU per 8 values; a (__bf16) cast of the float costs twice that.
template <typename T>
__device__ __forceinline__ typename MfmaOp<T>::vec widen8(u32x2_t w) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  u32x4 r;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const uint32_t d = w[p >> 1];
    const float lo = (float)(int)(int8_t)(d >> (16 * (p & 1)));
    const float hi = (float)(int)(int8_t)(d >> (16 * (p & 1) + 8));
    if constexpr (std::is_same<T, BF16>::value)
      r[p] = __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
    else
      r[p] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(lo, hi));
  }
  return __builtin_bit_cast(typename MfmaOp<T>::vec, r);
}

// v's 16 bytes shifted down by `back` bytes, zeros behind: with the 16 bytes that
// end with a row, the row's remainder as a chunk (back >= 16: a chunk past the row)
typedef uint64_t u64x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u64x2_t shift_down(u64x2_t v, int back) {
  const int s = 8 * (back & 7);
  u64x2_t r = {v[0] >> s | (v[1] << 1) << (63 - s), v[1] >> s};
  if (back & 8) r = u64x2_t{r[1], 0};
  return back < 16 ? r : u64x2_t{};
}

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint16_t u16x4_t __attribute__((ext_vector_type(4)));

// Four consecutive per-column values n .. n + 3 of a row vector (the int8
// scale, or a bias broadcast over rows) as floats: element k at
// base + off + k * stride, fp32 or of the output's 16-bit type T.  One
// vector load when all four columns exist, the stride is 1 and the address
// is aligned; else four loads with the column clamped to N - 1 (clamped
// columns only feed outputs that are never stored).
template <typename T>
__device__ __forceinline__ f32x4_t load_col4_t(const void* base, int dtype, int64_t n, int64_t stride,
                                               int64_t N, int64_t off) {
  f32x4_t r;
  if (dtype == MI_F32) {
    const float* b = (const float*)base + off;
    if (stride == 1 && n + 3 < N && (((uintptr_t)(b + n)) & 15) == 0) {
      r = *(const f32x4_t*)(b + n);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = b[min<int64_t>(n + e, N - 1) * stride];
    }
  } else {
    const uint16_t* b = (const uint16_t*)base + off;
    if (stride == 1 && n + 3 < N && (((uintptr_t)(b + n)) & 7) == 0) {
      const u16x4_t v = *(const u16x4_t*)(b + n);
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = MfmaOp<T>::load(v[e]);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = MfmaOp<T>::load(b[min<int64_t>(n + e, N - 1) * stride]);
    }
  }
  return r;
}

}  // namespace
}  // namespace mi
