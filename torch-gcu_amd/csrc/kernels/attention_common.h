// Shared by the attention kernels: MFMA operand types, arguments, and the
// chunk swizzles of K and V rows in LDS.
#pragma once

#include <cmath>

#include "iter.h"

namespace mi {

struct AttnArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  uint16_t* o;
  float* lse;
  int64_t H, Hk, Sq, Sk;
  int64_t q_sb, q_sh, q_ss;
  int64_t k_sb, k_sh, k_ss;
  int64_t v_sb, v_sh, v_ss;
  int64_t o_sb, o_sh, o_ss;
  int64_t lse_sb, lse_sh;
  float scale_log2;  // softmax scale * log2(e)
  int causal;
  int q_tiles;
  int head_group;    // (b, h) pairs whose query tiles are interleaved, longest first
  int n_blocks;      // q_tiles * H * B
  int xcd_remap;     // n_blocks % 8 == 0: renumber blocks per XCD
};

// Few query rows against a long cache (attention_decode.hip): no causal mask.
// Returns whether the call was taken; *st is its status then.
bool flash_decode(const AttnArgs& a, int64_t B, int64_t D, bool f16, hipStream_t s,
                  mi_status_t* st);

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

template <typename T>
struct AttnOp;
template <>
struct AttnOp<BF16> {
  typedef bf16x8 vec;
  typedef __bf16 elem;
  static __device__ __forceinline__ f32x16 mma(vec a, vec b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct AttnOp<F16> {
  typedef f16x8 vec;
  typedef _Float16 elem;
  static __device__ __forceinline__ f32x16 mma(vec a, vec b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

// 16-byte chunk c of key row r sits at chunk c ^ swz(r) of the row in LDS:
// K rows are read as MFMA fragments (16 rows a pass), V rows transposed by
// ds_read_b64_tr_b16 (4 rows x 4 chunks a pass); both without bank conflicts.
template <int D>
__device__ __forceinline__ int swz_k_of(int r) {
  return D == 128 ? (r & 15) : ((r >> 1) & 7);
}
template <int D>
__device__ __forceinline__ int swz_v_of(int r) {
  return D == 128 ? 4 * (r & 3) : 4 * ((r >> 1) & 1);
}

}  // namespace
}  // namespace mi
