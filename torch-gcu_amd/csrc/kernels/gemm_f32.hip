// fp32 matrix products on the fp32 matrix instructions (v_mfma_f32_32x32x2,
// fp32 operands and accumulation).
//
// What bounds it: the matrix cores, 157 TFLOP/s in fp32, twice what the VALU
// gives without packed instructions; the 64 x 64 VALU tiles that ran here
// before loaded single floats by any stride and reached 26 TFLOP/s.
//
// A block of 4 waves owns a BM x BN tile and walks K in steps of 32 through two
// LDS stages, the next step's 16-byte loads held in registers while one is
// multiplied, one barrier a step.  An operand that is contiguous along K is
// staged as [row][k] (pitch 36: 16-byte reads of 16 rows hit all banks), one
// contiguous along its rows as [k][row] (pitch + 8: the two half-waves, 4 k
// apart, read different banks), so forward (both along K), input gradients (B
// along N) and weight gradients (both along their rows) all load whole lines
// with no transposing copy.  Half-wave h takes k = 8 c + 4 h + i as step i of
// chunk c, the same for both operands, so [row][k] fragments are one 16-byte
// read per four MFMAs.
// MFMA layout: lane l supplies A[m = l % 32] and B[n = l % 32] of its half's k
// and receives D[m = 8 (r / 4) + 4 (l / 32) + r % 4][n = l % 32].
#include <algorithm>

#include "gemm_f32.h"

namespace mi {
namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef f32x4_t __attribute__((aligned(4))) f32x4_u;

constexpr int FK = 32;   // k per step
constexpr int FNT = 256;

// A tile of R rows x FK: KC when staged along K.  fill() loads a step into
// registers, put() stores it to LDS.
template <int R, bool KC>
struct Operand {
  static constexpr int PITCH = KC ? FK + 4 : R + 8;
  static constexpr int SIZE = (KC ? R : FK) * PITCH;
  static constexpr int V = R * FK / 4 / FNT;
  static constexpr int CPL = KC ? FK / 4 : R / 4;  // 16-byte chunks per line
  const float* base;
  int64_t s_row, s_k, rows, row0;
  f32x4_t r[V];

  __device__ __forceinline__ int line(int i) const { return (int)threadIdx.x / CPL + i * (FNT / CPL); }
  __device__ __forceinline__ int chunk() const { return (int)threadIdx.x % CPL; }
  // whole 16-byte loads: unit stride along the staged direction, and all R
  // rows inside the matrix when that direction is the rows
  __device__ __forceinline__ bool whole() const {
    return KC ? s_k == 1 : s_row == 1 && row0 + R <= rows;
  }
  __device__ __forceinline__ void fill(int64_t k0) {
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const float* q = KC ? base + min(row0 + line(i), rows - 1) * s_row + k0 + 4 * chunk()
                          : base + (k0 + line(i)) * s_k + row0 + 4 * chunk();
      r[i] = *(const f32x4_u*)q;
    }
  }
  // any strides and edges: rows clamped to the last (their outputs are not
  // stored), zeros past K; pieces wholly outside are not loaded
  __device__ __forceinline__ void fill_any(int64_t k0, int64_t K) {
#pragma unroll
    for (int i = 0; i < V; ++i) {
      r[i] = f32x4_t{};
      if (row0 + (KC ? line(i) : 4 * chunk()) >= rows || k0 + (KC ? 4 * chunk() : line(i)) >= K) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t row = row0 + (KC ? line(i) : 4 * chunk() + e);
        const int64_t k = k0 + (KC ? 4 * chunk() + e : line(i));
        r[i][e] = base[min(row, rows - 1) * s_row + min(k, K - 1) * s_k];
      }
    }
#pragma unroll
    for (int i = 0; i < V; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        r[i][e] = k0 + (KC ? 4 * chunk() + e : line(i)) < K ? r[i][e] : 0.f;
  }
  __device__ __forceinline__ void put(float* lds) const {
#pragma unroll
    for (int i = 0; i < V; ++i) *(f32x4_t*)(lds + line(i) * PITCH + 4 * chunk()) = r[i];
  }
  // four MFMA steps of chunk c for tile row `row`
  static __device__ __forceinline__ f32x4_t frag(const float* lds, int row, int c, int half) {
    if constexpr (KC) {
      return *(const f32x4_t*)(lds + row * PITCH + 8 * c + 4 * half);
    } else {
      f32x4_t v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = lds[(8 * c + 4 * half + i) * PITCH + row];
      return v;
    }
  }
};

template <int BM, int BN, bool AKC, bool BKC, bool HAS_BIAS, bool SPLIT>
__global__ __launch_bounds__(FNT, 2) void gemm_f32_kernel(GemmF32Args p, float* part) {
  typedef Operand<BM, AKC> OA;
  typedef Operand<BN, BKC> OB;
  constexpr int FM = BM / 64, FN = BN / 64;  // 32 x 32 tiles per wave (waves 2 x 2)
  __shared__ __align__(16) float smem[2][OA::SIZE + OB::SIZE];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int half = lane >> 5, col = lane & 31;
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
  // XCD-aware tile order, groups of 8 row panels
  const int tiles_m = (int)((p.M + BM - 1) / BM), tiles_n = (int)((p.N + BN - 1) / BN);
  int tm, tn;
  {
    const int total = tiles_m * tiles_n;
    int id = blockIdx.x;
    if (total % 8 == 0) id = (id % 8) * (total / 8) + id / 8;
    const int group = id / (8 * tiles_n), first = group * 8;
    const int gsize = min(tiles_m - first, 8), in = id - group * 8 * tiles_n;
    tm = first + in % gsize;
    tn = in / gsize;
  }
  const int64_t batch = SPLIT ? 0 : blockIdx.y;
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  // this block's K range [k0, k1): whole steps, the last one of all may be partial
  int64_t k0 = 0, k1 = p.K;
  if constexpr (SPLIT) {
    const int64_t steps = (p.K + FK - 1) / FK, s = blockIdx.y, S = gridDim.y;
    k0 = steps * s / S * FK;
    k1 = min(steps * (s + 1) / S * FK, p.K);
  }
  OA a;
  OB b;
  a.base = p.a + batch * p.sa;
  a.s_row = p.a_sm;
  a.s_k = p.a_sk;
  a.rows = p.M;
  a.row0 = m0;
  b.base = p.b + batch * p.sb;
  b.s_row = p.b_sn;
  b.s_k = p.b_sk;
  b.rows = p.N;
  b.row0 = n0;
  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x16{};
  // a wave whose tiles lie outside the matrix multiplies nothing, and a last
  // step only the chunks below `left` (with the pieces that fill_any leaves out,
  // 5000 batches of 8 x 8 x 8 take 12.8 us, 22 before)
  const bool idle = m0 + wm >= p.M || n0 + wn >= p.N;
  auto compute = [&](int st, int64_t left, bool skip) __attribute__((always_inline)) {
    if (skip) return;
    const float* as = smem[st];
    const float* bs = as + OA::SIZE;
#pragma unroll
    for (int c = 0; c < FK / 8; ++c) {
      if (8 * c >= left) break;
      f32x4_t af[FM], bf[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) af[i] = OA::frag(as, wm + 32 * i + col, c, half);
#pragma unroll
      for (int j = 0; j < FN; ++j) bf[j] = OB::frag(bs, wn + 32 * j + col, c, half);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[i][e], bf[j][e], acc[i][j], 0, 0, 0);
    }
  };
  const bool whole = a.whole() && b.whole();
  auto step = [&](int64_t k) __attribute__((always_inline)) {
    if (whole && k + FK <= k1) {
      a.fill(k);
      b.fill(k);
    } else {
      a.fill_any(k, k1);
      b.fill_any(k, k1);
    }
  };
  int st = 0;
  step(k0);
  a.put(smem[0]);
  b.put(smem[0] + OA::SIZE);
  __syncthreads();
  int64_t k = k0 + FK;
  if (whole) {
    for (; k + FK <= k1; k += FK) {
      a.fill(k);
      b.fill(k);
      __builtin_amdgcn_sched_barrier(0);  // the loads go out before the MFMAs
      compute(st, FK, false);
      st ^= 1;
      a.put(smem[st]);
      b.put(smem[st] + OA::SIZE);
      __syncthreads();
    }
  }
  for (; k < k1; k += FK) {
    a.fill_any(k, k1);
    b.fill_any(k, k1);
    __builtin_amdgcn_sched_barrier(0);
    compute(st, FK, idle);
    st ^= 1;
    a.put(smem[st]);
    b.put(smem[st] + OA::SIZE);
    __syncthreads();
  }
  compute(st, k1 - (k - FK), idle);

  float* C = SPLIT ? part + (int64_t)blockIdx.y * p.M * p.N : p.c + batch * p.sc;
  const int64_t ldc = SPLIT ? p.N : p.ldc;
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int64_t n = n0 + wn + 32 * j + col;
    if (n >= p.N) continue;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t m = m0 + wm + 32 * i + 8 * (r >> 2) + 4 * half + (r & 3);
        if (m >= p.M) continue;
        float v = acc[i][j][r];
        if constexpr (!SPLIT) {
          v *= p.alpha;
          if (HAS_BIAS)
            v += p.beta * load_as<float>(p.bias, batch * p.bias_sb + m * p.bias_sm + n * p.bias_sn,
                                         p.bias_dtype);
        }
        C[m * ldc + n] = v;
      }
  }
}

// out = alpha * sum_s part[s] + beta * bias, the slices added in order
template <bool HAS_BIAS>
__global__ __launch_bounds__(256) void f32_combine_kernel(GemmF32Args p, const float* part, int S) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x, MN = p.M * p.N;
  if (idx >= MN) return;
  const int64_t m = idx / p.N, n = idx - m * p.N;
  float x = 0.f;
  for (int s0 = 0; s0 < S; s0 += 8) {
    float v[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) v[s] = part[idx + min(s0 + s, S - 1) * MN];
#pragma unroll
    for (int s = 0; s < 8; ++s) x += s0 + s < S ? v[s] : 0.f;
  }
  x *= p.alpha;
  if (HAS_BIAS) x += p.beta * load_as<float>(p.bias, m * p.bias_sm + n * p.bias_sn, p.bias_dtype);
  p.c[m * p.ldc + n] = x;
}

template <int BM, int BN, bool AKC, bool BKC, bool HB>
mi_status_t launch(const GemmF32Args& q, int64_t batch, int S, hipStream_t s, const char* what) {
  const unsigned tiles = (unsigned)(((q.M + BM - 1) / BM) * ((q.N + BN - 1) / BN));
  Workspace ws;
  if (S > 1 && ws.alloc((size_t)S * (size_t)q.M * (size_t)q.N * sizeof(float), s) != MI_OK) {
    clear_error();  // the whole K in one block needs no workspace
    S = 1;
  }
  if (S <= 1) {
    hipLaunchKernelGGL((gemm_f32_kernel<BM, BN, AKC, BKC, HB, false>), dim3(tiles, (unsigned)batch),
                       dim3(FNT), 0, s, q, nullptr);
    return check_launch(what);
  }
  hipLaunchKernelGGL((gemm_f32_kernel<BM, BN, AKC, BKC, false, true>), dim3(tiles, (unsigned)S),
                     dim3(FNT), 0, s, q, (float*)ws.get());
  MI_RETURN_IF(check_launch(what));
  hipLaunchKernelGGL((f32_combine_kernel<HB>), dim3(ceil_div_u(q.M * q.N, 256)), dim3(256), 0, s, q,
                     (const float*)ws.get(), S);
  return check_launch(what);
}

// Tile and K slices by cost in us: a 128 x 128 tile's step takes 1.95 us of a
// CU's matrix cores and a 64 x 64 one's 0.53, or 2.2 and 0.6 when a CU has only
// one block to run; slices add the combine launch and their partial sums.
// Timed on 18 shapes (M 37 .. 4096, all layouts): M42 N1216 K768 18 us whole, 8
// in 8 slices (79 before); 2000 x 2048 x 1024 78 on either tile (237 before);
// 4096^3 1013 on 128 x 128 tiles, 1160 on 64 x 64 (4107 before).
template <bool AKC, bool BKC, bool HB>
mi_status_t pick(const GemmF32Args& q, int64_t batch, hipStream_t s, const char* what) {
  const int64_t cus = cu_count(), steps = (q.K + FK - 1) / FK;
  auto blocks = [&](int64_t t) { return ((q.M + t - 1) / t) * ((q.N + t - 1) / t) * batch; };
  auto rounds = [&](int64_t n) { return (float)((n + cus - 1) / cus); };
  float best = 5.f + (float)steps * std::max(2.2f, 1.95f * rounds(blocks(128)));
  int slices = 0;  // 0: 128 x 128 tiles
  for (int S : {1, 2, 4, 8, 16, 32}) {
    if (S > 1 && (batch > 1 || S > steps)) break;
    float t = 4.f + (float)((steps + S - 1) / S) * std::max(0.6f, 0.53f * rounds(blocks(64) * S));
    if (S > 1) t += 3.f + (float)S * (float)q.M * (float)q.N * (8.f / 5.8e6f);
    if (t < best) {
      best = t;
      slices = S;
    }
  }
  if (slices == 0) return launch<128, 128, AKC, BKC, HB>(q, batch, 1, s, what);
  return launch<64, 64, AKC, BKC, HB>(q, batch, slices, s, what);
}

template <bool HB>
mi_status_t by_layout(const GemmF32Args& q, int64_t batch, hipStream_t s, const char* what) {
  // staged along K unless only the rows are contiguous
  const bool akc = q.a_sk == 1 || q.a_sm != 1, bkc = q.b_sk == 1 || q.b_sn != 1;
  if (akc) return bkc ? pick<true, true, HB>(q, batch, s, what) : pick<true, false, HB>(q, batch, s, what);
  return bkc ? pick<false, true, HB>(q, batch, s, what) : pick<false, false, HB>(q, batch, s, what);
}

}  // namespace

mi_status_t launch_gemm_f32(const GemmF32Args& q, int64_t batch, bool has_bias, hipStream_t s,
                            const char* what) {
  return has_bias ? by_layout<true>(q, batch, s, what) : by_layout<false>(q, batch, s, what);
}

}  // namespace mi
