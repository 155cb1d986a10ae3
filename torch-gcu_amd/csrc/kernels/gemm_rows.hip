// Matrix products with few rows: out[m][n] = alpha * sum_k a[m][k] b[n][k]
// + beta * bias with M <= 64, 16-bit a and a 16-bit or int8 b: the linear layers
// of a decode step.
//
// What bounds it: the weight b [N][K] is streamed once from HBM and each of
// its elements meets at most 64 rows, so the matrix cores idle and the time is
// that of the stream plus about 3 us of launch, first latency and combine.
// (The 32 x 64 tiles that ran here before made N / 64 blocks of two waves: N =
// 4096 used a quarter of the CUs.)  us per call, before and now:
//   M8 N4096 K4096 51 -> 8.4     M8 N11008 K4096 49 -> 16.7 (5.4 TB/s)
//   M8 N32000 K4096 63 -> 45 (5.8 TB/s)   M1 N4096 K11008 128 -> 20
//   M64 N11008 K4096 60 -> 26    M48 N4096 K11008 145 -> 25
//
// A block owns 16 * RT rows of b (output columns) and all M rows of a; its NW
// waves take 64-deep units of K in turn, the next unit's loads in flight while
// one is multiplied.  A wave load takes 8 rows x 128 bytes (8 adjacent lanes a
// line: loaded in the MFMA's own layout, adjacent lanes in 16 different rows,
// every lane cost the address unit a cycle and N4096 K4096 took 9.7 us); the
// rows turn into MFMA fragments through LDS tiles private to the wave, so no
// barrier is met until the partial tiles are added in a fixed order (the turn
// by quad permutes in registers measured the same at twice the registers).
// b is the MFMA's A operand, so a lane ends up with 4 consecutive columns.
//
// Addresses need only the element's alignment (a global dwordx4 load may start
// at any 2-byte address), so odd K, row strides and bases run here as they
// are; the last K % 64 (int8: 128) elements are read by one wave, in chunks that end
// with the row where they would pass it (element by element, int8 M33 N8192 K320
// took 13.0 us, 6.3 so).
#include <algorithm>

#include "gemm_common.h"

namespace mi {
namespace {

// 16 rows of 128 bytes (8 chunks of 16 bytes): chunk c of row r at c ^ f(r),
// conflict-free for the row-major writes (8 lanes a row) and for the fragment
// reads (row l % 16, chunk 4 s + l / 16).
__device__ __forceinline__ int swz(int r, int c) {
  return c ^ (r & 3) ^ (((r >> 2) & 1) * 5) ^ ((r >> 1) & 4);
}

// out[m][n .. n + 3] = alpha * s (* scale[n]) + beta * bias, rounded once.  ANY: 8
// bytes at any element (not in blocks of 16 waves: it costs them their 64 registers)
template <typename T, bool HAS_BIAS, bool I8, bool ANY>
__device__ __forceinline__ void rows_store(const GemmArgs& p, int64_t m, int64_t n, f32x4_t s) {
  f32x4_t bb = {}, sc = {1.f, 1.f, 1.f, 1.f};
  if constexpr (I8) sc = load_col4_t<T>(p.scale, MI_F32, n, 1, p.N, 0);
  if constexpr (HAS_BIAS)
    bb = load_col4_t<T>(p.bias, p.bias_dtype, n, p.bias_sn, p.N, m * p.bias_sm);
  u16x4_t v;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float x = p.alpha * s[e];
    if constexpr (I8) x *= sc[e];
    if constexpr (HAS_BIAS) x += p.beta * bb[e];
    v[e] = MfmaOp<T>::store(x);
  }
  // (8 bytes at any element: element by element an odd row length, M17 N50257 K320,
  // took 10.9 us, 9.4 so)
  typedef u16x4_t __attribute__((aligned(2))) u16x4_u;
  uint16_t* dst = p.c + m * p.ldc + n;
  if (n + 3 < p.N && (ANY || (((uintptr_t)dst) & 7) == 0)) {
    *(u16x4_u*)dst = v;
  } else {
    for (int e = 0; e < 4 && n + e < p.N; ++e) dst[e] = v[e];
  }
}

// I8: b is an int8 weight with fp32 scale per row (the int8 linear), its unit
// 128 deep; a's 16 rows of a unit are then two tiles of 64.
// Blocks of 16 waves keep to 64 registers, so that two share a CU.
template <typename T, int MT, int RT, int NW, bool HAS_BIAS, bool SPLIT, bool I8>
__global__ __launch_bounds__(64 * NW, NW == 16 ? 8 : 1) void gemm_rows_kernel(GemmArgs p, float* part, int64_t ldp) {
  typedef typename MfmaOp<T>::vec vec;
  typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
  typedef u16x8 __attribute__((aligned(1))) u16x8_u1;
  typedef u16x8 __attribute__((aligned(2))) u16x8_u2;
  typedef typename std::conditional<I8, u16x8_u1, u16x8_u2>::type u16x8_u;
  constexpr int XS = I8 ? 2 : 1, KU = 64 * XS;  // a tiles per 16 rows, k per unit
  constexpr int BE = I8 ? 1 : 2;                // bytes per b element
  constexpr int NT = RT + MT * XS;     // tiles of 16 rows x 128 bytes: RT of b, then a's
  constexpr int TILE = 16 * 64;        // 16-bit elements of one tile
  constexpr int NTL = RT * MT;
  constexpr size_t kStage = (size_t)NW * NT * TILE * 2, kRed = (size_t)NW * NTL * 64 * 16;
  __shared__ __align__(16) char smem[kStage > kRed ? kStage : kRed];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t n0 = (int64_t)blockIdx.x * (16 * RT);
  // operand tile t, half h: rows 8 h + lane / 8, 16 bytes at chunk lane % 8 of
  // each 128-byte unit.  Per-lane byte offsets from a block-uniform base (the
  // host checked that they fit 32 bits); rows past the end re-read the last
  // one and feed outputs that are never stored
  const char* base[2] = {(const char*)p.b + n0 * p.ldb * BE, (const char*)p.a};
  uint32_t off[NT][2];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int row = 8 * h + (lane >> 3);
      const int mt = (t - RT) / XS, sub = (t - RT) % XS;
      const int64_t at = t < RT
                             ? (min<int64_t>(n0 + 16 * t + row, p.N - 1) - n0) * p.ldb * BE
                             : min<int64_t>(16 * mt + row, p.M - 1) * p.lda * 2 + 128 * sub;
      off[t][h] = (uint32_t)(at + 16 * (lane & 7));
    }
  uint16_t* tile = (uint16_t*)smem + wave * (NT * TILE);
  int wo[2], ro[2], ro8[4];
#pragma unroll
  for (int s = 0; s < 4; ++s)  // int8 k 32 s + 8 (l / 16) .. + 7
    ro8[s] = (lane & 15) * 64 + 8 * swz(lane & 15, 2 * s + (lane >> 5)) + 4 * ((lane >> 4) & 1);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int row = 8 * h + (lane >> 3);
    wo[h] = row * 64 + 8 * swz(row, lane & 7);
    ro[h] = (lane & 15) * 64 + 8 * swz(lane & 15, 4 * h + (lane >> 4));
  }
  f32x4_t acc[RT][MT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = f32x4_t{};
  auto mma = [](vec a, vec b, f32x4_t c) __attribute__((always_inline)) {
    if constexpr (std::is_same<T, BF16>::value)
      return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    else
      return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  };
  // one unit: the loaded rows through the wave's own LDS tiles into
  // MFMA fragments (LDS operations of a wave stay in order)
  struct Unit {
    u16x8 v[NT][2];
  };
  auto multiply = [&](const Unit& u) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) *(u16x8*)(tile + t * TILE + wo[h]) = u.v[t][h];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int s = 0; s < KU / 32; ++s) {
      vec fw[RT], fx[MT];
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        if constexpr (I8) fw[i] = widen8<T>(*(const u32x2_t*)(tile + i * TILE + ro8[s]));
        else fw[i] = *(const vec*)(tile + i * TILE + ro[s]);
      }
#pragma unroll
      for (int j = 0; j < MT; ++j)
        fx[j] = *(const vec*)(tile + (RT + XS * j + s / 2) * TILE + ro[s & 1]);
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = mma(fw[i], fx[j], acc[i][j]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };

  // whole units k_first .. KS - 1 of this block's K slice
  int KS = (int)(p.K / KU), k_first = 0;
  const bool has_tail = KS * (int64_t)KU < p.K && (!SPLIT || blockIdx.y + 1 == gridDim.y);
  if constexpr (SPLIT) {
    const int per = KS / (int)gridDim.y, rem = KS % (int)gridDim.y, s = (int)blockIdx.y;
    k_first = s * per + min(s, rem);
    KS = k_first + per + (s < rem ? 1 : 0);
  }
  const int NU = KS - k_first;  // wave w takes units w, w + NW, ...
  // loads are unconditional (a guarded load is waited for at once): a unit past
  // the end re-reads the last one and is not multiplied
  auto load = [&](Unit& u, int c) __attribute__((always_inline)) {
    const int64_t k = (int64_t)min(k_first + c, KS - 1) * 128;  // bytes of b
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        u.v[t][h] = *(const u16x8_u*)(base[t < RT ? 0 : 1] + (t < RT ? k : k * XS) + off[t][h]);
  };
  if (wave < NU) {
    Unit u0, u1;
    load(u0, wave);
    for (int c = wave; c < NU; c += 2 * NW) {
      load(u1, c + NW);
      __builtin_amdgcn_sched_barrier(0);
      multiply(u0);
      load(u0, c + 2 * NW);
      __builtin_amdgcn_sched_barrier(0);
      if (c + NW < NU) multiply(u1);
    }
  }
  // the last K % KU elements, one wave (one with the fewest units)
  if (has_tail && wave == NW - 1) {
    const int64_t k0 = p.K / KU * KU;
    Unit u;
    // k of the lane's first element of operand tile t
    auto k_of = [&](int t) __attribute__((always_inline)) {
      return k0 + (t < RT ? 16 / BE * (lane & 7) : 64 * ((t - RT) % XS) + 8 * (lane & 7));
    };
    auto src = [&](int t, int h) __attribute__((always_inline)) {
      return base[t < RT ? 0 : 1] + off[t][h] + (t < RT ? k0 * BE : k0 * 2);
    };
    if (p.K * BE >= 16) {
      // bytes of a lane's chunk that lie past the row
      auto past = [&](int t) __attribute__((always_inline)) {
        return (int)max((int64_t)0, (k_of(t) - p.K) * (t < RT ? BE : 2) + 16);
      };
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h) u.v[t][h] = *(const u16x8_u*)(src(t, h) - past(t));
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          u.v[t][h] = __builtin_bit_cast(u16x8, shift_down(__builtin_bit_cast(u64x2_t, u.v[t][h]), past(t)));
    } else {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const char* q = src(t, h);
          const int64_t k = k_of(t);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            // (elements per 16-bit word: two of an int8 b)
            if (I8 && t < RT) {
              const uint16_t lo = k + 2 * e < p.K ? (uint8_t)q[2 * e] : 0;
              const uint16_t hi = k + 2 * e + 1 < p.K ? (uint8_t)q[2 * e + 1] : 0;
              u.v[t][h][e] = lo | (hi << 8);
            } else {
              u.v[t][h][e] = k + e < p.K ? ((const uint16_t*)q)[e] : (uint16_t)0;
            }
          }
        }
    }
    multiply(u);
  }
  // the waves' partial tiles reuse the staging tiles
  __syncthreads();
  f32x4_t* red = (f32x4_t*)smem;
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) red[(wave * NTL + i * MT + j) * 64 + lane] = acc[i][j];
  __syncthreads();
  // one lane per run of 4 columns: tile t, row 16 (t % MT) + l % 16, columns
  // n0 + 16 (t / MT) + 4 (l / 16) .. + 3
  for (int id = threadIdx.x; id < NTL * 64; id += 64 * NW) {
    const int t = id >> 6, l = id & 63;
    f32x4_t s = red[t * 64 + l];
#pragma unroll
    for (int w = 1; w < NW; ++w) s += red[(w * NTL + t) * 64 + l];
    const int64_t m = 16 * (t % MT) + (l & 15), n = n0 + 16 * (t / MT) + 4 * (l >> 4);
    if (m >= p.M || n >= p.N) continue;
    if constexpr (SPLIT) {
      // (ldp is a multiple of 4, so a run that starts inside the row fits)
      *(f32x4_t*)(part + ((int64_t)blockIdx.y * p.M + m) * ldp + n) = s;
      continue;
    }
    rows_store<T, HAS_BIAS, I8, NW != 16>(p, m, n, s);
  }
}

// out = alpha * sum_s part[s] + beta * bias, the slices added in order
template <typename T, bool HAS_BIAS, bool I8>
__global__ __launch_bounds__(256) void rows_combine_kernel(GemmArgs p, const float* part, int S,
                                                           int64_t ldp) {
  const int64_t runs = ldp / 4;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t m = idx / runs, n = (idx - m * runs) * 4;
  if (m >= p.M) return;
  const float* src = part + m * ldp + n;
  f32x4_t s = *(const f32x4_t*)src;
#pragma unroll 8
  for (int i = 1; i < S; ++i) s += *(const f32x4_t*)(src + i * p.M * ldp);
  rows_store<T, HAS_BIAS, I8, true>(p, m, n, s);
}

template <typename T, int MT, int RT, int NW, bool HB, bool I8>
mi_status_t launch(const GemmArgs& q, int S, hipStream_t s, const char* what) {
  const unsigned tiles = ceil_div_u(q.N, 16 * RT);
  const int64_t ldp = (q.N + 3) / 4 * 4;
  Workspace ws;
  if (S > 1 && ws.alloc((size_t)S * (size_t)q.M * (size_t)ldp * sizeof(float), s) != MI_OK) {
    clear_error();  // the whole K in one block needs no workspace
    S = 1;
  }
  if (S <= 1) {
    hipLaunchKernelGGL((gemm_rows_kernel<T, MT, RT, NW, HB, false, I8>), dim3(tiles), dim3(64 * NW),
                       0, s, q, nullptr, (int64_t)0);
    return check_launch(what);
  }
  float* part = (float*)ws.get();
  hipLaunchKernelGGL((gemm_rows_kernel<T, MT, RT, NW, false, true, I8>), dim3(tiles, (unsigned)S),
                     dim3(64 * NW), 0, s, q, part, ldp);
  MI_RETURN_IF(check_launch(what));
  hipLaunchKernelGGL((rows_combine_kernel<T, HB, I8>), dim3(ceil_div_u(q.M * (ldp / 4), 256)),
                     dim3(256), 0, s, q, (const float*)part, S, ldp);
  return check_launch(what);
}

// K slices for blocks of 64 weight rows that fill less than half the CUs
int slices(int64_t tiles) { return (int)std::min<int64_t>(8, std::max<int64_t>(1, cu_count() / tiles)); }

// Launch shape.  M <= 16: blocks of 16 weight rows and 8 waves, or 16 waves without
// a bias for K = 4096 .. 8192 (M8 N4096 K8192 13.8 us against 14.8, N11008 K4096 16.4
// against 16.8; K2048 9.8 against 9.3, N128256 K4096 183 against 182, and with a bias
// M8 N4096 K4096 6.8 against 6.55).  Where such blocks go twice round the CUs and K <= 512, starting and adding
// up the waves is most of the time: blocks of 64 rows and 4 waves (M8 N32000 K256
// 5.4 us, 6.3 in 16-row blocks of 8 waves, 8.8 of 16).
// M > 16: a's rows are read again by every block, and a CU takes in about
// 55 KB/us whatever the source, so blocks of 64 weight rows (a quarter of that
// traffic) wherever they fill half the CUs (M64 N11008 K4096: 26 us against
// 37).  With fewer, K is split over blocks when a is large enough to pay for
// the combine, from M K = 2^18 (M48 N4096 K11008: 25 us against 31, M64 N1024
// K9344: 15 against 26, M64 N4096 K4096: 14.4 against 14.5); below it blocks
// of 16 rows stay (M32 N4096 K4096: 10.7 us against 12.5).
template <typename T, int MT, bool HB>
mi_status_t pick_mt(const GemmArgs& q, hipStream_t s, const char* what) {
  if constexpr (MT == 1) {
    const bool wide = q.N >= 32 * (int64_t)cu_count();
    if (wide && q.K <= 512) return launch<T, 1, 4, 4, HB, false>(q, 1, s, what);
    if constexpr (!HB)
      if (q.K >= 4096 && q.K <= 8192 && q.N <= 128 * (int64_t)cu_count())
        return launch<T, 1, 1, 16, HB, false>(q, 1, s, what);
    return launch<T, 1, 1, 8, HB, false>(q, 1, s, what);
  } else {
    const int64_t tiles = (q.N + 63) / 64;
    if (2 * tiles >= cu_count()) return launch<T, MT, 4, 4, HB, false>(q, 1, s, what);
    if (q.M * q.K < (1 << 18)) return launch<T, MT, 1, 8, HB, false>(q, 1, s, what);
    return launch<T, MT, 4, 4, HB, false>(q, slices(tiles), s, what);
  }
}

// The same for an int8 weight: half the bytes per element of b, so a's rows weigh
// twice as much, but a unit's widening and four MFMAs per fragment favour small
// blocks.  us: M8 N4096 K4224 10.8 -> 5.8, M15 N1920 K7123 106 -> 12.6, M24
// N11008 K4224 28 -> 17 in blocks of 64 rows (19.5 in 16), M64 N4096 K4224 24 ->
// 13 in 16 (16 sliced), M64 N4096 K8192 39 -> 19 sliced (22 in 16).  Up to 16 rows,
// 64-row blocks for K <= 512 from N = 40 x CUs (M8 N32000 K256 8.0 us in 16, 5.5 so;
// M8 N8192 K512 4.9 and 5.2) and for K <= 1152 from 64 x CUs.
template <typename T, int MT, bool HB>
mi_status_t pick_mt8(const GemmArgs& q, hipStream_t s, const char* what) {
  if constexpr (MT > 1) {
    const int64_t tiles = (q.N + 63) / 64;
    if (2 * tiles >= cu_count()) return launch<T, MT, 4, 4, HB, true>(q, 1, s, what);
    if (q.M * q.K >= (1 << 19))
      return launch<T, MT, 4, 4, HB, true>(q, slices(tiles), s, what);
  } else {
    const int64_t cus = cu_count();
    if ((q.N >= 40 * cus && q.K <= 512) || (q.N >= 64 * cus && q.K <= 1152))
      return launch<T, MT, 4, 4, HB, true>(q, 1, s, what);
  }
  return launch<T, MT, 1, 8, HB, true>(q, 1, s, what);
}

template <typename T, bool HB>
mi_status_t pick(const GemmArgs& q, bool i8, hipStream_t s, const char* what) {
  switch ((q.M + 15) / 16) {
    case 1: return i8 ? pick_mt8<T, 1, HB>(q, s, what) : pick_mt<T, 1, HB>(q, s, what);
    case 2: return i8 ? pick_mt8<T, 2, HB>(q, s, what) : pick_mt<T, 2, HB>(q, s, what);
    case 3: return i8 ? pick_mt8<T, 3, HB>(q, s, what) : pick_mt<T, 3, HB>(q, s, what);
    default: return i8 ? pick_mt8<T, 4, HB>(q, s, what) : pick_mt<T, 4, HB>(q, s, what);
  }
}

}  // namespace

bool gemm_rows_eligible(const GemmArgs& q) {
  // 32-bit byte offsets from the block's first weight row (64 rows) and from a
  return q.M <= kRowsMax && q.K > 0 && q.K < 0x7fffffff &&
         (64 * q.ldb + q.K) * 2 < 0x7fffffff && (q.M * q.lda + q.K) * 2 < 0x7fffffff;
}

mi_status_t launch_gemm_rows(const GemmArgs& q, bool f16, bool has_bias, hipStream_t s,
                             const char* what) {
  const bool i8 = q.scale != nullptr;
  if (f16) return has_bias ? pick<F16, true>(q, i8, s, what) : pick<F16, false>(q, i8, s, what);
  return has_bias ? pick<BF16, true>(q, i8, s, what) : pick<BF16, false>(q, i8, s, what);
}

}  // namespace mi
