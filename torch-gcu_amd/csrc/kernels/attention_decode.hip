// Attention of a few query rows against a long key/value cache (a decode
// step): out = softmax(scale q k^T) v with no mask, D = 64 or 128, bf16 / f16.
//
// What bounds it: K and V are read once from HBM; the queries that share a
// k/v head are few.  The 128-row flash kernel gave every query head a block of
// its own (grouped heads re-read their K and V, one row in 128 was used) and
// walked all keys in it.  Here the G query heads of a group times Sq rows are
// the rows of one MFMA tile (up to 32; more rows take further tiles), and the
// keys are split over blocks and, inside a block, over its four waves, which
// never wait for each other: a wave streams its own 32-key tiles of K and V by
// global_load_lds into a two-slot ring of its own (a block's rings hold 128 KiB at
// D = 128, 64 KiB at 64) and keeps its own running max, sum and O.  The four waves are merged through
// LDS, the blocks' fp32 partials by flash_decode_combine_kernel in a fixed order.
// MFMA layouts are the flash kernel's (S^T = K Q^T, P from registers,
// O^T += V^T P^T with V^T by ds_read_b64_tr_b16), P rounded to the input type.
#include <algorithm>

#include "attention_common.h"

namespace mi {
namespace {

constexpr int DKT = 32;  // keys per tile
constexpr int DNW = 4;   // waves per block

struct DecodeArgs {
  int64_t rows;       // query rows per k/v head: (H / Hk) * Sq
  int row_tiles;      // ceil(rows / 32)
  int splits;         // key splits (blocks) per k/v head and row tile
  int tiles;          // ceil(Sk / 32)
  int64_t all_rows;   // B * H * Sq
  float* part_o;      // [splits][all_rows][D], not normalised
  float* part_ml;     // [splits][all_rows][2]: max (log2 units), sum
};

template <int N>
__device__ __forceinline__ void decode_wait() {
  // vmcnt(N) alone
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

template <typename T, int D>
__global__ __launch_bounds__(64 * DNW, 1) void flash_decode_kernel(AttnArgs p, DecodeArgs d) {
  typedef typename AttnOp<T>::vec vec;
  constexpr int DF = D / 16, DT = D / 32;   // k-steps of K Q^T, 32-row tiles of O^T
  constexpr int CPR = D / 8, RPI = 64 / CPR;  // chunks per row, rows per 1 KiB copy
  constexpr int NINS = DKT / RPI;           // copies of a K (or V) tile
  constexpr int TILE = DKT * D;             // elements
  constexpr int KO = 16 / RPI;              // distinct K offsets: the swizzle repeats every 16 rows
  __shared__ __align__(16) uint16_t smem[DNW][2][2 * TILE];
  __shared__ float ml[DNW][32][2];

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5, col = lane & 31;
  const int split = (int)(blockIdx.x % d.splits);
  const int64_t t = blockIdx.x / d.splits;
  const int rt = (int)(t % d.row_tiles);
  const int64_t bh = t / d.row_tiles;
  const int64_t hk = bh % p.Hk, b = bh / p.Hk, G = p.H / p.Hk;
  // the query row this lane owns: row i of the group is head i / Sq, query i % Sq
  const int64_t row = (int64_t)rt * 32 + col, rc = min(row, d.rows - 1);
  const int64_t h = hk * G + rc / p.Sq, sq = rc % p.Sq;
  auto uniform = [](const uint16_t* ptr) __attribute__((always_inline)) {
    const uint64_t v = (uint64_t)ptr;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (const uint16_t*)(((uint64_t)hi << 32) | lo);
  };
  const uint16_t* Q = p.q + b * p.q_sb + h * p.q_sh + sq * p.q_ss;
  const uint16_t* K = uniform(p.k + b * p.k_sb + hk * p.k_sh);
  const uint16_t* V = uniform(p.v + b * p.v_sb + hk * p.v_sh);
  vec qf[DF];
#pragma unroll
  for (int i = 0; i < DF; ++i) qf[i] = *(const vec*)(Q + 16 * i + 8 * half);

  // per-lane byte offsets of a tile's copies (32-bit: the host checked that a
  // head's keys span less than 2^31 elements)
  const int k_ss = (int)p.k_ss, v_ss = (int)p.v_ss, Sk = (int)p.Sk;
  const int lr = lane / CPR, cp = lane % CPR;
  uint32_t kob[KO], vob;
#pragma unroll
  for (int i = 0; i < KO; ++i) {
    const int key = i * RPI + lr;
    kob[i] = (uint32_t)(((int64_t)key * k_ss + 8 * (cp ^ swz_k_of<D>(key))) * 2);
  }
  vob = (uint32_t)(((int64_t)lr * v_ss + 8 * (cp ^ swz_v_of<D>(lr))) * 2);
  auto copy_tile = [&](int j, int st) __attribute__((always_inline)) {
    uint16_t* ks = smem[wave][st];
    uint16_t* vs = ks + TILE;
    const int kv0 = j * DKT;
    if (kv0 + DKT <= Sk) {
#pragma unroll
      for (int q = 0; q < NINS; ++q)
        lds_copy16(K + (int64_t)(kv0 + q / KO * 16) * k_ss, kob[q % KO], ks + q * 512);
#pragma unroll
      for (int q = 0; q < NINS; ++q)
        lds_copy16(V + (int64_t)(kv0 + q * RPI) * v_ss, vob, vs + q * 512);
    } else {
      // keys past the end re-read the last one (masked below)
#pragma unroll
      for (int q = 0; q < NINS; ++q) {
        const int key = q * RPI + lr, gk = min(kv0 + key, Sk - 1);
        lds_copy16(K, (uint32_t)(gk * k_ss + 8 * (cp ^ swz_k_of<D>(key))) * 2u, ks + q * 512);
      }
#pragma unroll
      for (int q = 0; q < NINS; ++q) {
        const int key = q * RPI + lr, gk = min(kv0 + key, Sk - 1);
        lds_copy16(V, (uint32_t)(gk * v_ss + 8 * (cp ^ swz_v_of<D>(key))) * 2u, vs + q * 512);
      }
    }
  };
  // fragment offsets in bytes, as in the flash kernel
  int kbm, vbm;
  {
    const int sk = swz_k_of<D>(col);
    kbm = 2 * col * D + 16 * (half ^ (sk & 1)) + 32 * (sk >> 1);
    const int g = lane >> 4, j = lane & 15;
    const int key = 4 * (g >> 1) + (j >> 2);
    const int low = 2 * (g & 1) + ((j & 3) >> 1), within = 4 * (j & 1);
    vbm = 2 * key * D + 64 * (swz_v_of<D>(key) >> 2) + 16 * low + 2 * within;
  }
  f32x16 o[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i) o[i] = f32x16{};
  float m_run = -INFINITY, l_run = 0.f;
  const float sc = p.scale_log2;
  const bool neg = sc < 0.f;

  // this wave's tiles: first, first + stride, ...
  const int first = split * DNW + wave, stride = d.splits * DNW;
  if (first < d.tiles) copy_tile(first, 0);
  if (first + stride < d.tiles) copy_tile(first + stride, 1);
  int st = 0;
  for (int j = first; j < d.tiles; j += stride, st ^= 1) {
    if (j + stride < d.tiles) decode_wait<2 * NINS>();
    else decode_wait<0>();
    asm volatile("" ::: "memory");
    const char* ks = (const char*)smem[wave][st];
    const uint16_t* vs = smem[wave][st] + TILE;
    f32x16 s = f32x16{};
#pragma unroll
    for (int i = 0; i < DF; ++i)
      s = AttnOp<T>::mma(*(const vec*)(ks + (kbm ^ (32 * i))), qf[i], s);
    // accumulator r is key 8 (r / 4) + 4 half + r % 4 of the tile
    const int lim = Sk - j * DKT - 4 * half;
    if (j * DKT + DKT > Sk) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        s[r] = 8 * (r >> 2) + (r & 3) >= lim ? (neg ? INFINITY : -INFINITY) : s[r];
    }
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, neg ? -s[r] : s[r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64)) * fabsf(sc);
    if (mx > m_run) {
      const float corr = __builtin_amdgcn_exp2f(m_run - mx);
      m_run = mx;
      l_run *= corr;
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[i][r] *= corr;
    }
    const float m_use = m_run == -INFINITY ? 0.f : m_run;
    vec pk[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      f32x8 pf;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        pf[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[8 * k + i], sc, -m_use));
        l_run += pf[i];
      }
      pk[k] = __builtin_convertvector(pf, vec);
    }
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int i = 0; i < DT; ++i) {
        typedef short s16x4 __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
        const uint16_t* vb = (const uint16_t*)((const char*)(vs + 16 * k * D) + (vbm ^ (64 * i)));
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)vb);
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(vb + 8 * D));
        const vec vf =
            __builtin_bit_cast(vec, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        o[i] = AttnOp<T>::mma(vf, pk[k], o[i]);
      }
    // the slot's fragment reads have returned before its next copies go out
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (j + 2 * stride < d.tiles) copy_tile(j + 2 * stride, st);
  }

  // merge the waves: common max, scaled sums, O added in wave order
  float l = l_run + __shfl_xor(l_run, 32, 64);
  if (half == 0) {
    ml[wave][col][0] = m_run;
    ml[wave][col][1] = l;
  }
  __syncthreads();
  float M = -INFINITY;
#pragma unroll
  for (int w = 0; w < DNW; ++w) M = fmaxf(M, ml[w][col][0]);
  const float mu = M == -INFINITY ? 0.f : M;
  const float own = __builtin_amdgcn_exp2f(m_run - mu);
  l = 0.f;
#pragma unroll
  for (int w = 0; w < DNW; ++w) l += ml[w][col][1] * __builtin_amdgcn_exp2f(ml[w][col][0] - mu);
  float* red = (float*)&smem[0][0][0];  // [wave][DT * 16][64]
#pragma unroll
  for (int i = 0; i < DT; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) red[((wave * DT + i) * 16 + r) * 64 + lane] = o[i][r] * own;
  __syncthreads();
  if (row >= d.rows) return;
  const bool whole = d.splits == 1;
  const int64_t id = (b * p.H + h) * p.Sq + sq;
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  // wave w finishes runs w DT .. w DT + DT - 1 of the O^T tiles' 4-row runs
#pragma unroll
  for (int k = 0; k < DT; ++k) {
    const int run = wave * DT + k, i = run >> 2, g = run & 3;
    typedef float f4 __attribute__((ext_vector_type(4)));
    f4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float x = 0.f;
#pragma unroll
      for (int w = 0; w < DNW; ++w) x += red[((w * DT + i) * 16 + 4 * g + e) * 64 + lane];
      v[e] = x;
    }
    const int dd = 32 * i + 8 * g + 4 * half;
    if (whole) {
      typedef typename AttnOp<T>::elem E;
      typedef E e4 __attribute__((ext_vector_type(4)));
      *(e4*)(p.o + b * p.o_sb + h * p.o_sh + sq * p.o_ss + dd) = __builtin_convertvector(v * inv, e4);
    } else {
      *(f4*)(d.part_o + ((int64_t)split * d.all_rows + id) * D + dd) = v;
    }
  }
  if (wave == 0 && half == 0) {
    if (!whole) {
      d.part_ml[((int64_t)split * d.all_rows + id) * 2] = M;
      d.part_ml[((int64_t)split * d.all_rows + id) * 2 + 1] = l;
    } else if (p.lse) {
      p.lse[b * p.lse_sb + h * p.lse_sh + sq] =
          l > 0.f ? (M + __builtin_amdgcn_logf(l)) * 0.6931471805599453f : INFINITY;
    }
  }
}

// One block per query row: the splits' partials merged in a fixed order.  In
// every wave lane i holds split i's max and sum; wave w adds the O of splits w,
// w + 4, ... (four loads in flight: one split at a time, 31 splits took 10.8
// us), a lane D / 64 elements, and the waves are added through LDS.
template <typename T, int D>
__global__ __launch_bounds__(256) void flash_decode_combine_kernel(AttnArgs p, DecodeArgs d) {
  constexpr int E = D / 64;
  typedef float fe __attribute__((ext_vector_type(E)));
  __shared__ fe part[4][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t id = blockIdx.x;
  const float* pm = d.part_ml + ((int64_t)min(lane, d.splits - 1) * d.all_rows + id) * 2;
  const float m = pm[0], ls = pm[1];
  const float* src = d.part_o + id * D + lane * E;
  const float M = wave_fmax(m), mu = M == -INFINITY ? 0.f : M;
  const float w = lane < d.splits ? __builtin_amdgcn_exp2f(m - mu) : 0.f;
  const float l = wave_sum(lane < d.splits ? ls * w : 0.f);
  fe acc = {};
  for (int s = wave; s < d.splits; s += 16) {
    fe v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      v[k] = *(const fe*)(src + (int64_t)min(s + 4 * k, d.splits - 1) * d.all_rows * D);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (s + 4 * k < d.splits) acc += v[k] * readlane_f32(w, s + 4 * k);
  }
  part[wave][lane] = acc;
  __syncthreads();
  if (wave != 0) return;
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  acc = part[0][lane] + part[1][lane] + part[2][lane] + part[3][lane];
  const int64_t sq = id % p.Sq, h = id / p.Sq % p.H, b = id / p.Sq / p.H;
  typedef typename AttnOp<T>::elem Et;
  typedef Et ee __attribute__((ext_vector_type(E)));
  *(ee*)(p.o + b * p.o_sb + h * p.o_sh + sq * p.o_ss + lane * E) =
      __builtin_convertvector(acc * inv, ee);
  if (lane == 0 && p.lse)
    p.lse[b * p.lse_sb + h * p.lse_sh + sq] =
        l > 0.f ? (M + __builtin_amdgcn_logf(l)) * 0.6931471805599453f : INFINITY;
}

template <typename T, int D>
mi_status_t launch(const AttnArgs& a, const DecodeArgs& d, int64_t blocks, hipStream_t s) {
  hipLaunchKernelGGL((flash_decode_kernel<T, D>), dim3((unsigned)blocks), dim3(64 * DNW), 0, s, a, d);
  MI_RETURN_IF(check_launch("flash_attention_fwd"));
  if (d.splits == 1) return MI_OK;
  hipLaunchKernelGGL((flash_decode_combine_kernel<T, D>), dim3((unsigned)d.all_rows), dim3(256), 0,
                     s, a, d);
  return check_launch("flash_attention_fwd");
}

}  // namespace

bool flash_decode(const AttnArgs& a, int64_t B, int64_t D, bool f16, hipStream_t s,
                  mi_status_t* st) {
  // A cache of at least 8 tiles, and either grouped heads to share its reads or
  // too few (batch, k/v head) pairs for the CUs, so that keys are split.  us,
  // flash kernel and this one: 8 x 8 k/v heads of 4000 keys, G = 4: 96 / 30; 1 x
  // 32, 16000 keys, G = 1: 308 / 53; 12 x 16, 775 keys, G = 2, 8 queries: 33 /
  // 21; left out: 32 x 32, 512 keys, G = 1: 56 / 59; 4 x 8, 99 keys: 6.1 / 6.4.
  // More than 64 rows stay with the flash kernel, which is the slower one for the few
  // pairs of a long cache (4 k/v heads, 8000 keys, 72 rows: 156 / 18) and the faster
  // one for many rows (8 x 8, 4000 keys, 256 rows: 90 / 149).
  DecodeArgs d{};
  d.rows = a.H / a.Hk * a.Sq;
  if (a.causal || d.rows > 64) return false;
  d.row_tiles = (int)((d.rows + 31) / 32);
  d.tiles = (int)((a.Sk + DKT - 1) / DKT);
  d.all_rows = B * a.H * a.Sq;
  const int64_t base = B * a.Hk * d.row_tiles;
  if (d.tiles < 8 || base > 0x7fffffff / 64) return false;
  // one block per CU (at D = 128 its LDS holds no more), every wave at least two
  // tiles; pairs for more than half the CUs are not split (17 x 8 k/v heads of 4096
  // keys, 136 blocks: 53 us, flash kernel 191)
  d.splits = (int)std::min<int64_t>(64, std::min<int64_t>(cu_count() / base, d.tiles / (2 * DNW)));
  if (d.splits < 2 && a.H == a.Hk) return false;
  Workspace ws;
  if (d.splits > 1) {
    const size_t no = (size_t)d.splits * d.all_rows * D, nm = (size_t)d.splits * d.all_rows * 2;
    if (ws.alloc((no + nm) * sizeof(float), s) == MI_OK) {
      d.part_o = (float*)ws.get();
      d.part_ml = d.part_o + no;
    } else {
      clear_error();  // the flash kernel needs no workspace
      return false;
    }
  } else {
    d.splits = 1;
  }
  const int64_t blocks = base * d.splits;
  if (f16) *st = D == 128 ? launch<F16, 128>(a, d, blocks, s) : launch<F16, 64>(a, d, blocks, s);
  else *st = D == 128 ? launch<BF16, 128>(a, d, blocks, s) : launch<BF16, 64>(a, d, blocks, s);
  return true;
}

}  // namespace mi
