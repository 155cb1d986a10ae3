// Dense contractions on gfx950 MFMA: addmm / mm / bmm / baddbmm and the int8
// weight-only linear.
//
// 16-bit products run the few-row kernel (gemm_rows.hip) or the direct-to-LDS
// pipeline (gemm_dl.h, its tile shapes chosen in gemm_mid.hip); this file holds
// the dispatch, the int8 kernels, the fused epilogues and the register-staged
// kernel that remains for int8 B at other sizes and for operands whose byte
// offsets pass 32 bits: v_mfma_f32_32x32x16_{bf16,f16}, fp32 accumulation,
//   - a block owns a BM x BN output tile and walks K in steps of 64;
//   - WM x WN waves each own a (BM/WM) x (BN/WN) sub-tile, i.e. a grid of
//     32 x 32 MFMA tiles (the 256 x 256 configuration gives every wave
//     16 tiles = 256 fp32 accumulators, which live in AGPRs);
//   - A rows and B rows (B is read as [N, K], K contiguous) are staged
//     through LDS with a 72-element row pitch (16 bytes of padding) so the
//     16-byte operand reads of 32 consecutive rows fall in distinct banks;
//     two LDS stages let the global loads of step k+1 overlap the MFMAs of
//     step k with one barrier per step;
//   - for the int8 weight-only linear, B tiles arrive as int8 (half the
//     bytes) and are widened to bf16 on the way into LDS (an int8 value is
//     exactly a bf16 whose low 16 fp32 bits are zero), and the epilogue
//     multiplies by the per-output-channel fp32 scale.
// MFMA operand layout (checked on the device): lane l supplies
//   A[m = l % 32][k = 8 * (l / 32) + i] and B[k = 8 * (l / 32) + i][n = l % 32],
//   i < 8, and receives D[m = 8 * (r / 4) + 4 * (l / 32) + r % 4][n = l % 32]
//   in accumulator r < 16.
// Workgroups are renumbered so that each of the 8 XCDs (which receive
// workgroups round robin) gets a contiguous run of tiles, walked in groups
// of 8 row panels, so tiles sharing A and B panels meet in one L2.
// fp32 inputs run gemm_f32.hip.
#include <algorithm>

#include "gemm_dl.h"
#include "gemm_f32.h"

namespace mi {
namespace {

constexpr int BK = 64;
constexpr int PITCH = BK + 8;  // LDS row pitch in elements

__device__ __forceinline__ void tile_of(int bid, int tiles_m, int tiles_n, int* tm, int* tn) {
  const int total = tiles_m * tiles_n;
  constexpr int XCD = 8;
  int id = bid;
  if (total % XCD == 0) {
    const int per = total / XCD;
    id = (bid % XCD) * per + bid / XCD;
  }
  constexpr int GROUP_M = 8;
  const int group = id / (GROUP_M * tiles_n);
  const int first_m = group * GROUP_M;
  const int gsize = min(tiles_m - first_m, GROUP_M);
  const int in_group = id - group * GROUP_M * tiles_n;
  *tm = first_m + in_group % gsize;
  *tn = in_group / gsize;
}

// Per-lane loader of a ROWS x 64 tile of a K-contiguous 16-bit matrix: V
// 16-byte vectors per lane, 8 lanes per 128-byte row segment; vector i of a
// lane covers tile row row0 + i * (NT / 8).  Rows past the end of the matrix
// are clamped to its last row: their products only reach output rows or
// columns that are never stored.  The last, partial K step (load_tail) reads
// the elements at k >= K as zero.  Addresses are formed at load time so that
// no per-vector pointer stays live across the main loop.
template <int ROWS, int NT>
struct Tile16 {
  static constexpr int V = ROWS * 8 / NT;
  static constexpr int RS = NT / 8;  // rows between a lane's vectors
  const uint16_t* base;
  int64_t ld, last, row0;
  int kc;
  uint4 r[V];
  __device__ __forceinline__ void init(const uint16_t* b, int64_t ld_, int64_t rows, int64_t r0) {
    base = b;
    ld = ld_;
    last = rows - 1;
    row0 = r0 + (threadIdx.x >> 3);
    kc = (threadIdx.x & 7) * 8;
  }
  __device__ __forceinline__ const uint16_t* at(int i, int64_t k0) const {
    const int64_t gr = min(row0 + (int64_t)i * RS, last);
    return base + gr * ld + kc + k0;
  }
  __device__ __forceinline__ void load_full(int64_t k0) {
#pragma unroll
    for (int i = 0; i < V; ++i) r[i] = *(const uint4*)at(i, k0);
  }
  __device__ __forceinline__ void load_tail(int64_t k0, int64_t K) {
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const uint16_t* q = at(i, k0);
      const int64_t gk = k0 + kc;
      union {
        uint4 u;
        uint16_t h[8];
      } t;
#pragma unroll
      for (int e = 0; e < 8; ++e) t.h[e] = (gk + e < K) ? q[e] : (uint16_t)0;
      r[i] = t.u;
    }
  }
  __device__ __forceinline__ void store(uint16_t* lds) const {
    uint16_t* d = lds + (threadIdx.x >> 3) * PITCH + kc;
#pragma unroll
    for (int i = 0; i < V; ++i) *(uint4*)(d + i * RS * PITCH) = r[i];
  }
};

// int8 rows: ROWS x 64 bytes = ROWS*4 vectors of 16 values per tile, widened
// to T (bf16 or f16, exact) when written to LDS (same clamping and tail rules).
template <typename T, int ROWS, int NT>
struct Tile8 {
  static constexpr int V = ROWS * 4 / NT;
  static constexpr int RS = NT / 4;
  const int8_t* base;
  int64_t ld, last, row0;
  int kc;
  uint4 r[V];
  __device__ __forceinline__ void init(const int8_t* b, int64_t ld_, int64_t rows, int64_t r0) {
    base = b;
    ld = ld_;
    last = rows - 1;
    row0 = r0 + (threadIdx.x >> 2);
    kc = (threadIdx.x & 3) * 16;
  }
  __device__ __forceinline__ const int8_t* at(int i, int64_t k0) const {
    const int64_t gr = min(row0 + (int64_t)i * RS, last);
    return base + gr * ld + kc + k0;
  }
  __device__ __forceinline__ void load_full(int64_t k0) {
#pragma unroll
    for (int i = 0; i < V; ++i) r[i] = *(const uint4*)at(i, k0);
  }
  __device__ __forceinline__ void load_tail(int64_t k0, int64_t K) {
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int8_t* q = at(i, k0);
      const int64_t gk = k0 + kc;
      union {
        uint4 u;
        int8_t b[16];
      } t;
#pragma unroll
      for (int e = 0; e < 16; ++e) t.b[e] = (gk + e < K) ? q[e] : (int8_t)0;
      r[i] = t.u;
    }
  }
  __device__ __forceinline__ void store(uint16_t* lds) const {
    uint16_t* d = lds + (threadIdx.x >> 2) * PITCH + kc;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      union {
        uint4 u;
        int8_t b[16];
      } in;
      in.u = r[i];
      typedef typename MfmaOp<T>::vec vec;
      *(vec*)(d + i * RS * PITCH) = widen8<T>(u32x2_t{in.u.x, in.u.y});
      *(vec*)(d + i * RS * PITCH + 8) = widen8<T>(u32x2_t{in.u.z, in.u.w});
    }
  }
};

template <typename T, int BM, int BN, int WM, int WN, bool B_INT8, bool HAS_BIAS>
__global__ __launch_bounds__(64 * WM * WN, 1) void gemm_mfma_kernel(GemmArgs p) {
  constexpr int NT = 64 * WM * WN;
  constexpr int TM = BM / WM, TN = BN / WN;  // per-wave sub-tile
  constexpr int FM = TM / 32, FN = TN / 32;  // MFMA tiles per wave
  typedef typename MfmaOp<T>::vec vec;
  extern __shared__ __align__(16) uint16_t smem[];
  // stage s: A at smem + s*BM*PITCH, B at smem + 2*BM*PITCH + s*BN*PITCH
  auto As = [&](int s) { return smem + s * BM * PITCH; };
  auto Bs = [&](int s) { return smem + 2 * BM * PITCH + s * BN * PITCH; };

  int tm, tn;
  tile_of(blockIdx.x, p.tiles_m, p.tiles_n, &tm, &tn);
  const int64_t batch = blockIdx.y;
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int lrow = lane & 31, lk = (lane >> 5) * 8;

  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x16{};

  Tile16<BM, NT> ta;
  typename std::conditional<B_INT8, Tile8<T, BN, NT>, Tile16<BN, NT>>::type tb;
  ta.init(p.a + batch * p.sa, p.lda, p.M, m0);
  if constexpr (B_INT8)
    tb.init((const int8_t*)p.b + batch * p.sb, p.ldb, p.N, n0);
  else
    tb.init((const uint16_t*)p.b + batch * p.sb, p.ldb, p.N, n0);

  // MFMAs over one LDS stage, operand fragments double-buffered across the
  // four 16-deep substeps.
  auto compute = [&](int st) {
    const uint16_t* a_s = As(st) + (wm * TM + lrow) * PITCH + lk;
    const uint16_t* b_s = Bs(st) + (wn * TN + lrow) * PITCH + lk;
    vec af[2][FM], bf[2][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i) af[0][i] = *(const vec*)(a_s + i * 32 * PITCH);
#pragma unroll
    for (int j = 0; j < FN; ++j) bf[0][j] = *(const vec*)(b_s + j * 32 * PITCH);
#pragma unroll
    for (int s = 0; s < BK / 16; ++s) {
      const int c = s & 1;
      if (s + 1 < BK / 16) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
          af[c ^ 1][i] = *(const vec*)(a_s + i * 32 * PITCH + (s + 1) * 16);
#pragma unroll
        for (int j = 0; j < FN; ++j)
          bf[c ^ 1][j] = *(const vec*)(b_s + j * 32 * PITCH + (s + 1) * 16);
      }
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = MfmaOp<T>::mma(af[c][i], bf[c][j], acc[i][j]);
    }
  };

  // Steps 0 .. KF-1 are full 64-deep steps, step KF (if K % 64) is partial.
  // The main loop only ever prefetches full steps, so it has no branch.
  const int KF = (int)(p.K / BK);
  const bool tail = KF * (int64_t)BK < p.K;
  if (KF > 0) {
    ta.load_full(0);
    tb.load_full(0);
  } else {
    ta.load_tail(0, p.K);
    tb.load_tail(0, p.K);
  }
  ta.store(As(0));
  tb.store(Bs(0));
  __syncthreads();
  int kt = 0;
  for (; kt + 1 < KF; ++kt) {
    ta.load_full((int64_t)(kt + 1) * BK);
    tb.load_full((int64_t)(kt + 1) * BK);
    // keep the next step's global loads issued ahead of this step's MFMAs
    // (the scheduler would otherwise sink them next to their LDS stores and
    // expose their latency)
    __builtin_amdgcn_sched_barrier(0);
    compute(kt & 1);
    ta.store(As((kt + 1) & 1));
    tb.store(Bs((kt + 1) & 1));
    __syncthreads();
  }
  if (tail && KF > 0) {
    ta.load_tail((int64_t)KF * BK, p.K);
    tb.load_tail((int64_t)KF * BK, p.K);
    compute(kt & 1);
    ta.store(As((kt + 1) & 1));
    tb.store(Bs((kt + 1) & 1));
    __syncthreads();
    ++kt;
  }
  compute(kt & 1);

  // epilogue: out = alpha * acc (* scale[n]) + beta * bias, rounded once.  The
  // bias is fp32 or of the output's type (the host converts anything else).
  uint16_t* C = p.c + batch * p.sc;
  const bool bias_f32 = p.bias_dtype == MI_F32;
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int64_t n = n0 + wn * TN + j * 32 + lrow;
    if (n >= p.N) continue;
    const int64_t bcol = batch * p.bias_sb + n * p.bias_sn;
    const float colscale = B_INT8 ? p.alpha * p.scale[n] : p.alpha;
    // a bias broadcast over rows: one load per column
    const bool row_bias = HAS_BIAS && p.bias_sm == 0;
    float bcolv = 0.f;
    if (row_bias)
      bcolv = bias_f32 ? ((const float*)p.bias)[bcol] : MfmaOp<T>::load(((const uint16_t*)p.bias)[bcol]);
#pragma unroll
    for (int i = 0; i < FM; ++i) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t m = m0 + wm * TM + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        if (m < p.M) {
          float v = colscale * acc[i][j][r];
          if (HAS_BIAS) {
            float bv = bcolv;
            if (!row_bias) {
              const int64_t bo = bcol + m * p.bias_sm;
              bv = bias_f32 ? ((const float*)p.bias)[bo] : MfmaOp<T>::load(((const uint16_t*)p.bias)[bo]);
            }
            v += p.beta * bv;
          }
          C[m * p.ldc + n] = MfmaOp<T>::store(v);
        }
      }
    }
  }
}

// ---- int8 weight-only linear, mid-size M (64 < M <= 512): 128 x R tiles -------------
//
// (Runs where split-K over 256 x 256 tiles does not apply: a single K step,
// or enough tiles to fill the CUs; the sizes below are config 4's, which
// split-K now runs faster.)
// Config 4's M = 256 against W [11008, 4096] has 2 x 11008 / 256 = 86 W rows
// per CU: 128 x 256 tiles give 86 blocks, 128 x 64 tiles 344 (1.34 waves).
// Here a 256-lane block owns 128 rows of x (32 per wave) and R W rows, R a
// multiple of 8 up to 96 chosen so that the blocks about fill the CUs (R = 88
// for config 4: 252 blocks).  K steps of 64 flow through four LDS stages
// filled by global_load_lds (three steps in flight while one is multiplied:
// one block per CU has no other block to cover the latency): x rows as bf16
// (128-byte rows, chunk swizzle dl_swz), W rows as int8 (64-byte rows,
// dl_swz64), which waves 0..2 widen, 32 rows each, into one of two bf16
// copies (dl_swz) once their own copies of the next step have landed.
// (Measured on config 4's M = 256: 49 us, against 54-56 us for the 128 x 64
// register-staged tiles; two stages 53 us; widening spread over all four
// waves, or two steps ahead through a third copy with five stages, 53-58 us.
// The kernel stays far from its 11.7 us MFMA time: per K step its four waves
// stall on the barrier, the widening and the fragment reads in turn.)
// Each wave multiplies its 32 x rows with three 32-row W fragments
// (v_mfma_f32_32x32x16, W as the A operand, so a lane owns one output row and
// runs of 4 columns); the epilogue applies alpha, the per-column scale and
// the bias, rounds once and stores through LDS.
// cache policy operand of global_load_lds on gfx950: non-temporal (NT = bit 1)
constexpr int kCpolNT = 2;

namespace mid {
constexpr int BM = 128, BNF = 96, KB = 64, NT = 256, NW = 4;
constexpr int STAGES = 4;                     // copies in flight: steps kt + 1 .. kt + 3
constexpr int COPIES = 2;                     // bf16 W copies (steps kt, kt + 1)
constexpr int FN = BNF / 32;                  // W fragments per wave
constexpr int TA = BM * KB;                   // x tile, 16-bit elements
constexpr int TB8 = BNF * KB / 2;             // int8 W tile, in 16-bit units
constexpr int TB = BNF * KB;                  // bf16 copy of the W tile
constexpr int STAGE = TA + TB8;               // the part global_load_lds fills
constexpr int NQA = BM * KB * 2 / 1024 / NW;  // x copies per wave (4)
constexpr int NQB = 2;                        // W copies per wave 0..2 (16 rows each)
constexpr int KS = KB / 16;
constexpr int EP = BNF + 8;                   // epilogue row pitch
constexpr size_t LDS = ((size_t)STAGES * STAGE + (size_t)COPIES * TB) * 2;
static_assert(LDS >= (size_t)NW * 32 * EP * 2, "epilogue staging fits");
static_assert(LDS <= 160 * 1024, "one block's LDS");
}  // namespace mid

template <typename T, bool HAS_BIAS>
__global__ __launch_bounds__(mid::NT, 1) void int8_mid_kernel(GemmArgs p, int R) {
  using namespace mid;
  typedef typename MfmaOp<T>::vec vec;
  extern __shared__ __align__(16) uint16_t smem[];
  // XCD-aware order (round-robin dispatch over 8 XCDs): consecutive logical
  // blocks, the m tiles of one W panel first, run on one XCD and share the
  // panel through its L2
  int id = blockIdx.x;
  {
    const int total = p.tiles_m * p.tiles_n;
    if (total % 8 == 0) id = (id % 8) * (total / 8) + id / 8;
  }
  const int tm = id % p.tiles_m, tn = id / p.tiles_m;
  const int M = (int)p.M, N = (int)p.N, K = (int)p.K;
  const int m0 = tm * BM, n0 = tn * R;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool w_rows = wave < BNF / 32;  // waves copying and widening W rows
  const char* Bbase = (const char*)p.b;

  // per-lane byte offsets (the host checked they fit 32 bits); rows past the
  // matrix are clamped to its last row and only feed outputs never stored
  uint32_t ao[NQA], bo[NQB];
#pragma unroll
  for (int q = 0; q < NQA; ++q) {
    const int row = (wave * NQA + q) * 8 + lane / 8;
    ao[q] = (uint32_t)(((int64_t)min(m0 + row, M - 1) * p.lda + dl_swz(row, lane % 8) * 8) * 2);
  }
#pragma unroll
  for (int q = 0; q < NQB; ++q) {
    const int row = (wave * NQB + q) * 16 + lane / 4;
    bo[q] = (uint32_t)((int64_t)min(n0 + row, N - 1) * p.ldb + dl_swz64(row, lane % 4) * 16);
  }
  auto issue = [&](int st, int k0) __attribute__((always_inline)) {
    uint16_t* as = smem + st * STAGE;
    uint16_t* bs = as + TA;
    const char* Ab = (const char*)(p.a + k0);
    const char* Bb = Bbase + k0;
#pragma unroll
    for (int q = 0; q < NQA; ++q)
      __builtin_amdgcn_global_load_lds((const void*)(Ab + ao[q]),
                                       (lds_void_t*)(as + (wave * NQA + q) * 512), 16, 0, 0);
    if (w_rows) {
      // W is streamed once (non-temporal: it should not push x out of L2)
#pragma unroll
      for (int q = 0; q < NQB; ++q)
        __builtin_amdgcn_global_load_lds((const void*)(Bb + bo[q]),
                                         (lds_void_t*)(bs + (wave * NQB + q) * 512), 16, 0, kCpolNT);
    }
  };
  // wave w < 3 copied W rows 32 w .. 32 w + 31 of every stage itself and
  // widens exactly those rows into a bf16 copy; lane: row 32 w + l / 2, k half l % 2
  auto convert = [&](int st, int cb) __attribute__((always_inline)) {
    if (w_rows) {
      const char* b8 = (const char*)(smem + st * STAGE + TA);
      uint16_t* bb = smem + STAGES * STAGE + cb * TB;
      const int r = wave * 32 + (lane >> 1), h = lane & 1;
      const u32x4_t c0 = *(const u32x4_t*)(b8 + r * 64 + dl_swz64(r, 2 * h) * 16);
      const u32x4_t c1 = *(const u32x4_t*)(b8 + r * 64 + dl_swz64(r, 2 * h + 1) * 16);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const u32x4_t& c = j < 2 ? c0 : c1;
        const u32x2_t w = {c[2 * (j & 1)], c[2 * (j & 1) + 1]};
        *(vec*)(bb + r * KB + dl_swz(r, 4 * h + j) * 8) = widen8<T>(w);
      }
    }
  };
  // fragment read offsets: lane supplies row l % 32, k chunk 2 s + l / 32
  int roff[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) roff[s] = (lane & 31) * KB + dl_swz(lane & 31, 2 * s + (lane >> 5)) * 8;

  f32x16 acc[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) acc[j] = f32x16{};
  vec af[2], bfr[2][FN];
  auto read_frags = [&](int st, int cb, int s, int buf) __attribute__((always_inline)) {
    af[buf] = *(const vec*)(smem + st * STAGE + wave * 32 * KB + roff[s]);
    const uint16_t* bs = smem + STAGES * STAGE + cb * TB + roff[s];
#pragma unroll
    for (int j = 0; j < FN; ++j) bfr[buf][j] = *(const vec*)(bs + j * 32 * KB);
  };
  auto mfmas = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[j] = MfmaOp<T>::mma(bfr[buf][j], af[buf], acc[j]);
  };
  const int KT = K / KB;
  // this wave's copies of a step: the wait until step kt + 1 has landed
  // while `later` newer steps stay in flight
  auto wait_step = [&](int later) __attribute__((always_inline)) {
    if (w_rows) wait_later<STAGES - 1, NQA + NQB>(later);
    else wait_later<STAGES - 1, NQA>(later);
  };
  // One K step kt: x from stage kt % STAGES, W from bf16 copy kt % 2.  At
  // its last K substep step kt + 1 is waited for (steps kt + 2 .. kt +
  // STAGES - 1 stay in flight), widened, published by the barrier (which
  // also retires stage kt % STAGES, refilled with step kt + STAGES) and its
  // first fragments read.
  auto step = [&](int kt) __attribute__((always_inline)) {
    const int st = kt % STAGES, cb = kt & 1;
    const int st1 = (kt + 1) % STAGES, cb1 = cb ^ 1;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int buf = s & 1;
      if (s + 1 < KS) {
        read_frags(st, cb, s + 1, buf ^ 1);
        mfmas(buf);
        // MFMA, two fragment reads, then MFMA and one read each
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
        for (int k = 1; k < FN; ++k) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
      } else {
        if (kt + 1 < KT) {
          wait_step(min(STAGES - 2, KT - 2 - kt));
          convert(st1, cb1);
          __syncthreads();
          if (kt + STAGES < KT) issue(st, (kt + STAGES) * KB);
          read_frags(st1, cb1, 0, buf ^ 1);
        }
        mfmas(buf);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

#pragma unroll
  for (int s = 0; s < STAGES; ++s)
    if (s < KT) issue(s, s * KB);
  // step 0 has landed once only steps 1 .. STAGES - 1 (those that exist) are in flight
  wait_step(min(STAGES, KT) - 1);
  convert(0, 0);
  __syncthreads();
  read_frags(0, 0, 0, 0);
  for (int kt = 0; kt < KT; ++kt) step(kt);

  // epilogue: out = alpha * scale[n] * acc + beta * bias, one rounding,
  // staged per wave as [32 x rows][96 W rows] and stored in 16-byte pieces
  __syncthreads();
  uint16_t* es = smem + wave * 32 * EP;
  const float alpha = p.alpha, beta = p.beta;
  const bool bias_f32 = p.bias_dtype == MI_F32;
  const int ml = lane & 31;
  const int64_t m = m0 + wave * 32 + ml;
  // the per-column scale (and a bias broadcast over rows) four columns per load
  const bool row_bias = HAS_BIAS && p.bias_sm == 0;
#pragma unroll
  for (int j = 0; j < FN; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int nl = j * 32 + 8 * g + 4 * (lane >> 5);
      const f32x4_t sc4 = load_col4_t<T>(p.scale, MI_F32, n0 + nl, 1, p.N, 0);
      f32x4_t bb4 = {};
      if (row_bias) bb4 = load_col4_t<T>(p.bias, p.bias_dtype, n0 + nl, p.bias_sn, p.N, 0);
      u16x4_t v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float x = alpha * acc[j][4 * g + e] * sc4[e];
        if (HAS_BIAS) {
          float bv = bb4[e];
          if (!row_bias) {
            const int64_t n = min<int64_t>(n0 + nl + e, p.N - 1);
            const int64_t bo_ = min<int64_t>(m, p.M - 1) * p.bias_sm + n * p.bias_sn;
            bv = bias_f32 ? ((const float*)p.bias)[bo_]
                          : MfmaOp<T>::load(((const uint16_t*)p.bias)[bo_]);
          }
          x += beta * bv;
        }
        v[e] = MfmaOp<T>::store(x);
      }
      *(u16x4_t*)(es + ml * EP + nl) = v;
    }
  // the block's columns: n0 .. n0 + R - 1 (fewer in the last tile)
  const int ncols = min(R, N - n0);
  const bool vec_ok = (p.ldc % 8) == 0 && (((uintptr_t)p.c) & 15) == 0 && (n0 % 8) == 0;
  for (int idx = lane; idx < 32 * (BNF / 8); idx += 64) {
    const int r = idx / (BNF / 8), c = (idx % (BNF / 8)) * 8;
    const int64_t mr = m0 + wave * 32 + r;
    if (mr >= p.M || c >= ncols) continue;
    const uint4 v = *(const uint4*)(es + r * EP + c);
    uint16_t* dst = p.c + mr * p.ldc + n0 + c;
    if (vec_ok && c + 8 <= ncols) {
      *(uint4*)dst = v;
    } else {
      const uint16_t* pv = (const uint16_t*)&v;
      for (int e = 0; e < 8 && c + e < ncols; ++e) dst[e] = pv[e];
    }
  }
}

template <typename T, bool HB>
mi_status_t launch_mid(const GemmArgs& q0, hipStream_t s, const char* what) {
  static bool attr = [] {
    (void)hipFuncSetAttribute((const void*)int8_mid_kernel<T, HB>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)mid::LDS);
    return true;
  }();
  (void)attr;
  GemmArgs q = q0;
  q.tiles_m = (int)((q.M + mid::BM - 1) / mid::BM);
  // W rows per block: a multiple of 8 up to 96, so that the blocks about fill the CUs
  const int64_t want_n = std::max<int64_t>(1, cu_count() / q.tiles_m);
  int64_t R = (q.N + want_n - 1) / want_n;
  R = std::min<int64_t>(mid::BNF, std::max<int64_t>(32, (R + 7) / 8 * 8));
  q.tiles_n = (int)((q.N + R - 1) / R);
  hipLaunchKernelGGL((int8_mid_kernel<T, HB>), dim3((unsigned)(q.tiles_m * q.tiles_n)),
                     dim3(mid::NT), mid::LDS, s, q, (int)R);
  return check_launch(what);
}

template <typename T>
struct Mfma16;
template <>
struct Mfma16<BF16> {
  typedef bf16x8 vec;
  static __device__ __forceinline__ f32x4_t mma(vec a, vec b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mfma16<F16> {
  typedef f16x8 vec;
  static __device__ __forceinline__ f32x4_t mma(vec a, vec b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

// ---- int8 weight-only linear for few rows, weight staged through LDS ------------------
//
// For M <= 64, K % 1024 == 0, 16-byte aligned W rows and enough of them
// (gemm_rows.hip takes the rest): bound by the HBM stream of W.  A 512-lane block owns R consecutive W rows, R = N / CUs rounded up
// (43 for N = 11008 on 256 CUs) and at most 48, so every CU streams the same
// share of W once (with 32-row blocks, 344 blocks on 256 CUs left 88 CUs
// streaming twice the bytes of the others).  K is walked in 1 KiB slabs of
// 48 rows (three 16-row MFMA tiles; rows past R re-read the block's last
// row, an L2 hit, and feed columns that are never stored), and wave w owns
// bytes 128 w .. 128 w + 127 of every slab row: it copies them into its own
// LDS ring by global_load_lds_dwordx4 (one copy = 8 rows x 128 bytes, whole
// cache lines) together with the matching x fragments into registers, and
// multiplies them, so the waves never wait for each other until the final
// combine.  The ring holds three slabs (two slabs of lead on the one being
// multiplied; a wave refills a slot as soon as it has multiplied it).  Lane
// (r, g) reads 16 bytes of row 16 t + r at 64 kp + 16 g (kp = 0, 1), which
// feed two v_mfma_f32_16x16x32 (8 bytes each, widened to bf16 exactly) with
// x as the 16-row operand, x's fragments taken at the same k.  Rows are 128
// bytes in LDS, chunk c of row r stored at c ^ ((r >> 1) & 7) (the copying
// lane fetches the matching global chunk), so the 16 rows of a read pass hit
// 16 distinct 16-byte bank groups.  The 8 waves' partial tiles are added in
// a fixed order through LDS; the epilogue applies the per-column scale and
// bias and rounds once.
constexpr int kStTiles = 3, kStRows = 16 * kStTiles, kStSlab = 1024, kStWaves = 8;
constexpr int kStPart = kStSlab / kStWaves;    // bytes of a slab row per wave (128)
constexpr int kStCopies = kStRows * kStPart / 1024;  // wave copies per slab (6)
constexpr int kStRing = 3;
constexpr int kStWaveLds = kStRing * kStRows * kStPart;  // one wave's ring
constexpr int kStLds = kStWaves * kStWaveLds;
static_assert(kStLds <= 160 * 1024, "slab rings fit the LDS");
static_assert(kStLds >= kStWaves * kStTiles * 16 * 17 * 4, "combine staging fits");

// SFIX > 0 fixes the slab count at compile time (K = 1024 SFIX): the loop is
// then fully unrolled and the compiler can count the loads in flight at
// every step (through the loop's back edge it waits for all of them before
// a step's first MFMA).
template <typename T, int MT, int RING, bool HAS_BIAS, int SFIX>
__global__ __launch_bounds__(64 * kStWaves, 1) void int8_stream_kernel(GemmArgs p, int R) {
  typedef typename Mfma16<T>::vec vec;
  extern __shared__ __align__(16) char st_lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int64_t n0 = (int64_t)blockIdx.x * R;
  const int nrows = (int)min<int64_t>(R, p.N - n0);
  const int S = SFIX > 0 ? SFIX : (int)(p.K / kStSlab);
  char* ring = st_lds + wave * kStWaveLds;
  // copy q moves slab rows 8 q .. 8 q + 7: lane l fetches row 8 q + l / 8, the
  // global chunk that lands at chunk l % 8 of the swizzled row (source rows
  // past the block's nrows re-read its last row)
  const int8_t* wsrc[kStCopies];
#pragma unroll
  for (int q = 0; q < kStCopies; ++q) {
    const int row = 8 * q + (lane >> 3);
    const int c = (lane & 7) ^ ((row >> 1) & 7);
    wsrc[q] = (const int8_t*)p.b + (n0 + min(row, nrows - 1)) * p.ldb + kStPart * wave + 16 * c;
  }
  // x fragment j = 2 kp + h of slab s: row 16 mt + r, k = 1024 s + 128 wave + 64 kp + 16 g + 8 h
  const uint16_t* xrow[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    xrow[mt] = p.a + min<int64_t>(16 * mt + r, p.M - 1) * p.lda + kStPart * wave + 16 * g;
  // slab s: this wave's W copies into ring slot s % RING, then its x fragments
  vec xf[RING][MT][4];
  auto issue = [&](auto B, int s) __attribute__((always_inline)) {
    constexpr int buf = decltype(B)::value;
    char* dst = ring + buf * (kStRows * kStPart);
#pragma unroll
    for (int q = 0; q < kStCopies; ++q)
      __builtin_amdgcn_global_load_lds((const void*)(wsrc[q] + (int64_t)s * kStSlab),
                                       (lds_void_t*)(dst + q * 1024), 16, 0, kCpolNT);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        xf[buf][mt][j] = *(const vec*)(xrow[mt] + (int64_t)s * kStSlab + 64 * (j >> 1) + 8 * (j & 1));
  };
  f32x4_t acc[MT][kStTiles];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < kStTiles; ++t) acc[mt][t] = f32x4_t{};
  // lane (r, g) reads chunk 4 kp + g of row 16 t + r: swizzled by (r >> 1) & 7
  const int rsw = (r >> 1) & 7;
  auto compute = [&](auto B) __attribute__((always_inline)) {
    constexpr int buf = decltype(B)::value;
    const char* wb = ring + buf * (kStRows * kStPart) + r * kStPart;
#pragma unroll
    for (int kp = 0; kp < 2; ++kp)
#pragma unroll
      for (int t = 0; t < kStTiles; ++t) {
        const u32x4_t w16 = *(const u32x4_t*)(wb + t * 16 * kStPart + 16 * ((4 * kp + g) ^ rsw));
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const vec wk = widen8<T>(u32x2_t{w16[2 * h], w16[2 * h + 1]});
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            acc[mt][t] = Mfma16<T>::mma(xf[buf][mt][2 * kp + h], wk, acc[mt][t]);
        }
      }
  };
  // slab s has landed once at most the later slabs' loads (each kStCopies W
  // copies and 4 MT x loads, issued together and in slab order) are
  // outstanding; the copies are this wave's own, so no barrier is needed
  constexpr int PER = kStCopies + 4 * MT;
  auto wait_slab = [&](int later) __attribute__((always_inline)) {
    if (RING > 2 && later >= 2) wait_vmcnt<2 * PER>();
    else if (later >= 1) wait_vmcnt<PER>();
    else wait_vmcnt<0>();
  };
  // one slab step: U = s % RING picks the slot (the loop is unrolled by RING)
  auto step = [&](auto U, int s) __attribute__((always_inline)) {
    wait_slab(min(RING - 1, S - 1 - s));
    compute(U);
    if (s + RING < S) issue(U, s + RING);
  };
  static_assert(RING == 2 || RING == 3, "two or three slabs in flight");
  issue(std::integral_constant<int, 0>{}, 0);
  if (S > 1) issue(std::integral_constant<int, 1>{}, 1);
  if constexpr (RING == 3) {
    if (S > 2) issue(std::integral_constant<int, 2>{}, 2);
  }
  auto round = [&](int s) __attribute__((always_inline)) {
    step(std::integral_constant<int, 0>{}, s);
    if (s + 1 < S) step(std::integral_constant<int, 1>{}, s + 1);
    if constexpr (RING == 3) {
      if (s + 2 < S) step(std::integral_constant<int, 2>{}, s + 2);
    }
  };
  if constexpr (SFIX > 0) {
#pragma unroll
    for (int s = 0; s < SFIX; s += RING) round(s);
  } else {
    for (int s = 0; s < S; s += RING) round(s);
  }
  // fixed-order combine of the 8 waves' partial tiles (the rings are free
  // once every wave is done)
  __syncthreads();
  float(*red)[kStTiles][16][17] = (float(*)[kStTiles][16][17])st_lds;
  const bool bias_f32 = p.bias_dtype == MI_F32;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    if (mt > 0) __syncthreads();
#pragma unroll
    for (int t = 0; t < kStTiles; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[wave][t][4 * g + i][r] = acc[mt][t][i];
    __syncthreads();
    for (int idx = threadIdx.x; idx < kStTiles * 256; idx += 64 * kStWaves) {
      const int tt = idx >> 8, tm = (idx >> 4) & 15, tn = idx & 15;
      const int64_t m = mt * 16 + tm;
      if (m >= p.M || 16 * tt + tn >= nrows) continue;
      const int64_t n = n0 + 16 * tt + tn;
      float sum = red[0][tt][tm][tn];
#pragma unroll
      for (int w = 1; w < kStWaves; ++w) sum += red[w][tt][tm][tn];
      float v = p.alpha * p.scale[n] * sum;
      if (HAS_BIAS) {
        const int64_t bo = m * p.bias_sm + n * p.bias_sn;
        v += p.beta * (bias_f32 ? ((const float*)p.bias)[bo]
                                : MfmaOp<T>::load(((const uint16_t*)p.bias)[bo]));
      }
      p.c[m * p.ldc + n] = MfmaOp<T>::store(v);
    }
  }
}

template <typename T, int MT, bool HB, int SFIX>
mi_status_t launch_stream_k(const GemmArgs& q, hipStream_t s, int R) {
  constexpr int RING = MT <= 2 ? 3 : 2;
  static bool attr = [] {
    (void)hipFuncSetAttribute((const void*)int8_stream_kernel<T, MT, RING, HB, SFIX>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, kStLds);
    return true;
  }();
  (void)attr;
  hipLaunchKernelGGL((int8_stream_kernel<T, MT, RING, HB, SFIX>), dim3((unsigned)ceil_div_u(q.N, R)),
                     dim3(64 * kStWaves), kStLds, s, q, R);
  return check_launch("int8_linear stream");
}

template <typename T, int MT, bool HB>
mi_status_t launch_stream_mt(const GemmArgs& q, hipStream_t s) {
  // rows per block: N / CUs rounded up, at least one tile and at most a slab
  const int64_t cus = std::max(1, cu_count());
  const int R = (int)std::min<int64_t>(kStRows, std::max<int64_t>(16, (q.N + cus - 1) / cus));
  // K = 4096 (a 4096-wide hidden layer) with the slab count fixed
  if (q.K == 4 * kStSlab) return launch_stream_k<T, MT, HB, 4>(q, s, R);
  return launch_stream_k<T, MT, HB, 0>(q, s, R);
}

template <typename T, bool HB>
mi_status_t launch_stream(const GemmArgs& q, hipStream_t s) {
  switch ((int)((q.M + 15) / 16)) {
    case 1: return launch_stream_mt<T, 1, HB>(q, s);
    case 2: return launch_stream_mt<T, 2, HB>(q, s);
    case 3: return launch_stream_mt<T, 3, HB>(q, s);
    default: return launch_stream_mt<T, 4, HB>(q, s);
  }
}

// ---- host side --------------------------------------------------------------------

// A batched matrix view: element (b, r, c) at data + b*sb + r*s0 + c*s1.
struct Mat {
  void* data;
  int dtype;
  int64_t batch, rows, cols;
  int64_t sb, s0, s1;
};

mi_status_t as_mat(const mi_tensor_t* t, const char* name, Mat* m) {
  MI_RETURN_IF(validate(t, name));
  if (t->ndim == 2) {
    *m = Mat{t->data, t->dtype, 1, t->sizes[0], t->sizes[1], 0, t->strides[0], t->strides[1]};
  } else if (t->ndim == 3) {
    *m = Mat{t->data, t->dtype, t->sizes[0], t->sizes[1], t->sizes[2],
             t->sizes[0] == 1 ? 0 : t->strides[0], t->strides[1], t->strides[2]};
  } else {
    MI_FAIL(MI_ERR_INVALID, "%s: expected a 2-D or 3-D tensor, got %d dims", name, t->ndim);
  }
  return MI_OK;
}

mi_tensor_t mat_desc(const Mat& m) {
  mi_tensor_t t{};
  t.data = m.data;
  t.dtype = m.dtype;
  t.ndim = 3;
  t.sizes[0] = m.batch;
  t.sizes[1] = m.rows;
  t.sizes[2] = m.cols;
  t.strides[0] = m.sb;
  t.strides[1] = m.s0;
  t.strides[2] = m.s1;
  return t;
}

// Rows of `m` must be contiguous along the columns, 16-byte aligned, with a
// leading dim that keeps every row 16-byte aligned; otherwise `m` is copied
// densely (leading dim rounded up to 16 bytes) into workspace.
mi_status_t dense_rows(Mat& m, Workspace& ws, hipStream_t stream) {
  const int es = dtype_size(m.dtype);
  const int64_t align_el = 16 / es;
  const bool unit = m.s1 == 1 || m.cols == 1;
  const bool ok = unit && (m.rows == 1 || (m.s0 % align_el == 0 && m.s0 >= m.cols)) &&
                  ((uintptr_t)m.data % 16) == 0 && (m.batch == 1 || m.sb % align_el == 0);
  if (ok) {
    if (m.rows == 1) m.s0 = (m.cols + align_el - 1) / align_el * align_el;
    m.s1 = 1;
    return MI_OK;
  }
  const int64_t ld = (m.cols + align_el - 1) / align_el * align_el;
  MI_RETURN_IF(ws.alloc((size_t)(m.batch * m.rows * ld) * es, stream));
  Mat d{ws.get(), m.dtype, m.batch, m.rows, m.cols, m.rows * ld, ld, 1};
  mi_tensor_t dt = mat_desc(d), st = mat_desc(m);
  MI_RETURN_IF(mi_copy(&dt, &st, (mi_stream_t)stream));
  m = d;
  return MI_OK;
}

Mat transposed(const Mat& m) {
  return Mat{m.data, m.dtype, m.batch, m.cols, m.rows, m.sb, m.s1, m.s0};
}

template <typename T, int BM, int BN, int WM, int WN, bool I8, bool HB>
struct Cfg {
  static void* fn() { return (void*)gemm_mfma_kernel<T, BM, BN, WM, WN, I8, HB>; }
  static size_t lds() { return (size_t)2 * (BM + BN) * PITCH * sizeof(uint16_t); }
  static mi_status_t launch(const GemmArgs& q0, int64_t batch, hipStream_t s, const char* what) {
    static bool attr = [] {
      (void)hipFuncSetAttribute(fn(), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds());
      return true;
    }();
    (void)attr;
    GemmArgs q = q0;
    q.tiles_m = (int)((q.M + BM - 1) / BM);
    q.tiles_n = (int)((q.N + BN - 1) / BN);
    dim3 grid((unsigned)(q.tiles_m * q.tiles_n), (unsigned)batch);
    hipLaunchKernelGGL((gemm_mfma_kernel<T, BM, BN, WM, WN, I8, HB>), grid, dim3(64 * WM * WN),
                       lds(), s, q);
    return check_launch(what);
  }
};

// The direct-to-LDS kernel needs K % 64 == 0, 16-byte aligned rows and
// per-batch byte offsets that fit 32 bits (lane offsets are 32-bit).
bool dl_eligible(const GemmArgs& q, bool int8) {
  const int bes = int8 ? 1 : 2;  // bytes per B element
  if (q.K % dl::BK != 0 || q.K == 0) return false;
  if (q.lda % 8 != 0 || (q.ldb * bes) % 16 != 0) return false;
  if ((((uintptr_t)q.a) | ((uintptr_t)q.b)) & 15) return false;
  if ((q.sa % 8) != 0 || (q.sb * bes) % 16 != 0) return false;
  if (q.M > 0x7fffffff || q.N > 0x7fffffff || q.K > 0x7fffffff) return false;
  const int64_t amax = (q.M - 1) * q.lda * 2 + q.K * 2,
                bmax = ((q.N - 1) * q.ldb + q.K) * bes;
  return amax < ((int64_t)1 << 32) && bmax < ((int64_t)1 << 32);
}

template <typename T, bool HB, bool I8, bool KN = false>
mi_status_t launch_dl(const GemmArgs& q0, int64_t batch, hipStream_t s, const char* what) {
  constexpr size_t lds = I8 ? dl::LDS_BYTES8 : dl::LDS_BYTES;
  static bool attr = [] {
    (void)hipFuncSetAttribute((const void*)gemm_dl_kernel<T, HB, I8, false, KN>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    return true;
  }();
  (void)attr;
  GemmArgs q = q0;
  q.tiles_m = (int)((q.M + dl::BM - 1) / dl::BM);
  q.tiles_n = (int)((q.N + dl::BN - 1) / dl::BN);
  dim3 grid((unsigned)(q.tiles_m * q.tiles_n), (unsigned)batch);
  hipLaunchKernelGGL((gemm_dl_kernel<T, HB, I8, false, KN>), grid, dim3(dl::NT), lds, s, q,
                     nullptr, (int64_t)0);
  return check_launch(what);
}

// Row-major [K][N] B read in place by the large-tile kernel: enough tiles to
// fill the CUs, K % 64 == 0, 16-byte aligned rows of both operands, N a
// multiple of 8 (whole 16-byte column chunks) and 32-bit lane offsets.
// The transposed fragment reads make the main loop about 9 % slower than
// with K-contiguous B (M8192 N4096 K4096: 0.257 against 0.236 ms), while a
// K-contiguous copy of B costs a fixed 2 K N x 2 bytes at about 6 TB/s
// (16 us there, 0.247 ms in all): in place wins while M x batch <= 4096.
bool dl_kn_eligible(const GemmArgs& q, int64_t batch) {
  if (q.M * batch > 4096) return false;
  const int64_t tiles = ((q.M + dl::BM - 1) / dl::BM) * ((q.N + dl::BN - 1) / dl::BN) * batch;
  if (tiles < cu_count()) return false;
  if (q.K % dl::BK != 0 || q.K == 0 || q.N % 8 != 0 || q.N < 8) return false;
  if (q.lda % 8 != 0 || q.ldb % 8 != 0 || q.ldb < q.N) return false;
  if ((((uintptr_t)q.a) | ((uintptr_t)q.b)) & 15) return false;
  if ((q.sa % 8) != 0 || (q.sb % 8) != 0) return false;
  if (q.M > 0x7fffffff || q.N > 0x7fffffff || q.K > 0x7fffffff) return false;
  const int64_t amax = (q.M - 1) * q.lda * 2 + q.K * 2, bmax = (dl::BK * q.ldb + q.N) * 2;
  return amax < ((int64_t)1 << 32) && bmax < ((int64_t)1 << 32);
}

// ---- split-K over 256 x 256 tiles, for too few tiles to fill the CUs ----------------
//
// The int8 linear at M = 256 has 43 tiles of 256 x 256 for 256 CUs.  With S
// K slices per tile (one block per CU, S = 5 there) each block keeps the
// large tile's low LDS traffic per MFMA, which 128-row tiles over the whole
// K cannot (every CU would copy all of x into LDS); the price is the fp32
// partial sums, written once and read once by the combine (M = 256: 34.5 us
// for the slices, 10.5 us for the combine of 56 MB).
//
// out = alpha * scale[n] * sum_s part[s] + beta * bias, the slices added in
// order s = 0 .. S - 1 (deterministic) and rounded once.  One lane per run
// of 4 columns of a row.
template <typename T, bool HAS_BIAS>
__global__ __launch_bounds__(256) void splitk_combine_kernel(GemmArgs p, const float* part, int S,
                                                             int64_t ldp) {
  const int64_t runs = ldp / 4;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t m = idx / runs, n = (idx - m * runs) * 4;
  if (m >= p.M || n >= p.N) return;
  const float* src = part + m * ldp + n;
  const int64_t slice = p.M * ldp;
  f32x4_t acc = *(const f32x4_t*)src;
#pragma unroll 4
  for (int s = 1; s < S; ++s) acc += *(const f32x4_t*)(src + s * slice);
  f32x4_t sc4 = {1.f, 1.f, 1.f, 1.f}, bb4 = {};
  if (p.scale != nullptr) sc4 = load_col4_t<T>(p.scale, MI_F32, n, 1, p.N, 0);
  const bool row_bias = HAS_BIAS && p.bias_sm == 0;
  if (row_bias) bb4 = load_col4_t<T>(p.bias, p.bias_dtype, n, p.bias_sn, p.N, 0);
  u16x4_t v;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float x = p.alpha * acc[e] * sc4[e];
    if (HAS_BIAS) {
      float bv = bb4[e];
      if (!row_bias) {
        const int64_t bo = m * p.bias_sm + min<int64_t>(n + e, p.N - 1) * p.bias_sn;
        bv = p.bias_dtype == MI_F32 ? ((const float*)p.bias)[bo]
                                    : MfmaOp<T>::load(((const uint16_t*)p.bias)[bo]);
      }
      x += p.beta * bv;
    }
    v[e] = MfmaOp<T>::store(x);
  }
  uint16_t* dst = p.c + m * p.ldc + n;
  if (n + 3 < p.N && (p.ldc % 4) == 0 && (((uintptr_t)p.c) & 7) == 0) {
    *(u16x4_t*)dst = v;
  } else {
    for (int e = 0; e < 4 && n + e < p.N; ++e) dst[e] = v[e];
  }
}

// Slices for split-K over 256 x 256 tiles: as many as fill the CUs with one
// block each (at least 2, at most one 64-wide K step per slice); 1 = no split.
int splitk_slices(const GemmArgs& q) {
  const int64_t tiles = ((q.M + dl::BM - 1) / dl::BM) * ((q.N + dl::BN - 1) / dl::BN);
  const int64_t s = std::min<int64_t>(cu_count() / std::max<int64_t>(tiles, 1), q.K / dl::BK);
  return s >= 2 ? (int)std::min<int64_t>(s, 16) : 1;
}

// Above 512 rows the slices have to beat 128 x 64 tiles over the whole K, by cost
// in us: those take 0.42 us a K step, 0.7 where K is long, or 0.45 per block and
// CU; a slice 1.3 us a step, and its partial sums go through the caches.  A fit to
// 356 shapes (M 513 .. 4096, N 256 .. 8192, K 64 .. 8192; 0.7 % from the faster of
// the two on average, 8 % at worst): M600 N1024 K1024 12.4 us whole, 25.5 in 16
// slices; M2000 N1024 K4096 48.2 and 42.2; M3500 N2048 K4096 108 and 77.
bool slices_pay(const GemmArgs& q, int S) {
  const int64_t blocks = ((q.M + 127) / 128) * ((q.N + 63) / 64), steps = q.K / dl::BK;
  const float step = std::max(q.K <= 2240 ? 0.42f : 0.7f, 0.45f * (float)blocks / (float)cu_count());
  const float sliced = 14.f + 1.3f * (float)((steps + S - 1) / S) +
                       (float)S * (float)q.M * (float)q.N * (8.f / 8.5e6f);
  return sliced < 5.f + step * (float)steps;
}

template <typename T, bool HB>
mi_status_t combine(const GemmArgs& q, const float* part, int S, int64_t ldp, hipStream_t s,
                    const char* what) {
  hipLaunchKernelGGL((splitk_combine_kernel<T, HB>), dim3(ceil_div_u(q.M * (ldp / 4), 256)),
                     dim3(256), 0, s, q, part, S, ldp);
  return check_launch(what);
}

template <typename T, bool HB, bool I8>
mi_status_t launch_splitk(const GemmArgs& q0, int S, hipStream_t s, const char* what) {
  constexpr size_t lds = I8 ? dl::LDS_BYTES8 : dl::LDS_BYTES;
  static bool attr = [] {
    (void)hipFuncSetAttribute((const void*)gemm_dl_kernel<T, false, I8, true>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    return true;
  }();
  (void)attr;
  GemmArgs q = q0;
  q.tiles_m = (int)((q.M + dl::BM - 1) / dl::BM);
  q.tiles_n = (int)((q.N + dl::BN - 1) / dl::BN);
  const int64_t ldp = (q.N + 3) / 4 * 4;
  Workspace wp;
  MI_RETURN_IF(wp.alloc((size_t)S * (size_t)q.M * (size_t)ldp * sizeof(float), s));
  float* part = (float*)wp.get();
  hipLaunchKernelGGL((gemm_dl_kernel<T, false, I8, true>),
                     dim3((unsigned)(q.tiles_m * q.tiles_n), (unsigned)S), dim3(dl::NT), lds, s, q,
                     part, ldp);
  MI_RETURN_IF(check_launch(what));
  return combine<T, HB>(q, part, S, ldp, s, what);
}

template <typename T, bool I8, bool HB>
mi_status_t launch_mfma(const GemmArgs& q, int64_t batch, hipStream_t s, const char* what) {
  // int8 W and 64 < M: split-K over 256 x 256 tiles when they are too few to fill
  // the CUs (M = 256: 43 tiles x 5 K slices, 43.6 us against 49.9 us for 128-row
  // tiles over the whole K; M = 96 .. 512 all faster; M2862 N2240 K4032, 108
  // tiles x 2: 75 us against 107), else 128-row tiles sized to the CUs
  if (I8 && batch == 1 && q.M > 64 && dl_eligible(q, true)) {
    const int S = splitk_slices(q);
    if (S > 1 && (q.M <= 4 * mid::BM || slices_pay(q, S))) {
      const mi_status_t st = launch_splitk<T, HB, true>(q, S, s, what);
      if (st != MI_ERR_WORKSPACE && st != MI_ERR_TOO_LARGE) return st;
      clear_error();  // no room for the partial sums: the whole K in one block
    }
    if (q.M <= 4 * mid::BM) return launch_mid<T, HB>(q, s, what);
  }
  if constexpr (!I8) {
    // tile shape and K slices by gemm_mid.hip's cost rule
    if (gemm_mid_eligible(q))
      return launch_gemm_mid(q, batch, std::is_same<T, F16>::value, HB, s, what);
    // byte offsets beyond 32 bits
    return Cfg<T, 128, 128, 2, 2, false, HB>::launch(q, batch, s, what);
  } else {
    const int64_t cus = cu_count();
    const int64_t big = ((q.M + 255) / 256) * ((q.N + 255) / 256) * batch;
    // (too many tiles to slice: from half the CUs on, M3000 N4096 K4096 on 192
    // tiles 102 us against 162 on 128 x 64 ones)
    if (big >= cus / 2 && dl_eligible(q, true)) return launch_dl<T, HB, true>(q, batch, s, what);
    if (big >= cus) return Cfg<T, 256, 256, 2, 4, true, HB>::launch(q, batch, s, what);
    // 128 x 64 tiles: twice the blocks of 128 x 128, so CUs hold two and overlap
    // one's loads with the other's MFMAs (about 15 % faster at M = 256)
    return Cfg<T, 128, 64, 2, 2, true, HB>::launch(q, batch, s, what);
  }
}

template <typename T>
mi_status_t dispatch_mfma(const GemmArgs& q, bool int8, bool has_bias, int64_t batch,
                          hipStream_t s, const char* what) {
  if (int8) {
    if (has_bias) return launch_mfma<T, true, true>(q, batch, s, what);
    return launch_mfma<T, true, false>(q, batch, s, what);
  }
  if (has_bias) return launch_mfma<T, false, true>(q, batch, s, what);
  return launch_mfma<T, false, false>(q, batch, s, what);
}

struct BiasView {
  const void* data = nullptr;
  int dtype = MI_F32;
  int64_t sb = 0, sm = 0, sn = 0;
};

mi_status_t bias_view(const mi_tensor_t* bias, int64_t batch, int64_t M, int64_t N,
                      const char* what, BiasView* bv) {
  MI_RETURN_IF(validate(bias, "bias"));
  MI_CHECK_ARG(bias->ndim <= 3, "%s: bias has too many dims", what);
  int64_t sz[3] = {1, 1, 1}, st[3] = {0, 0, 0};
  const int off = 3 - bias->ndim;
  for (int d = 0; d < bias->ndim; ++d) {
    sz[off + d] = bias->sizes[d];
    st[off + d] = bias->sizes[d] == 1 ? 0 : bias->strides[d];
  }
  MI_CHECK_ARG((sz[0] == 1 || sz[0] == batch) && (sz[1] == 1 || sz[1] == M) &&
                   (sz[2] == 1 || sz[2] == N),
               "%s: bias does not broadcast to the output", what);
  bv->data = bias->data;
  bv->dtype = bias->dtype;
  bv->sb = st[0];
  bv->sm = st[1];
  bv->sn = st[2];
  return MI_OK;
}

// Converts a bias of a dtype the epilogue does not read into a dense fp32
// copy in workspace (same shape, so the broadcast view is unchanged).
mi_status_t bias_to_f32(const mi_tensor_t* bias, Workspace& ws, hipStream_t stream,
                        BiasView* bv) {
  mi_tensor_t dst = *bias;
  MI_RETURN_IF(ws.alloc((size_t)numel(*bias) * 4, stream));
  dst.data = ws.get();
  dst.dtype = MI_F32;
  int64_t s = 1;
  for (int d = dst.ndim - 1; d >= 0; --d) {
    dst.strides[d] = s;
    s *= dst.sizes[d];
  }
  MI_RETURN_IF(mi_copy(&dst, bias, (mi_stream_t)stream));
  int64_t st[3] = {0, 0, 0};
  const int off = 3 - dst.ndim;
  for (int d = 0; d < dst.ndim; ++d) st[off + d] = dst.sizes[d] == 1 ? 0 : dst.strides[d];
  bv->data = ws.get();
  bv->dtype = MI_F32;
  bv->sb = st[0];
  bv->sm = st[1];
  bv->sn = st[2];
  return MI_OK;
}

// out[b] = beta * bias[b] + alpha * a[b] @ b[b]; `wt` (when not NULL) is an
// int8 weight [N, K] with per-N fp32 `scale`, used instead of `b`.
mi_status_t run_gemm(const mi_tensor_t* out, const mi_tensor_t* a, const mi_tensor_t* b,
                     const mi_tensor_t* wt, const mi_tensor_t* scale, const mi_tensor_t* bias,
                     double alpha, double beta, hipStream_t stream, const char* what) {
  clear_error();
  Mat A, B, C;
  const bool int8 = wt != nullptr;
  MI_RETURN_IF(as_mat(a, "mat1", &A));
  if (int8) {
    MI_RETURN_IF(as_mat(wt, "weight", &B));
    MI_CHECK_ARG(B.batch == 1 && wt->ndim == 2, "%s: weight must be 2-D [N, K]", what);
    MI_CHECK_ARG(B.dtype == MI_I8, "%s: weight must be int8", what);
    B = transposed(B);  // [K, N] view of the weight
  } else {
    MI_RETURN_IF(as_mat(b, "mat2", &B));
  }
  MI_RETURN_IF(as_mat(out, "out", &C));
  MI_CHECK_ARG(A.dtype == C.dtype && (int8 || B.dtype == A.dtype),
               "%s: expected operands and out of one dtype, got %s, %s, %s", what,
               dtype_name(A.dtype), dtype_name(B.dtype), dtype_name(C.dtype));
  MI_CHECK_ARG(A.dtype == MI_BF16 || A.dtype == MI_F16 || (A.dtype == MI_F32 && !int8),
               "%s: dtype %s is not supported", what, dtype_name(A.dtype));
  MI_CHECK_ARG(A.cols == B.rows,
               "%s: mat1 and mat2 shapes cannot be multiplied (%lldx%lld and %lldx%lld)", what,
               (long long)A.rows, (long long)A.cols, (long long)B.rows, (long long)B.cols);
  const int64_t batch = std::max(A.batch, std::max(B.batch, C.batch));
  MI_CHECK_ARG((A.batch == batch || A.batch == 1) && (B.batch == batch || B.batch == 1) &&
                   C.batch == batch,
               "%s: batch sizes differ", what);
  MI_CHECK_ARG(C.rows == A.rows && C.cols == B.cols,
               "%s: out has shape %lldx%lld, expected %lldx%lld", what, (long long)C.rows,
               (long long)C.cols, (long long)A.rows, (long long)B.cols);
  MI_CHECK_ARG(batch <= 65535, "%s: batch too large", what);
  if (A.batch == 1) A.sb = 0;
  if (B.batch == 1) B.sb = 0;
  A.batch = B.batch = batch;
  const int64_t M = A.rows, N = B.cols, K = A.cols;
  if (int8) {
    MI_RETURN_IF(validate(scale, "scales"));
    MI_CHECK_ARG(scale->dtype == MI_F32 && numel(*scale) == N && is_contiguous(*scale),
                 "%s: scales must be a dense fp32 vector of %lld elements", what, (long long)N);
  }
  if (M == 0 || N == 0 || batch == 0) return MI_OK;
  const bool has_bias = bias != nullptr && bias->data != nullptr && beta != 0.0;
  BiasView bv;
  Workspace wbias;
  if (has_bias) {
    MI_RETURN_IF(bias_view(bias, batch, M, N, what, &bv));
    if (A.dtype != MI_F32 && bv.dtype != MI_F32 && bv.dtype != A.dtype)
      MI_RETURN_IF(bias_to_f32(bias, wbias, stream, &bv));
  }
  if (K == 0) {
    mi_tensor_t ct = mat_desc(C);
    mi_scalar_t z{};
    z.dtype = MI_F64;
    z.wrapped = 1;
    if (!has_bias) return mi_fill(&ct, z, (mi_stream_t)stream);
    mi_tensor_t bt{};
    bt.data = (void*)bv.data;
    bt.dtype = bv.dtype;
    bt.ndim = 3;
    bt.sizes[0] = batch;
    bt.sizes[1] = M;
    bt.sizes[2] = N;
    bt.strides[0] = bv.sb;
    bt.strides[1] = bv.sm;
    bt.strides[2] = bv.sn;
    mi_scalar_t bs = z;
    bs.f = beta;
    return mi_mul_scalar(&ct, &bt, bs, (mi_stream_t)stream);
  }

  if (A.dtype == MI_F32) {
    MI_CHECK_ARG(C.s1 == 1 || N == 1, "%s: out must have unit column stride", what);
    GemmF32Args q{};
    q.a = (const float*)A.data;
    q.b = (const float*)B.data;
    q.c = (float*)C.data;
    q.bias = bv.data;
    q.bias_dtype = bv.dtype;
    q.bias_sm = bv.sm;
    q.bias_sn = bv.sn;
    q.bias_sb = bv.sb;
    q.M = M;
    q.N = N;
    q.K = K;
    q.a_sm = A.s0;
    q.a_sk = A.s1;
    q.b_sk = B.s0;
    q.b_sn = B.s1;
    q.ldc = C.s0;
    q.sa = A.sb;
    q.sb = B.sb;
    q.sc = C.sb;
    q.alpha = (float)alpha;
    q.beta = (float)beta;
    return launch_gemm_f32(q, batch, has_bias, stream, what);
  }

  // MFMA path: A as [M, K] rows, B as [N, K] rows (B^T with K contiguous),
  // or B as row-major [K, N] rows read in place by the large-tile kernel
  Workspace wa, wb, wc;
  Mat Bt = transposed(B);
  // Few rows: the weight stream kernels.  An int8 weight of whole 1 KiB slabs
  // keeps int8_stream_kernel from N = 32 x CUs.  Against the few-row kernel, us (N 8192
  // .. 32000, K 1024 .. 11264): ahead up to 24 rows on N 9216 .. 11008 (M8 N11008 K4096
  // 9.5 and 12.1, M24 13.9 and 16.1), even at N 8192 or 32 rows (M24 N8192 K4096 13.0
  // and 15.0, M8 9.0 and 8.6), behind with more rows (M64 N11008 K8192 41 and 34) and
  // where its 48-row slabs make an uneven last round (M24 N16384 K4096 24.6 and 17.2);
  // below N = 32 x CUs behind (M8 N4096 K4096 8.1 and 6.7, M64 N4096 K8192 39 and 19).
  // Asked of the operands as they are, and for
  // int8 of the dense copies where those were needed (M8 N4096 K4096, x at a column
  // stride of 2: 46 us on the large-M tiles, 9 so).
  auto few_rows = [&](const Mat& a, const Mat& bt, const Mat& c, mi_status_t* st) {
    if (batch != 1 || M > kRowsMax || (a.s1 != 1 && K != 1) || (bt.s1 != 1 && K != 1) ||
        (c.s1 != 1 && N != 1))
      return false;
    GemmArgs q{};
    q.a = (const uint16_t*)a.data;
    q.b = bt.data;
    q.c = (uint16_t*)c.data;
    q.bias = bv.data;
    q.bias_dtype = bv.dtype;
    q.bias_sm = bv.sm;
    q.bias_sn = bv.sn;
    q.M = M;
    q.N = N;
    q.K = K;
    q.lda = a.s0;
    q.ldb = bt.s0;
    q.ldc = c.s0;
    q.scale = int8 ? (const float*)scale->data : nullptr;
    q.alpha = (float)alpha;
    q.beta = (float)beta;
    const bool f16 = a.dtype == MI_F16;
    if (int8 && K % kStSlab == 0 && N >= 32 * cu_count() && (q.lda % 8 == 0 || M == 1) &&
        q.ldb % 16 == 0 && ((((uintptr_t)q.a) | ((uintptr_t)q.b)) & 15) == 0) {
      if (f16) *st = has_bias ? launch_stream<F16, true>(q, stream) : launch_stream<F16, false>(q, stream);
      else *st = has_bias ? launch_stream<BF16, true>(q, stream) : launch_stream<BF16, false>(q, stream);
      return true;
    }
    // (a short K is over before the waves that share it have paid: M64 N128256 K64
    // 16.4 us here, 10.0 on the tiles of gemm_mid.hip; int8 M64 N28672 K320 12.2 and
    // 9.1 on 128 x 64 ones)
    if (!int8 && M > 32 && K <= 128 && gemm_mid_eligible(q)) return false;
    if (int8 && M > 32 && K <= 768 && N >= 64 * cu_count()) return false;
    if (!gemm_rows_eligible(q)) return false;
    *st = launch_gemm_rows(q, f16, has_bias, stream, what);
    return true;
  };
  mi_status_t few_st;
  if (few_rows(A, Bt, C, &few_st)) return few_st;
  MI_RETURN_IF(dense_rows(A, wa, stream));
  bool b_kn = false;
  if (!int8 && B.s1 == 1 && N > 1 && Bt.s1 != 1) {
    GemmArgs kq{};
    kq.a = (const uint16_t*)A.data;
    kq.b = B.data;
    kq.M = M;
    kq.N = N;
    kq.K = K;
    kq.lda = A.s0;
    kq.ldb = B.s0;
    kq.sa = A.sb;
    kq.sb = B.sb;
    b_kn = dl_kn_eligible(kq, batch);
  }
  if (!b_kn) MI_RETURN_IF(dense_rows(Bt, wb, stream));
  Mat Cw = C;
  const bool c_ok = (C.s1 == 1 || N == 1) && (C.batch == 1 || C.sb != 0);
  if (!c_ok) {
    MI_RETURN_IF(wc.alloc((size_t)(batch * M * N) * 2, stream));
    Cw = Mat{wc.get(), C.dtype, batch, M, N, M * N, N, 1};
  }
  GemmArgs q{};
  q.a = (const uint16_t*)A.data;
  q.b = Bt.data;
  q.c = (uint16_t*)Cw.data;
  q.bias = bv.data;
  q.scale = int8 ? (const float*)scale->data : nullptr;
  q.bias_dtype = bv.dtype;
  q.bias_sm = bv.sm;
  q.bias_sn = bv.sn;
  q.bias_sb = bv.sb;
  q.M = M;
  q.N = N;
  q.K = K;
  q.lda = A.s0;
  q.ldb = Bt.s0;
  q.ldc = Cw.s0;
  q.sa = A.sb;
  q.sb = Bt.sb;
  q.sc = Cw.sb;
  q.alpha = (float)alpha;
  q.beta = (float)beta;
  if (b_kn) {
    q.b = B.data;
    q.ldb = B.s0;
    q.sb = B.sb;
    mi_status_t st;
    if (A.dtype == MI_BF16)
      st = has_bias ? launch_dl<BF16, true, false, true>(q, batch, stream, what)
                    : launch_dl<BF16, false, false, true>(q, batch, stream, what);
    else
      st = has_bias ? launch_dl<F16, true, false, true>(q, batch, stream, what)
                    : launch_dl<F16, false, false, true>(q, batch, stream, what);
    MI_RETURN_IF(st);
    if (!c_ok) {
      mi_tensor_t dst = mat_desc(C), src = mat_desc(Cw);
      MI_RETURN_IF(mi_copy(&dst, &src, (mi_stream_t)stream));
    }
    return MI_OK;
  }
  if (int8 && few_rows(A, Bt, Cw, &few_st)) {
    MI_RETURN_IF(few_st);
  } else if (A.dtype == MI_BF16) {
    MI_RETURN_IF(dispatch_mfma<BF16>(q, int8, has_bias, batch, stream, what));
  } else {
    MI_RETURN_IF(dispatch_mfma<F16>(q, int8, has_bias, batch, stream, what));
  }
  if (!c_ok) {
    mi_tensor_t dst = mat_desc(C), src = mat_desc(Cw);
    MI_RETURN_IF(mi_copy(&dst, &src, (mi_stream_t)stream));
  }
  return MI_OK;
}

// x [M, K] @ W^T with W [N, K] (a linear layer's weight) and a fused
// epilogue: EPI_RESID adds `aux` (residual [M, N]) to the rounded product,
// EPI_SILU multiplies silu(x Wg^T) by x Wu^T (W = Wg, aux = Wu), each product
// rounded first, as the unfused ops do.  One kernel takes the whole op where its
// alignment and 32-bit offset rules hold and gemm_mid.hip's cost rule has it
// faster; otherwise the products go to workspace through the regular matmul and
// the elementwise op follows, with the same results.
mi_status_t run_linear_epi(int epi, const mi_tensor_t* out, const mi_tensor_t* x,
                           const mi_tensor_t* w, const mi_tensor_t* aux, hipStream_t stream,
                           const char* what) {
  clear_error();
  MI_CHECK_ARG(out && x && w && aux, "%s: NULL descriptor", what);
  MI_RETURN_IF(validate(out, "out"));
  MI_RETURN_IF(validate(x, "x"));
  MI_RETURN_IF(validate(w, "weight"));
  MI_RETURN_IF(validate(aux, epi == EPI_SILU ? "w_up" : "residual"));
  MI_CHECK_ARG(x->ndim == 2 && w->ndim == 2 && out->ndim == 2 && aux->ndim == 2,
               "%s: x, weights, residual and out must be 2-D", what);
  const int dt = x->dtype;
  MI_CHECK_ARG(dt == MI_BF16 || dt == MI_F16, "%s: dtype %s is not supported", what,
               dtype_name(dt));
  MI_CHECK_ARG(w->dtype == dt && out->dtype == dt && aux->dtype == dt,
               "%s: x, weights, residual and out must share a dtype", what);
  const int64_t M = x->sizes[0], K = x->sizes[1], N = w->sizes[0];
  MI_CHECK_ARG(w->sizes[1] == K, "%s: x has %lld features, the weight expects %lld", what,
               (long long)K, (long long)w->sizes[1]);
  MI_CHECK_ARG(out->sizes[0] == M && out->sizes[1] == N, "%s: out must be [%lld, %lld]", what,
               (long long)M, (long long)N);
  MI_CHECK_ARG(aux->sizes[0] == (epi == EPI_SILU ? N : M) && aux->sizes[1] == (epi == EPI_SILU ? K : N),
               "%s: %s has the wrong shape", what, epi == EPI_SILU ? "w_up" : "residual");
  if (M == 0 || N == 0) return MI_OK;
  // the fused kernel: unit column strides, enough tiles, the dl kernel's rules
  GemmArgs q{};
  q.a = (const uint16_t*)x->data;
  q.b = w->data;
  q.c = (uint16_t*)out->data;
  q.M = M;
  q.N = N;
  q.K = K;
  q.lda = x->strides[0];
  q.ldb = w->strides[0];
  q.ldc = out->strides[0];
  q.alpha = 1.f;
  q.beta = 0.f;
  // (up to kRowsMax rows the products take the few-row kernel, which adds K in
  // another order)
  bool fused = M > kRowsMax && x->strides[1] == 1 && w->strides[1] == 1 && out->strides[1] == 1 &&
               aux->strides[1] == 1 && K > 0 && dl_eligible(q, false);
  if (epi == EPI_SILU) {
    q.b2 = aux->data;
    fused = fused && aux->strides[0] == q.ldb && ((uintptr_t)aux->data & 15) == 0 &&
            ((N - 1) * q.ldb + K) * 2 < ((int64_t)1 << 32);
  } else {
    q.res = (const uint16_t*)aux->data;
    q.ldr = aux->strides[0];
  }
  mi_status_t st;
  if (fused && launch_gemm_fused(q, epi == EPI_SILU, dt == MI_F16, stream, what, &st)) return st;
  // unfused: the product(s) into workspace, then the elementwise op
  auto wt = [](const mi_tensor_t* t) {  // [K, N] view of a [N, K] weight
    mi_tensor_t v = *t;
    v.sizes[0] = t->sizes[1];
    v.sizes[1] = t->sizes[0];
    v.strides[0] = t->strides[1];
    v.strides[1] = t->strides[0];
    return v;
  };
  mi_tensor_t tmp{};
  tmp.dtype = dt;
  tmp.ndim = 2;
  tmp.sizes[0] = M;
  tmp.sizes[1] = N;
  tmp.strides[0] = N;
  tmp.strides[1] = 1;
  Workspace w1, w2;
  MI_RETURN_IF(w1.alloc((size_t)(M * N) * 2, stream));
  tmp.data = w1.get();
  const mi_tensor_t wv = wt(w);
  MI_RETURN_IF(run_gemm(&tmp, x, &wv, nullptr, nullptr, nullptr, 1.0, 0.0, stream, what));
  if (epi == EPI_RESID) {
    mi_scalar_t one{};
    one.dtype = MI_F64;
    one.f = 1.0;
    one.i = 1;
    one.wrapped = 1;
    return mi_add(out, aux, &tmp, one, (mi_stream_t)stream);
  }
  mi_tensor_t tmp2 = tmp;
  MI_RETURN_IF(w2.alloc((size_t)(M * N) * 2, stream));
  tmp2.data = w2.get();
  const mi_tensor_t uv = wt(aux);
  MI_RETURN_IF(run_gemm(&tmp2, x, &uv, nullptr, nullptr, nullptr, 1.0, 0.0, stream, what));
  return mi_silu_mul(out, &tmp, &tmp2, (mi_stream_t)stream);
}

}  // namespace

mi_status_t launch_splitk_combine(const GemmArgs& q, bool f16, bool has_bias, const float* part,
                                  int S, int64_t ldp, hipStream_t s, const char* what) {
  if (f16)
    return has_bias ? combine<F16, true>(q, part, S, ldp, s, what)
                    : combine<F16, false>(q, part, S, ldp, s, what);
  return has_bias ? combine<BF16, true>(q, part, S, ldp, s, what)
                  : combine<BF16, false>(q, part, S, ldp, s, what);
}

}  // namespace mi

using namespace mi;

extern "C" {

mi_status_t mi_addmm(const mi_tensor_t* out, const mi_tensor_t* self, const mi_tensor_t* mat1,
                     const mi_tensor_t* mat2, double beta, double alpha, mi_stream_t stream) {
  return run_gemm(out, mat1, mat2, nullptr, nullptr, self, alpha, beta, (hipStream_t)stream,
                  "addmm");
}

mi_status_t mi_mm(const mi_tensor_t* out, const mi_tensor_t* self, const mi_tensor_t* mat2,
                  mi_stream_t stream) {
  return run_gemm(out, self, mat2, nullptr, nullptr, nullptr, 1.0, 0.0, (hipStream_t)stream, "mm");
}

mi_status_t mi_bmm(const mi_tensor_t* out, const mi_tensor_t* self, const mi_tensor_t* mat2,
                   mi_stream_t stream) {
  clear_error();
  MI_CHECK_ARG(self && mat2 && out, "bmm: NULL descriptor");
  MI_CHECK_ARG(self->ndim == 3 && mat2->ndim == 3 && out->ndim == 3, "bmm: expected 3-D tensors");
  MI_CHECK_ARG(self->sizes[0] == mat2->sizes[0], "bmm: batch sizes differ");
  return run_gemm(out, self, mat2, nullptr, nullptr, nullptr, 1.0, 0.0, (hipStream_t)stream, "bmm");
}

mi_status_t mi_baddbmm(const mi_tensor_t* out, const mi_tensor_t* self, const mi_tensor_t* batch1,
                       const mi_tensor_t* batch2, double beta, double alpha, mi_stream_t stream) {
  return run_gemm(out, batch1, batch2, nullptr, nullptr, self, alpha, beta, (hipStream_t)stream,
                  "baddbmm");
}

mi_status_t mi_linear_residual(const mi_tensor_t* out, const mi_tensor_t* x,
                               const mi_tensor_t* weight, const mi_tensor_t* residual,
                               mi_stream_t stream) {
  return run_linear_epi(EPI_RESID, out, x, weight, residual, (hipStream_t)stream,
                        "linear_residual");
}

mi_status_t mi_linear_silu_mul(const mi_tensor_t* out, const mi_tensor_t* x,
                               const mi_tensor_t* w_gate, const mi_tensor_t* w_up,
                               mi_stream_t stream) {
  return run_linear_epi(EPI_SILU, out, x, w_gate, w_up, (hipStream_t)stream, "linear_silu_mul");
}

mi_status_t mi_int8_linear(const mi_tensor_t* out, const mi_tensor_t* x, const mi_tensor_t* weight,
                           const mi_tensor_t* scales, const mi_tensor_t* bias, mi_stream_t stream) {
  clear_error();
  MI_CHECK_ARG(out && x && weight && scales, "int8_linear: NULL descriptor");
  MI_CHECK_ARG(x->ndim == 2 && out->ndim == 2, "int8_linear: x and out must be 2-D");
  return run_gemm(out, x, nullptr, weight, scales, bias, 1.0, 1.0, (hipStream_t)stream,
                  "int8_linear");
}

}  // extern "C"
