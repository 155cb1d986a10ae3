// The direct-to-LDS matmul pipeline (gemm_dl_kernel), shared by the large-tile
// launches (gemm.hip) and the middle-size ones (gemm_mid.hip).
#pragma once

#include "gemm_common.h"

namespace mi {
namespace {

// ---- direct-to-LDS pipeline --------------------------
//
// DlCfg: WM x WN waves of TM x TN each, a ring of STAGES.  The description and
// figures below are the large tile's:
// 256 x 256 output tile per 512-lane block (8 waves as 4 along M x 2 along N,
// each wave 64 x 128 = 2 x 4 MFMA tiles, so two waves share a SIMD and one
// issues MFMAs while the other waits).  K steps of 64 flow through a ring of
// two LDS stages that global_load_lds_dwordx4 fills straight from global
// memory (no VGPR staging, no ds_write): the end of step k refills the stage
// it just finished with step k + 2.  Rows are 128 B (8 chunks of 16 B) and
// chunk c of row r is stored at chunk c ^ (r & 7) ^ ((r >> 3) & 1), which
// keeps the 16-byte fragment reads of 16 consecutive rows on distinct banks
// (whether the LDS is banked 32 or 64 wide).  Each substep's fragment reads
// for the next substep, and at the step boundary the refill loads, are
// interleaved with the MFMAs.  The epilogue applies alpha / beta * bias,
// rounds once, stages each wave's 64 x 128 tile through LDS and stores whole
// 256-byte row segments.
template <int WM_, int WN_, int TM_, int TN_, int STAGES_>
struct DlCfg {
  static constexpr int BK = 64, STAGES = STAGES_, WM = WM_, WN = WN_;
  static constexpr int NW = WM * WN, NT = 64 * NW;
  static constexpr int TM = TM_, TN = TN_, EP = TN + 8;  // wave tile, epilogue LDS pitch
  static constexpr int BM = WM * TM, BN = WN * TN;
  static constexpr int CH = BK / 8;                      // 16-byte chunks per row
  static constexpr int RPK = 512 / BK;                   // rows per 1 KiB wave load
  static constexpr int NQA = BM / RPK / NW, NQB = BN / RPK / NW;
  static constexpr int LPS = NQA + NQB;                  // wave loads per step
  static constexpr int TA = BM * BK, TB = BN * BK;
  static constexpr size_t LDS_BYTES =
      (size_t)STAGES * (TA + TB) * 2 > (size_t)NW * TM * EP * 2 ? (size_t)STAGES * (TA + TB) * 2
                                                                  : (size_t)NW * TM * EP * 2;
  static constexpr int GROUP_M = 4;
  // int8 B: 64-byte rows (4 chunks of 16 B), 16 rows per 1 KiB wave load
  static constexpr int CH8 = 4, RPK8 = 16, NQB8 = BN / RPK8 / NW;
  static constexpr int TB8 = BN * BK / 2;                // in 16-bit units
  // int8 B adds a bf16 copy of each stage's W rows: 160 KiB in all
  static constexpr size_t LDS_BYTES8 = (size_t)STAGES * (TA + TB8) * 2 + (size_t)STAGES * TB * 2;
};
typedef DlCfg<4, 2, 64, 128, 2> dl;  // 256 x 256
static_assert(dl::LDS_BYTES8 <= 160 * 1024 &&
                  dl::LDS_BYTES8 >= (size_t)dl::NW * dl::TM * dl::EP * 2, "int8 LDS");

typedef __attribute__((address_space(3))) void lds_void_t;
typedef short s16x4_t __attribute__((ext_vector_type(4)));

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  // s_waitcnt: vmcnt[3:0] | expcnt[6:4] = 7 | lgkmcnt[11:8] = 15 | vmcnt[5:4] at [15:14]
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// waits until at most `later` steps' loads (LPW per step) are outstanding
template <int MAXL, int LPW>
__device__ __forceinline__ void wait_later(int later) {
  if constexpr (MAXL > 0) {
    if (later >= MAXL) {
      wait_vmcnt<MAXL * LPW>();
      return;
    }
    wait_later<MAXL - 1, LPW>(later);
  } else {
    wait_vmcnt<0>();
  }
}

// 128-byte rows (8 chunks of 16 B): chunk c of row r at c ^ f(r), with
// f(r) = (r & 3) ^ 5 (bit 2 of r) ^ 4 (bit 3 of r): bit 0 = r0 ^ r2, bit 1 =
// r1, bit 2 = r2 ^ r3.  Chosen by timing every linear map of the row's low 4
// bits to a chunk mask on this LDS (a 64-lane ds_read_b128 takes 4 cycles
// without conflicts, 5.5 with the 2-way ones): it reads without conflicts
// 16 x 16 x 32 fragments (row l % 16, chunk 4 s + l / 16), 32 x 32 x 16
// fragments (row l % 32, chunk 2 s + l / 32), and the int8 widening's
// patterns (2 lanes a row x 4 chunks, 4 lanes a row x 2 chunks).  The mask
// (r & 7) ^ (r >> 3 & 1) it replaces made every 16 x 16 x 32 fragment read
// two-way conflicted (SQ_LDS_BANK_CONFLICT half of the LDS-active cycles).
__device__ __forceinline__ int dl_swz(int r, int c) {
  return c ^ (r & 3) ^ (((r >> 2) & 1) * 5) ^ ((r >> 1) & 4);
}
// 64-byte rows: chunk c of row r at c ^ ((r >> 1) & 3) ^ ((r >> 3) & 1), conflict-free for
// 16-byte reads of 16 consecutive rows under 32- or 64-bank LDS
__device__ __forceinline__ int dl_swz64(int r, int c) { return c ^ (((r >> 1) & 3) ^ ((r >> 3) & 1)); }

// SPLIT: blockIdx.y is a K slice instead of a batch; the block multiplies
// its slice's whole 64-wide steps (slice s of S gets KT / S steps, one more
// for s < KT % S) and stores the raw fp32 sums to part[s][M][ldp] for
// splitk_combine_kernel (no scale, bias or rounding here).
// B_KN: B is a row-major [K][N] matrix (ldb = its row stride, N contiguous),
// read in place: a stage holds the step's 64 k rows of the tile's 256
// columns (512 B each, 16-byte chunk c of row k at c ^ 4 (k & 3)), and the
// B fragments are read transposed by ds_read_b64_tr_b16, which hands each
// lane one column for 4 consecutive k (two reads per 8-k fragment).  Per
// read, lanes 0..31 cover 4 rows x 128 bytes and land on 64 distinct banks.
// TAIL: K need not be a multiple of 64: the last K % 64 columns (zeros past K)
// are multiplied before the pipelined whole steps, in the last slice of a SPLIT.
// EPI: fused epilogues of two matmuls of a decoder layer, each reproducing
// the rounding of the unfused ops bit for bit:
//   EPI_RESID: out = residual + round(x W^T), as linear then add (the sum in
//     fp32, rounded once), the residual read in the coalesced store pass;
//   EPI_SILU:  out = silu(round(x Wg^T)) * round(x Wu^T), as two linears then
//     silu_mul: a 256-wide tile holds 128 gate columns (waves 0..3 copy their
//     B rows from Wg) and the same 128 up columns (waves 4..7 from Wu), the
//     waves of column half 0 stage gate, those of half 1 up, and after a
//     barrier each wave combines half of its row band's pairs.
constexpr int EPI_NONE = 0, EPI_RESID = 1, EPI_SILU = 2;

template <typename T, bool HAS_BIAS, bool B_INT8, bool SPLIT = false, bool B_KN = false,
          int EPI = EPI_NONE, class C = dl, bool TAIL = false>
__global__ __launch_bounds__(C::NT, 2) void gemm_dl_kernel(GemmArgs p, float* part, int64_t ldp) {
  static_assert(!B_KN || (!B_INT8 && !SPLIT), "row-major B: 16-bit, no split");
  static_assert(EPI == EPI_NONE || (!HAS_BIAS && !B_INT8 && !SPLIT && !B_KN),
                "fused epilogues: plain 16-bit K-contiguous matmul");
  static_assert(!TAIL || (!B_INT8 && !B_KN && EPI == EPI_NONE), "K tail: plain 16-bit operands");
  static_assert(EPI != EPI_SILU || (C::WN == 2 && C::NQB * C::RPK * C::NW / 2 == C::BN / 2),
                "gate rows come from waves 0..NW/2-1, up rows from the others");
  // MFMA shape: 16 x 16 x 32 (MD = 16) for K-contiguous operands, 32 x 32 x 16
  // for the transposed row-major B reads, whose lane layout is built for it
  constexpr bool M16 = !B_KN;
  constexpr int MD = M16 ? 16 : 32, KPM = 512 / MD;  // MFMA tile edge, k per MFMA
  constexpr int BK = C::BK, STAGES = C::STAGES, WN = C::WN, TM = C::TM, TN = C::TN;
  constexpr int FM = TM / MD, FN = TN / MD, KS = BK / KPM;
  constexpr int BM = C::BM, BN = C::BN, CH = C::CH, RPK = C::RPK, NQA = C::NQA,
                TA = C::TA, EP = C::EP, GROUP_M = C::GROUP_M;
  // the B tile: 16-bit rows of 128 B, or int8 rows of 64 B (widened at fragment read)
  constexpr int NQB = B_INT8 ? C::NQB8 : C::NQB;
  constexpr int TB = B_INT8 ? C::TB8 : C::TB;
  constexpr int LPS = NQA + NQB;
  typedef typename MfmaOp<T>::vec vec;
  typedef typename std::conditional<M16, f32x4_t, f32x16>::type acc_t;
  auto mma = [](vec a, vec b, acc_t c) __attribute__((always_inline)) {
    if constexpr (!M16) return MfmaOp<T>::mma(a, b, c);
    else if constexpr (std::is_same<T, BF16>::value)
      return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    else
      return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  };
  extern __shared__ __align__(16) uint16_t smem[];
  // XCD-aware tile order (round-robin dispatch over 8 XCDs), then groups of
  // GROUP_M row panels so the tiles an XCD runs together share A and B panels
  int tm, tn;
  {
    const int total = p.tiles_m * p.tiles_n;
    int id = blockIdx.x;
    if (total % 8 == 0) {
      const int per = total / 8;
      id = (id % 8) * per + id / 8;
    }
    const int group = id / (GROUP_M * p.tiles_n);
    const int first_m = group * GROUP_M;
    const int gsize = min(p.tiles_m - first_m, GROUP_M);
    const int in_group = id - group * GROUP_M * p.tiles_n;
    tm = first_m + in_group % gsize;
    tn = in_group / gsize;
  }
  const int64_t batch = SPLIT ? 0 : blockIdx.y;
  const int M = (int)p.M, N = (int)p.N, K = (int)p.K;
  const int m0 = tm * BM, n0 = tn * BN;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;
  int KT = K / BK, k_first = 0;
  if constexpr (SPLIT) {
    const int S = gridDim.y, sl = blockIdx.y, base = KT / S, rem = KT % S;
    k_first = sl * base + min(sl, rem);
    KT = base + (sl < rem ? 1 : 0);
  }
  const uint16_t* A = p.a + batch * p.sa + (int64_t)k_first * BK;
  // EPI_SILU: waves 0..NW/2-1 copy gate rows, the others up rows
  const void* bsrc = (EPI == EPI_SILU && wave >= C::NW / 2) ? p.b2 : p.b;
  const char* Bbase = (const char*)bsrc + (batch * p.sb + (int64_t)k_first * BK * (B_KN ? p.ldb : 1)) *
                                              (B_INT8 ? 1 : 2);

  // per-lane byte offsets (the host checked they fit 32 bits); rows past the
  // matrix are clamped to its last row and only feed outputs never stored
  uint32_t ao[NQA], bo[NQB];
#pragma unroll
  for (int q = 0; q < NQA; ++q) {
    const int row = (wave * NQA + q) * RPK + lane / CH;
    ao[q] = (uint32_t)(((int64_t)min(m0 + row, M - 1) * p.lda + dl_swz(row, lane % CH) * 8) * 2);
  }
#pragma unroll
  for (int q = 0; q < NQB; ++q) {
    if constexpr (B_KN) {
      // wave copy q: k rows 2 (wave NQB + q) and the next, 32 chunks each;
      // columns past N re-read the last chunk (their outputs are not stored)
      const int row = 2 * (wave * NQB + q) + lane / 32, c = (lane & 31) ^ (4 * (row & 3));
      bo[q] = (uint32_t)(((int64_t)row * p.ldb + min(n0 + 8 * c, N - 8)) * 2);
    } else if constexpr (B_INT8) {
      const int row = (wave * NQB + q) * C::RPK8 + lane / C::CH8;
      bo[q] = (uint32_t)((int64_t)min(n0 + row, N - 1) * p.ldb + dl_swz64(row, lane % C::CH8) * 16);
    } else {
      const int row = (wave * NQB + q) * RPK + lane / CH;
      // EPI_SILU: tile tn covers output columns 128 tn .. 128 tn + 127 (rows
      // 0..127 of the tile from the gate weight, 128..255 from the up weight)
      const int grow = EPI == EPI_SILU ? tn * (BN / 2) + (row & (BN / 2 - 1)) : n0 + row;
      bo[q] = (uint32_t)(((int64_t)min(grow, N - 1) * p.ldb + dl_swz(row, lane % CH) * 8) * 2);
    }
  }
  auto issue = [&](int st, int k0) __attribute__((always_inline)) {
    uint16_t* as = smem + st * (TA + TB);
    uint16_t* bs = as + TA;
    const char* Ab = (const char*)(A + k0);
    const char* Bb = Bbase + (int64_t)k0 * (B_KN ? p.ldb * 2 : (B_INT8 ? 1 : 2));
#pragma unroll
    for (int q = 0; q < NQA; ++q) lds_copy16(Ab, ao[q], as + (wave * NQA + q) * 512);
#pragma unroll
    for (int q = 0; q < NQB; ++q) lds_copy16(Bb, bo[q], bs + (wave * NQB + q) * 512);
  };
  // fragment read offsets: lane supplies row l % MD, 16-byte k chunk
  // (KPM / 8) s + l / MD of substep s
  int roff[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    roff[s] = (lane % MD) * BK + dl_swz(lane % MD, (KPM / 8) * s + lane / MD) * 8;
  }

  // acc[j][i] = D^T tile (n rows j, m cols i): B fragments are the MFMA's A
  // operand, so a lane ends up owning one output row m and runs of 4 n
  // (4 runs for 32 x 32 tiles, one for 16 x 16)
  acc_t acc[FN][FM];
#pragma unroll
  for (int j = 0; j < FN; ++j)
#pragma unroll
    for (int i = 0; i < FM; ++i) acc[j][i] = acc_t{};
  vec af[2][FM], bfr[2][FN];
  // row-major B: lane (G = lane / 16, j = lane % 16) reads k row
  // 8 (G / 2) + j / 4 (+ 4 for the second half) of a substep, columns
  // wn TN + 32 jt + 16 (G % 2) + 4 (j % 4) .. + 3; the chunk swizzle makes
  // the fragment jt's offset 64 (jt ^ (j / 4)) bytes, per lane
  int kno[FN];
  if constexpr (B_KN) {
    const int G = lane >> 4, j = lane & 15;
    const int kr = 8 * (G >> 1) + (j >> 2);
    const int x = 2 * (G & 1) + ((j & 3) >> 1);
#pragma unroll
    for (int jt = 0; jt < FN; ++jt)
      kno[jt] = kr * BN + (wn * 16 + 4 * (jt ^ (j >> 2)) + x) * 8 + 4 * (j & 1);  // in elements
  }
  auto read_frags = [&](int st, int s, int buf) __attribute__((always_inline)) {
    const uint16_t* as = smem + st * (TA + TB) + wm * TM * BK + roff[s];
#pragma unroll
    for (int i = 0; i < FM; ++i) af[buf][i] = *(const vec*)(as + i * MD * BK);
    if constexpr (B_KN) {
      typedef __attribute__((address_space(3))) s16x4_t lds_s16x4_t;
      const uint16_t* bs = smem + st * (TA + TB) + TA + 16 * s * BN;
#pragma unroll
      for (int jt = 0; jt < FN; ++jt) {
        const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(bs + kno[jt]));
        const s16x4_t hi =
            __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(bs + kno[jt] + 4 * BN));
        bfr[buf][jt] = __builtin_bit_cast(vec, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    } else if constexpr (B_INT8) {
      // the bf16 copy of the stage's W rows (converted once per block)
      const uint16_t* bs = smem + STAGES * (TA + TB) + st * C::TB + wn * TN * BK + roff[s];
#pragma unroll
      for (int j = 0; j < FN; ++j) bfr[buf][j] = *(const vec*)(bs + j * MD * BK);
    } else {
      const uint16_t* bs = smem + st * (TA + TB) + TA + wn * TN * BK + roff[s];
#pragma unroll
      for (int j = 0; j < FN; ++j) bfr[buf][j] = *(const vec*)(bs + j * MD * BK);
    }
  };
  auto mfmas = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int i = 0; i < FM; ++i) acc[j][i] = mma(bfr[buf][j], af[buf][i], acc[j][i]);
  };
  // int8 W: wave w copied rows 32 w .. 32 w + 31 of every stage itself, so
  // once its own loads have landed it widens exactly those rows into the
  // stage's bf16 copy (same chunk swizzle as a 16-bit B tile); the barrier
  // that follows publishes them.  Lane: row 32 w + l / 2, k half l % 2.
  auto convert = [&](int st) __attribute__((always_inline)) {
    if constexpr (B_INT8) {
      const char* b8 = (const char*)(smem + st * (TA + TB) + TA);
      uint16_t* bb = smem + STAGES * (TA + TB) + st * C::TB;
      const int r = wave * 32 + (lane >> 1), h = lane & 1;
      const u32x4_t c0 = *(const u32x4_t*)(b8 + r * 64 + dl_swz64(r, 2 * h) * 16);
      const u32x4_t c1 = *(const u32x4_t*)(b8 + r * 64 + dl_swz64(r, 2 * h + 1) * 16);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const u32x4_t& c = j < 2 ? c0 : c1;
        const u32x2_t w = {c[2 * (j & 1)], c[2 * (j & 1) + 1]};
        *(vec*)(bb + r * BK + dl_swz(r, 4 * h + j) * 8) = widen8<T>(w);
      }
    }
  };
  constexpr int NMF = FM * FN, NDS = FM + FN;
  // 16 x 16 x 32 schedule, in an order the compiler keeps (a scheduling fence
  // after every MFMA): A fragments double-buffered, read for the next
  // substep during the first FM MFMAs; B fragments single-buffered, fragment
  // j of the next substep read right after its last MFMA (j FM + FM - 1) of
  // this one, so each read has most of a substep to land; the refill loads
  // one per two MFMAs of the step's last substep.  Against the 32 x 32
  // tiles with grouped reads this is 4-10 % faster on the decoder-layer and
  // config-4 shapes, with bit-identical results.
  auto issue_one = [&](int st, int k0, int q) __attribute__((always_inline)) {
    uint16_t* as = smem + st * (TA + TB);
    uint16_t* bs = as + TA;
    if (q < NQA) {
      lds_copy16(A + k0, ao[q], as + (wave * NQA + q) * 512);
    } else {
      const char* Bb = Bbase + (int64_t)k0 * (B_INT8 ? 1 : 2);
      lds_copy16(Bb, bo[q - NQA], bs + (wave * NQB + q - NQA) * 512);
    }
  };
  auto read_a = [&](int st, int s, int buf, int i) __attribute__((always_inline)) {
    const uint16_t* as = smem + st * (TA + TB) + wm * TM * BK + roff[s];
    af[buf][i] = *(const vec*)(as + i * MD * BK);
  };
  auto read_b = [&](int st, int s, int j) __attribute__((always_inline)) {
    const uint16_t* bs = B_INT8 ? smem + STAGES * (TA + TB) + st * C::TB + wn * TN * BK + roff[s]
                                : smem + st * (TA + TB) + TA + wn * TN * BK + roff[s];
    bfr[0][j] = *(const vec*)(bs + j * MD * BK);
  };
  auto mfma_one = [&](int buf, int m) __attribute__((always_inline)) {
    const int j = m / FM, i = m % FM;
    acc[j][i] = mma(bfr[0][j], af[buf][i], acc[j][i]);
  };
  // one K step over stage st.  ISSUE: refill stage st with step kt + STAGES;
  // NEXT: step kt + 1 exists and its first fragments are read here.
  auto step = [&](int st, int kt, bool ISSUE, bool NEXT) __attribute__((always_inline)) {
    if constexpr (M16) {
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int buf = s & 1;
        if (s + 1 < KS) {
#pragma unroll
          for (int m = 0; m < NMF; ++m) {
            mfma_one(buf, m);
            if (m < FM) read_a(st, s + 1, buf ^ 1, m);
            if (m % FM == FM - 1) read_b(st, s + 1, m / FM);
            __builtin_amdgcn_sched_barrier(0);
          }
        } else {
          const int nst = st + 1 == STAGES ? 0 : st + 1;
          if (NEXT) {
            // as below: step kt + 1 has landed and every wave is done with
            // stage st (its last fragments were read in the previous substep)
            if (ISSUE) wait_vmcnt<(STAGES - 2) * LPS>();
            else wait_vmcnt<0>();
            convert(nst);
            __syncthreads();
          }
          // one refill load per two MFMAs, from the substep's first MFMA (the
          // loads spread over all of it measured 1-3 % slower on the decoder
          // shapes, back to back 2-4 % slower)
          constexpr int MPL = NMF >= 2 * LPS ? 2 : 1;
          static_assert(MPL * LPS <= NMF, "every refill load is issued in the substep");
#pragma unroll
          for (int m = 0; m < NMF; ++m) {
            mfma_one(buf, m);
            if (ISSUE && m % MPL == 0 && m / MPL < LPS) issue_one(st, (kt + STAGES) * BK, m / MPL);
            if (NEXT) {
              if (m < FM) read_a(nst, 0, buf ^ 1, m);
              if (m % FM == FM - 1) read_b(nst, 0, m / FM);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
      return;
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int buf = s & 1;
      if (s + 1 < KS) {
        read_frags(st, s + 1, buf ^ 1);
        mfmas(buf);
#pragma unroll
        for (int k = 0; k < NDS; ++k) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // DS read
        }
        __builtin_amdgcn_sched_group_barrier(0x008, NMF - NDS, 0);
      } else {
        if (NEXT) {
          // step kt + 1 has landed once at most the newer steps' loads are
          // outstanding; the barrier also tells every wave that all waves
          // are done reading stage st
          if (ISSUE) wait_vmcnt<(STAGES - 2) * LPS>();
          else wait_vmcnt<0>();
          convert(st + 1 == STAGES ? 0 : st + 1);
          __syncthreads();
          if (ISSUE) issue(st, (kt + STAGES) * BK);
          read_frags(st + 1 == STAGES ? 0 : st + 1, 0, buf ^ 1);
        }
        mfmas(buf);
#pragma unroll
        for (int k = 0; k < NMF; ++k) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (ISSUE && k < LPS) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // VMEM
          if (NEXT && k < NDS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // The epilogue's pointers are formed (and their scalar loads waited for)
  // before the main loop: left to the compiler, such a load (the batch
  // stride, the int8 scales) was issued just before the loop and stayed in
  // flight through it, and since scalar loads return out of order every LDS
  // wait in the loop became lgkmcnt(0), so each step's first MFMA waited for
  // reads issued after the ones it needs.
  uint16_t* Cb = p.c + batch * p.sc;
  asm volatile("" : : "s"(Cb));
  const float* scale = p.scale;
  if constexpr (B_INT8) asm volatile("" : : "s"(scale));
  if constexpr (TAIL) {
    // the last K % 64 columns first, through the last stage, while the copies
    // of the other stages are in flight
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
      if (s < KT) issue(s, s * BK);
    const int kt0 = K / BK * BK;
    if (kt0 < K && (!SPLIT || blockIdx.y + 1 == gridDim.y)) {
      typedef uint16_t u16x8_t __attribute__((ext_vector_type(8)));
      uint16_t* ts = smem + (STAGES - 1) * (TA + TB);
      const uint16_t* A0 = p.a + batch * p.sa;
      const uint16_t* B0 = (const uint16_t*)p.b + batch * p.sb;
      // the copies' layout: LDS chunk lane % CH of a row holds global chunk
      // dl_swz(row, lane % CH); loads past K re-read inside the row
      auto row_of = [&](int q) __attribute__((always_inline)) {
        return (q < NQA ? wave * NQA + q : wave * NQB + q - NQA) * RPK + lane / CH;
      };
      auto src = [&](int q) __attribute__((always_inline)) {
        return q < NQA ? A0 + (int64_t)min(m0 + row_of(q), M - 1) * p.lda
                       : B0 + (int64_t)min(n0 + row_of(q), N - 1) * p.ldb;
      };
      auto k_of = [&](int q) __attribute__((always_inline)) {
        return kt0 + 8 * dl_swz(row_of(q), lane % CH);
      };
      u16x8_t v[NQA + NQB];
      if (K >= 8) {
        // a chunk that passes K as the row's last 8 elements, shifted down (M1500 N1000
        // K130 12.3 us; 14.7 with a load per element)
        typedef u16x8_t __attribute__((aligned(2))) u16x8_u;
#pragma unroll
        for (int q = 0; q < NQA + NQB; ++q) v[q] = *(const u16x8_u*)(src(q) + min(k_of(q), K - 8));
#pragma unroll
        for (int q = 0; q < NQA + NQB; ++q)
          v[q] = __builtin_bit_cast(u16x8_t, shift_down(__builtin_bit_cast(u64x2_t, v[q]),
                                                        2 * max(0, k_of(q) - (K - 8))));
      } else {
#pragma unroll
        for (int q = 0; q < NQA + NQB; ++q)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const uint16_t x = src(q)[min(k_of(q) + e, K - 1)];
            v[q][e] = k_of(q) + e < K ? x : (uint16_t)0;
          }
      }
#pragma unroll
      for (int q = 0; q < NQA + NQB; ++q)
        *(u16x8_t*)(ts + (q < NQA ? (wave * NQA + q) * 512 : TA + (wave * NQB + q - NQA) * 512) +
                    lane * 8) = v[q];
      __syncthreads();
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        read_frags(STAGES - 1, s, 0);
        mfmas(0);
      }
      __syncthreads();
    }
    if (STAGES - 1 < KT) issue(STAGES - 1, (STAGES - 1) * BK);
  } else {
#pragma unroll
    for (int s = 0; s < STAGES; ++s)
      if (s < KT) issue(s, s * BK);
  }
  if (STAGES <= KT) wait_vmcnt<(STAGES - 1) * LPS>();
  else wait_vmcnt<0>();
  convert(0);
  __syncthreads();
  read_frags(0, 0, 0);
  int st = 0, kt = 0;
  for (; kt < KT - STAGES; ++kt) {
    step(st, kt, true, true);
    st = st + 1 == STAGES ? 0 : st + 1;
  }
  for (; kt < KT; ++kt) {
    step(st, kt, false, kt + 1 < KT);
    st = st + 1 == STAGES ? 0 : st + 1;
  }

  if constexpr (SPLIT) {
    // raw sums of this K slice: a lane's runs of 4 columns as 16-byte stores
    // (ldp is a multiple of 4, so a run that starts inside the row fits)
    float* P = part + (int64_t)blockIdx.y * p.M * ldp;
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int g = 0; g < MD * MD / 256; ++g) {
        const int64_t n = n0 + wn * TN + j * MD + (M16 ? 4 * (lane >> 4) : 8 * g + 4 * (lane >> 5));
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          const int64_t m = m0 + wm * TM + i * MD + (lane % MD);
          if (m < p.M && n < p.N) {
            const f32x4_t v = {acc[j][i][4 * g], acc[j][i][4 * g + 1], acc[j][i][4 * g + 2],
                               acc[j][i][4 * g + 3]};
            *(f32x4_t*)(P + m * ldp + n) = v;
          }
        }
      }
    return;
  }
  // epilogue: out = alpha * acc + beta * bias, one rounding, staged per wave.
  // A lane's outputs come in runs of 4 columns; the per-column factors (the
  // int8 scale, a bias broadcast over rows) are loaded once per run, four
  // at a time, and used for both row fragments (one scalar load per output
  // made the bias epilogue cost 13 % of config 4's addmm)
  __syncthreads();
  uint16_t* es = smem + wave * TM * EP;
  const float alpha = p.alpha, beta = p.beta;
  const bool row_bias = HAS_BIAS && p.bias_sm == 0;
  auto load_col4 = [&](const void* base, int dtype, int64_t n, int64_t stride, int64_t N,
                       int64_t off = 0) __attribute__((always_inline)) {
    return load_col4_t<T>(base, dtype, n, stride, N, off);
  };
#pragma unroll
  for (int j = 0; j < FN; ++j)
#pragma unroll
    for (int g = 0; g < MD * MD / 256; ++g) {
      const int nl = j * MD + (M16 ? 4 * (lane >> 4) : 8 * g + 4 * (lane >> 5));
      const int64_t n = n0 + wn * TN + nl;
      f32x4_t sc4 = {1.f, 1.f, 1.f, 1.f}, bb4 = {};
      if constexpr (B_INT8) sc4 = load_col4(scale, MI_F32, n, 1, p.N);
      if (row_bias) bb4 = load_col4(p.bias, p.bias_dtype, n, p.bias_sn, p.N, batch * p.bias_sb);
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const int ml = i * MD + (lane % MD);
        const int64_t m = m0 + wm * TM + ml;
        u16x4_t v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float x = alpha * acc[j][i][4 * g + e] * sc4[e];
          if (HAS_BIAS) {
            float bv = bb4[e];
            if (!row_bias) {
              const int64_t bo_ = batch * p.bias_sb + min<int64_t>(m, p.M - 1) * p.bias_sm +
                                  min<int64_t>(n + e, p.N - 1) * p.bias_sn;
              bv = p.bias_dtype == MI_F32 ? ((const float*)p.bias)[bo_]
                                          : MfmaOp<T>::load(((const uint16_t*)p.bias)[bo_]);
            }
            x += beta * bv;
          }
          v[e] = MfmaOp<T>::store(x);
        }
        *(u16x4_t*)(es + ml * EP + nl) = v;
      }
    }
  const int64_t rbase = m0 + wm * TM, cbase = n0 + wn * TN;
  constexpr int LPR = TN / 8, RPI = 64 / LPR;  // lanes per row, rows per pass
  const bool vec_ok = (p.ldc % 8) == 0 && (((uintptr_t)Cb) & 15) == 0;
  typedef uint16_t u16x8_t __attribute__((ext_vector_type(8)));
  if constexpr (EPI == EPI_SILU) {
    // the row band's gate values are in the staging of wave (wm, 0), its up
    // values in that of wave (wm, 1); wave (wm, wn) takes rows 32 wn .. 32 wn + 31
    __syncthreads();
    const uint16_t* eg = smem + (wm * WN) * TM * EP;
    const uint16_t* eu = eg + TM * EP;
    const int64_t cb = (int64_t)tn * (BN / 2);
#pragma unroll 4
    for (int it = 0; it < TM / 2 / RPI; ++it) {
      const int r = wn * (TM / 2) + it * RPI + lane / LPR, c = (lane % LPR) * 8;
      const u16x8_t g8 = *(const u16x8_t*)(eg + r * EP + c);
      const u16x8_t u8 = *(const u16x8_t*)(eu + r * EP + c);
      u16x8_t v;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        v[e] = MfmaOp<T>::store(silu_mul_f32(MfmaOp<T>::load(g8[e]), MfmaOp<T>::load(u8[e])));
      const int64_t m = rbase + r, n = cb + c;
      if (m < p.M) {
        if (vec_ok && n + 7 < p.N) {
          *(u16x8_t*)(Cb + m * p.ldc + n) = v;
        } else {
          for (int e = 0; e < 8; ++e)
            if (n + e < p.N) Cb[m * p.ldc + n + e] = v[e];
        }
      }
    }
    return;
  }
  const bool res_vec = EPI == EPI_RESID && (p.ldr % 8) == 0 && (((uintptr_t)p.res) & 15) == 0;
#pragma unroll 4
  for (int it = 0; it < TM / RPI; ++it) {
    const int r = it * RPI + lane / LPR, c = (lane % LPR) * 8;
    u16x8_t v = *(const u16x8_t*)(es + r * EP + c);
    const int64_t m = rbase + r, n = cbase + c;
    if (m < p.M) {
      if constexpr (EPI == EPI_RESID) {
        // residual + the rounded product, as the add kernel: fma(other, 1, self)
        u16x8_t rv;
        if (res_vec && n + 7 < p.N) {
          rv = *(const u16x8_t*)(p.res + m * p.ldr + n);
        } else {
          for (int e = 0; e < 8; ++e) rv[e] = n + e < p.N ? p.res[m * p.ldr + n + e] : (uint16_t)0;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e)
          v[e] = MfmaOp<T>::store(
              __builtin_fmaf(MfmaOp<T>::load(v[e]), 1.0f, MfmaOp<T>::load(rv[e])));
      }
      if (vec_ok && n + 7 < p.N) {
        *(u16x8_t*)(Cb + m * p.ldc + n) = v;
      } else {
        for (int e = 0; e < 8; ++e)
          if (n + e < p.N) Cb[m * p.ldc + n + e] = v[e];
      }
    }
  }
}

}  // namespace
}  // namespace mi
