// 16-bit matrix products: the direct-to-LDS pipeline (gemm_dl.h) on 256 x 256
// tiles, and on smaller tiles, deeper rings and K slices for problems whose
// large tiles do not fill the CUs evenly.
//
// What bounds the middle sizes: with one block or less per CU a K step costs its latency
// until the ring holds enough steps in flight (two stages of 128 x 128 took
// 0.80 us a step with 64 blocks, four stages 0.50), then the matrix cores, with the
// fragment reads behind them (M777 N4096 K11008: MFMA 0.68 of the busy cycles, LDS
// 0.34; a wave's 64 x 64 tile reads 16 KiB for 32 MFMAs).  So smaller tiles buy
// parallelism at more LDS traffic per MFMA, and K slices buy it at fp32
// partial sums; which is cheaper depends on how many tiles there are.  The
// register-staged 128 x 128 / 128 x 64 tiles that ran here had one step in
// flight.  us, before and now (K-contiguous bf16 B):
//   M128 N11008 K4096 60 -> 30      M256 N4096 K11008 140 -> 39
//   M777 N4096 K11008 161 -> 92     M512 N1024 K1024  11 -> 6.2
//   M1024 N4096 K4096 58 -> 35      M2048 N4096 K4096 85 -> 55
//   M4352 N4096 K4096 (272 tiles of 256 x 256, two rounds) 164 -> 144
#include <algorithm>

#include "gemm_dl.h"

namespace mi {
namespace {

typedef DlCfg<4, 2, 64, 128, 2> C256;
typedef DlCfg<4, 2, 64, 64, 3> C256x128;
typedef DlCfg<2, 2, 64, 64, 4> C128;
typedef DlCfg<2, 2, 64, 32, 3> C128x64;
typedef DlCfg<2, 2, 32, 32, 5> C64;

template <typename T, bool HB, class C>
mi_status_t launch(const GemmArgs& q0, int S, int64_t batch, hipStream_t s, const char* what) {
  static bool attr = [] {
    (void)hipFuncSetAttribute((const void*)gemm_dl_kernel<T, false, false, true, false, EPI_NONE, C, true>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)C::LDS_BYTES);
    (void)hipFuncSetAttribute((const void*)gemm_dl_kernel<T, HB, false, false, false, EPI_NONE, C, true>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)C::LDS_BYTES);
    return true;
  }();
  (void)attr;
  GemmArgs q = q0;
  q.tiles_m = (int)((q.M + C::BM - 1) / C::BM);
  q.tiles_n = (int)((q.N + C::BN - 1) / C::BN);
  const unsigned tiles = (unsigned)(q.tiles_m * q.tiles_n);
  const int64_t ldp = (q.N + 3) / 4 * 4;
  Workspace ws;
  if (S > 1 && ws.alloc((size_t)S * (size_t)q.M * (size_t)ldp * sizeof(float), s) != MI_OK) {
    clear_error();  // the whole K in one block needs no workspace
    S = 1;
  }
  if (S <= 1) {
    hipLaunchKernelGGL((gemm_dl_kernel<T, HB, false, false, false, EPI_NONE, C, true>),
                       dim3(tiles, (unsigned)batch), dim3(C::NT), C::LDS_BYTES, s, q, nullptr,
                       (int64_t)0);
    return check_launch(what);
  }
  hipLaunchKernelGGL((gemm_dl_kernel<T, false, false, true, false, EPI_NONE, C, true>),
                     dim3(tiles, (unsigned)S), dim3(C::NT), C::LDS_BYTES, s, q, (float*)ws.get(), ldp);
  MI_RETURN_IF(check_launch(what));
  return launch_splitk_combine(q, std::is_same<T, F16>::value, HB, (const float*)ws.get(), S, ldp, s, what);
}

// The cost in us of a tile shape and a slice count: rounds of one block per
// CU, each `steps` K steps of lo (few CUs busy) to hi (all busy) us, plus the
// launch, first latency and epilogue, and for every further round the part of
// those that the CU's other blocks do not cover; slices add a combine launch
// and their partial sums through the caches at 5.8 TB/s.  The constants are a fit to
// 1900 timings of these kernels (60 shapes, M 65 .. 4352, N 280 .. 11008, K
// 256 .. 11008, 1 to 8 slices); what it picks was within 2 % of the fastest on
// average, 20 % at worst.
struct Shape {
  int bm, bn;
  float lo, hi, fixed, round, round_short;  // round_short: below four K steps
};
constexpr Shape kShapes[] = {{256, 256, 1.03f, 1.26f, 6.9f, 4.7f, 4.7f},
                             {256, 128, 0.55f, 0.70f, 5.4f, 2.4f, 2.4f},
                             {128, 128, 0.30f, 0.455f, 5.3f, 1.8f, 1.8f},
                             {128, 64, 0.23f, 0.30f, 3.85f, 0.25f, 1.0f},
                             {64, 64, 0.15f, 0.195f, 3.8f, 0.5f, 0.8f}};
constexpr int kSlices[] = {1, 2, 3, 4, 6, 8};

struct Pick {
  int shape, slices;
  float cost;
};

// bn_div 2: a tile's columns are half gate and half up columns (EPI_SILU)
Pick pick_shape(const GemmArgs& q, int64_t batch, bool split, int bn_div) {
  const int64_t steps = (q.K + 63) / 64, cus = cu_count();
  auto tiles_of = [&](int bm, int bn) {
    return ((q.M + bm - 1) / bm) * ((q.N + bn / bn_div - 1) / (bn / bn_div)) * batch;
  };
  const bool full = tiles_of(256, 256) >= cus;
  Pick best{0, 1, 3e38f};
  for (int i = 0; i < 5; ++i) {
    const Shape& c = kShapes[i];
    const int64_t tiles = tiles_of(c.bm, c.bn);
    for (int s : kSlices) {
      if (s > 1 && (!split || batch > 1 || steps < s || tiles * s > 4 * cus)) break;
      const int64_t blocks = tiles * s, rounds = (blocks + cus - 1) / cus;
      const float load = std::min(1.f, (float)blocks / (float)cus);
      float t = c.fixed + (float)(rounds * ((steps + s - 1) / s)) * (c.lo + (c.hi - c.lo) * load) +
                (steps / s < 4 ? c.round_short : c.round) * (float)(rounds - 1);
      if (s > 1) t += 3.1f + (float)s * (float)q.M * (float)q.N * (8.f / 5.8e6f);
      // where 256 x 256 tiles fill the CUs, others have to be clearly faster: at
      // the sustained clock they lose about that much (M6000 N11008 K4096, 1 %
      // apart by this rule: 481 us on 256 x 256 tiles, 506 on 256 x 128)
      if (i > 0 && full) t *= 1.05f;
      if (t < best.cost) best = Pick{i, s, t};
    }
  }
  return best;
}

template <typename T, bool HB>
mi_status_t run(const GemmArgs& q, Pick c, int64_t batch, hipStream_t s, const char* what) {
  switch (c.shape) {
    case 0: return launch<T, HB, C256>(q, c.slices, batch, s, what);
    case 1: return launch<T, HB, C256x128>(q, c.slices, batch, s, what);
    case 2: return launch<T, HB, C128>(q, c.slices, batch, s, what);
    case 3: return launch<T, HB, C128x64>(q, c.slices, batch, s, what);
    default: return launch<T, HB, C64>(q, c.slices, batch, s, what);
  }
}

template <typename T, int EPI, class C>
mi_status_t launch_epi(const GemmArgs& q0, hipStream_t s, const char* what) {
  static bool attr = [] {
    (void)hipFuncSetAttribute((const void*)gemm_dl_kernel<T, false, false, false, false, EPI, C>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)C::LDS_BYTES);
    return true;
  }();
  (void)attr;
  GemmArgs q = q0;
  constexpr int BN = EPI == EPI_SILU ? C::BN / 2 : C::BN;
  q.tiles_m = (int)((q.M + C::BM - 1) / C::BM);
  q.tiles_n = (int)((q.N + BN - 1) / BN);
  hipLaunchKernelGGL((gemm_dl_kernel<T, false, false, false, false, EPI, C>),
                     dim3((unsigned)(q.tiles_m * q.tiles_n)), dim3(C::NT), C::LDS_BYTES, s, q, nullptr,
                     (int64_t)0);
  return check_launch(what);
}

template <typename T, int EPI>
mi_status_t run_epi(const GemmArgs& q, int shape, hipStream_t s, const char* what) {
  switch (shape) {
    case 0: return launch_epi<T, EPI, C256>(q, s, what);
    case 1: return launch_epi<T, EPI, C256x128>(q, s, what);
    case 2: return launch_epi<T, EPI, C128>(q, s, what);
    case 3: return launch_epi<T, EPI, C128x64>(q, s, what);
    default: return launch_epi<T, EPI, C64>(q, s, what);
  }
}

}  // namespace

bool gemm_mid_eligible(const GemmArgs& q) {
  if (q.K <= 0 || q.lda % 8 != 0 || q.ldb % 8 != 0 || q.sa % 8 != 0 || q.sb % 8 != 0) return false;
  if ((((uintptr_t)q.a) | ((uintptr_t)q.b)) & 15) return false;
  if (q.M > 0x7fffffff || q.N > 0x7fffffff || q.K > 0x7fffffff) return false;
  const int64_t amax = ((q.M - 1) * q.lda + q.K) * 2, bmax = ((q.N - 1) * q.ldb + q.K) * 2;
  return amax < ((int64_t)1 << 32) && bmax < ((int64_t)1 << 32);
}

mi_status_t launch_gemm_mid(const GemmArgs& q, int64_t batch, bool f16, bool has_bias, hipStream_t s,
                            const char* what) {
  const Pick c = pick_shape(q, batch, true, 1);
  if (f16)
    return has_bias ? run<F16, true>(q, c, batch, s, what) : run<F16, false>(q, c, batch, s, what);
  return has_bias ? run<BF16, true>(q, c, batch, s, what) : run<BF16, false>(q, c, batch, s, what);
}

// A fused epilogue (residual add, or SiLU-mul of two products) on the tile
// shape of least cost.  Its bits are the unfused ops' only if those sum K in one
// piece, so a product that launch_gemm_mid would slice is left to them (its
// slices are also what makes it fast), and so is one whose products and
// elementwise pass cost less.  us of kernel time
// where only 256 x 256 tiles were fused, and now: gate / up of 168 tokens (N11008
// K4096) 106 -> 46, of 1496 tokens (N5504 K2048, 258 tiles) 92 -> 84.
bool launch_gemm_fused(const GemmArgs& q, bool silu, bool f16, hipStream_t s, const char* what,
                       mi_status_t* st) {
  const Pick plain = pick_shape(q, 1, true, 1);
  if (plain.slices > 1) return false;
  const Pick c = pick_shape(q, 1, false, silu ? 2 : 1);
  const float pass = 3.f + (float)q.M * (float)q.N * (6.f / 5.8e6f);
  if (c.cost > (silu ? 2.f : 1.f) * plain.cost + pass) return false;
  if (silu) *st = f16 ? run_epi<F16, EPI_SILU>(q, c.shape, s, what) : run_epi<BF16, EPI_SILU>(q, c.shape, s, what);
  else *st = f16 ? run_epi<F16, EPI_RESID>(q, c.shape, s, what) : run_epi<BF16, EPI_RESID>(q, c.shape, s, what);
  return true;
}

}  // namespace mi
