// k_gemm.hip -- the unified bf16 GEMM of the encoder path on gfx950 MFMA.
//
// C[M, N] = epilogue(A[M, K] @ W[K, N] + bias) (+ residual), A bf16 row-major,
// W held as its transpose Wt[N, K] (K contiguous, the layout mx_stage_weight
// writes once) so both operands are read the same way. fp32 accumulation in
// v_mfma_f32_32x32x16_bf16; one rounding to bf16 (the host's to_bf16
// formula) at the very end when C is bf16 -- the single-narrowing contract of
// kernels/narrow_f32_bf16.cc, here fused into the store.
//
// Tiling: a BM x BN block tile over (BM/WM) x (BN/WN) waves, each wave owning
// a WM x WN sub-tile of (WM/32) x (WN/32) MFMA tiles. K advances BK at a time
// through two LDS buffers: the next K-slab is fetched from HBM into registers
// while the MFMAs consume the current one, then written to the other buffer,
// so there is one barrier per slab. LDS rows are padded by 16 bytes, which
// makes the 16-byte fragment reads of 8 consecutive rows hit distinct banks.
//
// Blocks are numbered so that each XCD (workgroups go round-robin over the 8
// XCDs) owns a contiguous run of tiles in row-major (m, n) order: the blocks
// resident on one XCD share A row-panels and the whole of W in its L2.
#include "mx_common.hpp"
#include "mx_kernels.hpp"

using namespace mxd;

namespace {

template <int BM, int BN, int BK, int WM, int WN>
struct GemmCfg {
  static constexpr int NWM = BM / WM, NWN = BN / WN;
  static constexpr int NT = NWM * NWN * 64;
  static constexpr int LDK = BK + 8;  // padded LDS row, elements
  static constexpr int TM = WM / 32, TN = WN / 32;
  static constexpr int CPR = BK / 8;  // 16-byte chunks per row
  static constexpr int A_PER_T = BM * CPR / NT;
  static constexpr int B_PER_T = BN * CPR / NT;
  static constexpr int LDS_BYTES = 2 * (BM + BN) * LDK * 2;
  static_assert(BM * CPR % NT == 0 && BN * CPR % NT == 0, "chunks must divide threads");
  static_assert(WM % 32 == 0 && WN % 32 == 0 && BK % 16 == 0, "MFMA tile shape");
};

template <int BM, int BN, int BK, int WM, int WN>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64) void gemm_bf16_k(
    const uint16_t *__restrict__ A, int64_t lda, const uint16_t *__restrict__ Wt, int M, int N,
    int K, const float *__restrict__ bias, int epi, const float *residual, void *C, int c_bf16,
    int64_t ldc, int tiles_m, int tiles_n, const int32_t *rows_dev) {
  using Cfg = GemmCfg<BM, BN, BK, WM, WN>;
  constexpr int LDK = Cfg::LDK, NT = Cfg::NT, CPR = Cfg::CPR;
  constexpr int TM = Cfg::TM, TN = Cfg::TN;
  __shared__ __attribute__((aligned(16))) uint16_t smA[2][BM * LDK];
  __shared__ __attribute__((aligned(16))) uint16_t smB[2][BN * LDK];

  // XCD-aware tile order.
  const int total = tiles_m * tiles_n;
  int tile = blockIdx.x;
  if ((total & 7) == 0) tile = (blockIdx.x & 7) * (total >> 3) + (blockIdx.x >> 3);
  const int tm = tile / tiles_n, tn = tile - tm * tiles_n;
  const int m0 = tm * BM, n0 = tn * BN;
  M = (int)live_rows(M, rows_dev);
  if (m0 >= M) return;  // the whole block: a tile past the live rows

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / Cfg::NWN, wn = wave - wm * Cfg::NWN;

  uint4 ra[Cfg::A_PER_T], rb[Cfg::B_PER_T];
  auto gload = [&](int k0) {
#pragma unroll
    for (int i = 0; i < Cfg::A_PER_T; ++i) {
      const int c = tid + i * NT, r = c / CPR, kc = (c - r * CPR) * 8;
      const int gr = m0 + r, gk = k0 + kc;
      ra[i] = (gr < M && gk < K) ? *(const uint4 *)(A + (int64_t)gr * lda + gk)
                                 : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < Cfg::B_PER_T; ++i) {
      const int c = tid + i * NT, r = c / CPR, kc = (c - r * CPR) * 8;
      const int gr = n0 + r, gk = k0 + kc;
      rb[i] = (gr < N && gk < K) ? *(const uint4 *)(Wt + (int64_t)gr * K + gk)
                                 : make_uint4(0, 0, 0, 0);
    }
  };
  auto sstore = [&](int buf) {
#pragma unroll
    for (int i = 0; i < Cfg::A_PER_T; ++i) {
      const int c = tid + i * NT, r = c / CPR, kc = (c - r * CPR) * 8;
      *(uint4 *)&smA[buf][r * LDK + kc] = ra[i];
    }
#pragma unroll
    for (int i = 0; i < Cfg::B_PER_T; ++i) {
      const int c = tid + i * NT, r = c / CPR, kc = (c - r * CPR) * 8;
      *(uint4 *)&smB[buf][r * LDK + kc] = rb[i];
    }
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  const int nk = (K + BK - 1) / BK;
  gload(0);
  sstore(0);
  __syncthreads();
  const int frow = lane & 31, fk = (lane >> 5) * 8;
  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < nk) gload((kt + 1) * BK);
#pragma unroll
    for (int kk = 0; kk < BK / 16; ++kk) {
      bf16x8 af[TM], bfr[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i)
        af[i] = *(const bf16x8 *)&smA[cur][(wm * WM + i * 32 + frow) * LDK + kk * 16 + fk];
#pragma unroll
      for (int j = 0; j < TN; ++j)
        bfr[j] = *(const bf16x8 *)&smB[cur][(wn * WN + j * 32 + frow) * LDK + kk * 16 + fk];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], bfr[j], acc[i][j], 0, 0, 0);
    }
    if (kt + 1 < nk) sstore(cur ^ 1);
    __syncthreads();
  }

  // Epilogue. 32x32 accumulator layout: lane holds column (lane & 31) and rows
  // 8*(r/4) + 4*(lane/32) + (r%4), r = 0..15.
  const int rbase = (lane >> 5) * 4;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int col = n0 + wn * WN + j * 32 + (lane & 31);
    if (col >= N) continue;
    const float bj = bias ? bias[col] : 0.0f;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = m0 + wm * WM + i * 32 + (r >> 2) * 8 + rbase + (r & 3);
        if (row >= M) continue;
        float v = gemm_epilogue(acc[i][j][r] + bj, epi);
        const int64_t off = (int64_t)row * ldc + col;
        if (residual) v += residual[off];
        if (c_bf16)
          ((uint16_t *)C)[off] = f2bf(v);
        else
          ((float *)C)[off] = v;
      }
    }
  }
}

template <int BM, int BN, int BK, int WM, int WN>
hipError_t launch(const mxk::GemmArgs &a, hipStream_t s) {
  using Cfg = GemmCfg<BM, BN, BK, WM, WN>;
  const int tiles_m = (int)((a.M + BM - 1) / BM), tiles_n = (int)((a.N + BN - 1) / BN);
  const int blocks = tiles_m * tiles_n;
  gemm_bf16_k<BM, BN, BK, WM, WN><<<blocks, Cfg::NT, 0, s>>>(
      a.A, a.lda, a.Wt, (int)a.M, (int)a.N, (int)a.K, a.bias, a.epilogue, a.residual, a.C,
      a.c_bf16, a.ldc, tiles_m, tiles_n, a.rows_dev);
  return hipGetLastError();
}

}  // namespace

namespace mxk {

// The persistent LDS-pipelined kernel (k_gemm_lds.hip) serves every call it
// can: K a multiple of 32 and at least 128 (four slabs, the deepest ring), N a
// multiple of 4, a bias, and C, bias and residual aligned for 16-byte vector
// access; the register-staged kernel above serves the rest.
template <int BM, int BN, int WGM, int WGN, int NS>
hipError_t gemm_lds_launch(const GemmArgs &a, int grid, hipStream_t s);
hipError_t gemm_lds_deep_launch(const GemmArgs &a, int grid, hipStream_t s);
hipError_t gemm_lds_128_deep_launch(const GemmArgs &a, int grid, hipStream_t s);
hipError_t gemm_lds_nc_launch(const GemmArgs &a, int grid, hipStream_t s);
hipError_t gemm_lds16_glu_launch(const GemmArgs &a, int grid, hipStream_t s);
template <int BM, int BN, int WGM, int WGN, int NS, int RB>
hipError_t gemm_lds16_launch(const GemmArgs &a, int grid, hipStream_t s);

namespace {

enum GemmPath {
  PATH_STAGED,
  PATH_LDS_256x256,
  PATH_LDS_256x192,
  PATH_LDS_128x256,
  PATH_LDS_128x128,
  PATH_LDS_256x256_DEEP,
  PATH_LDS_128x128_DEEP,
  PATH_LDS16_128x128,      // 8 waves, 128-byte slabs, one block per CU
  PATH_LDS16_64x64,        // 256-byte slabs, three slots, one block per CU
  PATH_LDS16_64x64_PAIR,   // 256-byte slabs, two slots, two blocks per CU
  PATH_LDS16_64x64_RB128,  // 128-byte slabs, four slots, two blocks per CU
  PATH_LDS16_64x128_GLU    // the gated FFN, 256-byte slabs, three slots, one block per CU
};

// The 256 x 256 tile on 128-byte slabs: a bf16 C without a residual or an
// fp32 C with one, K a multiple of 64.
bool deep_ok(const GemmArgs &a) {
  return ((a.c_bf16 && !a.residual) || (!a.c_bf16 && a.residual)) && a.K % 64 == 0;
}

bool lds_path_ok(const GemmArgs &a) {
  const uintptr_t c = (uintptr_t)a.C;
  return a.K % 32 == 0 && a.K >= 128 && a.N % 4 == 0 && a.lda % 8 == 0 && a.bias &&
         lds_offsets_fit(a.lda, a.K, 2) &&
         a.ldc % (a.c_bf16 ? 8 : 4) == 0 && c % 16 == 0 && (uintptr_t)a.bias % 16 == 0 &&
         (!a.residual || (uintptr_t)a.residual % 16 == 0);
}

// The least estimated time over the paths whose C is staged compactly
// (deep_ok). A launch of T tiles runs n = ceil(T / CUs) of them on the fullest
// CU, one after another or (two blocks per CU) in pairs, so
//   us = start + K * (pair * (n / 2) + one * (n % 2)) + n * tile
//        (+ n * res: an fp32 C with a residual),
// `one` and `pair` the cost per K of one tile on a CU and of two: constants
// fitted to products measured on an MI355X (weights rotating over eight copies),
// but for three: the 128 x 256 row's cost per K, the best of four tried; the 256
// x 256 row's cost per tile, raised from 3.28 for the sake of K below 512; and the
// 128 x 128 pairs' start, raised from 0.63, which leaves them and the 8-wave tile
// level at one tile a CU and K = 384: repeated on the same operands the pairs are
// faster (6000 x 384 x 384 7.0 us for 7.4), within a pass the 8-wave tile's three
// slabs ahead are (MiniLM 32 x 128: 301 us a batch, 311 on the pairs). Over 700
// further products (M 1 to 40,000, N 64 to 6144, K 128 to 5120; bf16, fp32 +
// residual, gated) the choice takes 0.66 of the time of the choice by tile areas
// over the 32 x 32 MFMA tiles alone, in the geometric mean, and 1.010 of the best
// tile's; none of them takes over 1.2 % longer than by area. 700 x 1024 x 4096
// takes 16.4 us for 42.2, 1500 x 768 x 768 7.9 for 11.1, 3000 x 1280 x 5120 with a
// residual 49.7 for 54.7, 300 x 768 x 128 4.5 for 4.9. The bounds on K keep a tile
// at least as deep as the ring: a ring that held slabs of three tiles would hold
// two tiles' epilogue vectors in one place. A 64-column tile over a ragged N is
// left out unmeasured.
GemmPath pick_deep(int64_t M, int64_t N, int64_t K, bool res, bool glu) {
  struct Cost {
    GemmPath path;
    int bm, bn;
    double start, one, pair, tile, res;
  };
  static const Cost costs[] = {
      {PATH_LDS_256x256_DEEP, 256, 256, 3.27, .0198, .0396, 4.00, 3.84},
      {PATH_LDS_256x192, 256, 192, 1.73, .0183, .0366, 4.54, 2.54},
      {PATH_LDS_128x256, 128, 256, 0.00, .0150, .0300, 5.11, 1.73},
      {PATH_LDS_128x128_DEEP, 128, 128, 0.85, .0103, .0135, 2.55, 2.64},
      {PATH_LDS16_128x128, 128, 128, 1.22, .0082, .0164, 2.94, 1.44},
      {PATH_LDS16_64x64_PAIR, 64, 64, 1.64, .0052, .0061, 0.86, 0.36},
      {PATH_LDS16_64x64, 64, 64, 2.16, .0036, .0072, 0.77, 1.14},
      {PATH_LDS16_64x64_RB128, 64, 64, 1.85, .0056, .0070, 0.80, 0.70}};
  const int64_t cus = cu_count();
  GemmPath best = PATH_LDS_256x256_DEEP;
  double best_t = 0.0;
  for (const Cost &c : costs) {
    const int64_t tiles = ((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn);
    const int64_t n = (tiles + cus - 1) / cus;
    // The gated FFN needs an even number of column blocks per wave. More than
    // three 64 x 64 tiles to a CU read W too often for the cost per K: 1065 x 3840
    // x 3072 with a residual takes 60 us on four, 47 on the 128 x 128 pairs.
    const bool small = !glu && N % 64 == 0 && n <= 3;
    switch (c.path) {
      case PATH_LDS_256x192:  // 96-column waves cannot pair the gated FFN's blocks
        if (glu) continue;
        break;
      case PATH_LDS16_128x128:
        if (glu || K < 256) continue;
        break;
      case PATH_LDS16_64x64:
        if (!small || K % 128 || K < 384) continue;
        break;
      case PATH_LDS16_64x64_PAIR:
        if (!small || K % 128 || K < 256) continue;
        break;
      case PATH_LDS16_64x64_RB128:
        // Only where K has no 256-byte slabs: they halve the barriers per K.
        if (!small || K % 128 == 0 || K < 256) continue;
        break;
      default: break;
    }
    const double t = c.start + (double)K * (c.pair * (double)(n / 2) + c.one * (double)(n % 2)) +
                     (double)n * (c.tile + (res ? c.res : 0.0));
    if (best_t == 0.0 || t < best_t) {
      best = c.path;
      best_t = t;
    }
  }
  if (glu && best == PATH_LDS_128x128_DEEP) {
    // Few tiles of the gated FFN: 64 x 128 ones of 16 x 16 MFMAs while each has
    // a CU (an even number of column blocks per wave, which 64 x 64 lacks). K 768,
    // N 6144: 20 rows 8.2 us for 12.5, 320 rows (240 tiles) 11.8 for 13.9.
    if (K % 128 == 0 && K >= 384 && ((M + 63) / 64) * ((N + 127) / 128) <= cus)
      return PATH_LDS16_64x128_GLU;
    // The 64-byte form keeps three slabs in flight ahead, not one: a launch of
    // a few tiles waits on every slab's load.
    if (((M + 127) / 128) * ((N + 127) / 128) * 8 <= cus) return PATH_LDS_128x128;
  }
  return best;
}

GemmPath pick(const GemmArgs &a) {
  if (!lds_path_ok(a)) return PATH_STAGED;
  static const GemmPath paths[] = {PATH_LDS_256x256, PATH_LDS_256x192, PATH_LDS_128x256,
                                   PATH_LDS_128x128};
  const int64_t m = gemm_pick_rows(a.M, a.m_hint);
  const bool glu = a.epilogue >= EPI_GLU_SILU;
  if (deep_ok(a)) return pick_deep(m, a.N, a.K, a.residual != nullptr, glu);
  // An fp32 C of few tiles (the ViT's patches): one small tile per CU, 300 x 768
  // x 768 in 5.9 us for 11.7.
  if (!a.c_bf16 && !a.residual && a.epilogue == 0 && a.K % 128 == 0 && a.K >= 384 &&
      a.N % 64 == 0 &&
      ((a.M + 63) / 64) * (a.N / 64) <= cu_count())
    return PATH_LDS16_64x64;
  int t = gemm_lds_tile(m, a.N);
  if (t == 1 && glu) t = 0;  // 96-column waves cannot pair blocks
  return paths[t];
}

}  // namespace

// The tile with the least estimated time: rounds of tiles over the CUs (the
// last round costs a whole one) times the tile's area over its relative
// throughput per unit area, measured on MI355X on the encoder's GEMM shapes
// when every tile count is a whole number of rounds (256 x 256: 1.0, 256 x
// 192: 0.88, 128 x 256: 0.86, 128 x 128: 0.65), for the products that have
// 64-byte slabs only. The 256 x 192 tile wins where N = 768 leaves 256 x
// 256 tiles at 1.5 rounds; small problems take the small tiles that spread
// over the most CUs.
int gemm_lds_tile(int64_t M, int64_t N) {
  struct Cand {
    int bm, bn;
    double eff;
  };
  const Cand cands[] = {{256, 256, 1.0}, {256, 192, 0.88}, {128, 256, 0.86},
                        {128, 128, 0.65}};
  const int64_t G = cu_count();
  int best = 3;
  double best_t = 0.0;
  for (int i = 0; i < 4; ++i) {
    const Cand &c = cands[i];
    const int64_t tiles = ((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn);
    const double t = (double)((tiles + G - 1) / G) * c.bm * c.bn / c.eff;
    if (best_t == 0.0 || t < best_t) {
      best = i;
      best_t = t;
    }
  }
  return best;
}

// The current device's CUs. A persistent launch has as many blocks, or twice as
// many for the tiles of which two share a CU.
int cu_count() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (!cached[dev]) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        n <= 0)
      n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}


const char *gemm_plan_name(int64_t M, int64_t N, int64_t K, bool c_bf16, bool residual,
                           bool i8, bool gated) {
  static const float aligned_probe[4] __attribute__((aligned(16))) = {0, 0, 0, 0};
  if (i8) {
    // The int8 kernels are the same tiles with slabs of 64 (or, deep, 128) int8.
    GemmI8Args a{};
    a.M = M;
    a.N = N;
    a.K = K;
    a.c_dtype = c_bf16 ? 1 : 0;
    a.residual = residual ? aligned_probe : nullptr;
    a.epilogue = gated ? EPI_GLU_SILU : 0;
    const bool deep = gemm_i8_deep(a);
    switch (gemm_i8_tile(a)) {
      case 0:
        return deep ? "lds_256x256x128_w64x128_ns2_persistent"
                    : "lds_256x256x64_w128x64_ns3_persistent";
      case 1: return "lds_256x192x64_w64x96_ns4_persistent";
      case 2: return "lds_128x256x64_w64x64_ns4_persistent";
      case 4: return "lds_128x128x128_w64x32_ns3_mfma16_persistent";
      case 5: return "lds_64x64x256_w32x32_ns3_mfma16_persistent";
      default: return "lds_128x128x64_w64x64_ns4_persistent";
    }
  }
  GemmArgs a{};
  a.M = M;
  a.N = N;
  a.K = K;
  a.lda = K;
  a.ldc = N;
  a.bias = aligned_probe;
  a.residual = residual ? aligned_probe : nullptr;
  a.C = (void *)aligned_probe;
  a.c_bf16 = c_bf16 ? 1 : 0;
  a.epilogue = gated ? EPI_GLU_SILU : 0;
  switch (pick(a)) {
    case PATH_LDS_256x256_DEEP: return "lds_256x256x64_w64x128_ns2_persistent";
    case PATH_LDS_128x128_DEEP: return "lds_128x128x64_w64x64_ns2_persistent";
    case PATH_LDS_256x256: return "lds_256x256x32_w128x64_ns3_persistent";
    case PATH_LDS_256x192: return "lds_256x192x32_w64x96_ns4_persistent";
    case PATH_LDS_128x256: return "lds_128x256x32_w64x64_ns4_persistent";
    case PATH_LDS_128x128: return "lds_128x128x32_w64x64_ns4_persistent";
    case PATH_LDS16_128x128: return "lds_128x128x64_w64x32_ns4_mfma16_persistent";
    case PATH_LDS16_64x64: return "lds_64x64x128_w32x32_ns3_mfma16_persistent";
    case PATH_LDS16_64x64_PAIR: return "lds_64x64x128_w32x32_ns2_mfma16_persistent";
    case PATH_LDS16_64x128_GLU: return "lds_64x128x128_w32x64_ns3_mfma16_persistent";
    case PATH_LDS16_64x64_RB128: return "lds_64x64x64_w32x32_ns4_mfma16_persistent";
    default: return "staged_128x128x64_w64x64";
  }
}

const char *gemm_config_name(int64_t M, int64_t N, int64_t K) {
  return gemm_plan_name(M, N, K, false, false, false);
}

hipError_t gemm(const GemmArgs &a, hipStream_t s) {
  if (a.epilogue & EPI_NARROW_C) {
    if (!lds_path_ok(a) || a.residual) return hipErrorInvalidValue;
    return gemm_lds_nc_launch(a, cu_count(), s);
  }
  const GemmPath p = pick(a);
  // The fused gated FFN exists only on the LDS-pipelined kernel.
  if (a.epilogue >= EPI_GLU_SILU && (p == PATH_STAGED || a.N % 64)) return hipErrorInvalidValue;
  switch (p) {
    case PATH_LDS_256x256_DEEP: return gemm_lds_deep_launch(a, cu_count(), s);
    case PATH_LDS_128x128_DEEP: return gemm_lds_128_deep_launch(a, 2 * cu_count(), s);
    case PATH_LDS16_128x128: return gemm_lds16_launch<128, 128, 2, 4, 4, 128>(a, cu_count(), s);
    case PATH_LDS16_64x64: return gemm_lds16_launch<64, 64, 2, 2, 3, 256>(a, cu_count(), s);
    case PATH_LDS16_64x128_GLU: return gemm_lds16_glu_launch(a, cu_count(), s);
    case PATH_LDS16_64x64_PAIR:
      return gemm_lds16_launch<64, 64, 2, 2, 2, 256>(a, 2 * cu_count(), s);
    case PATH_LDS16_64x64_RB128:
      return gemm_lds16_launch<64, 64, 2, 2, 4, 128>(a, 2 * cu_count(), s);
    case PATH_LDS_256x256: return gemm_lds_launch<256, 256, 2, 4, 3>(a, cu_count(), s);
    case PATH_LDS_256x192: return gemm_lds_launch<256, 192, 4, 2, 4>(a, cu_count(), s);
    case PATH_LDS_128x256: return gemm_lds_launch<128, 256, 2, 4, 4>(a, cu_count(), s);
    case PATH_LDS_128x128: return gemm_lds_launch<128, 128, 2, 2, 4>(a, cu_count(), s);
    default: return launch<128, 128, 64, 64, 64>(a, s);
  }
}

}  // namespace mxk
