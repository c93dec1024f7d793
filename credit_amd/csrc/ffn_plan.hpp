// How the FFN's products run: sizes to kernels, tiles and K slices.  Host
// arithmetic alone, so that the CPU tests build it with g++
// (tests/cpp/ffn_plan_query.cpp); the kernels are ffn.hip's.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace credit {
namespace ffn {

constexpr int kBig = 256;    // rows and columns of a tile of ffn_gemm256_kernel
constexpr int kBigK = 64;    // K of a step, in every kernel
constexpr int kTileN = 128;  // columns of a tile of the other two

// How a product C[M, N] over K runs.  The slices and the skew follow from the
// sizes alone, whatever B's layout and kernel, and the slices are the same for
// (M, N) and (N, M), so that every entry point that forms a product (either
// weight layout, recomputed or saved) adds its terms in the same order.
//  - slices: K pieces.  Time of the units on 256 CUs (flat_us; unsplit, the
//    held kernel's where it can run), plus, when split, kReduceUs and the fp32
//    sums written and read at kReduceGBs.  1024 x 2048 x 8192 (128 tiles): 131
//    us on 32 256-tiles, 47 + 5 us in 2 slices; 128 x 8192 x 28672 (64 tiles):
//    472 us, 103 + 5 us in 4.  1920 x 3200 x 9600 (375 tiles) unsplit: the FFN
//    takes 339 us, 358 in 2 slices ([K, N], without the held kernel, 342 and
//    355).
//  - bm: 256 where its rounds take less by the same count; a tall step costs
//    less than two flat ones (fewer LDS bytes per MFMA), but 256 x 6144 x
//    18944 gains (245 -> 196 us) where 512 x 28672 x 8192 would leave half the
//    CUs idle (490 -> 540 us).
//  - skew: one M-tile, but for the sizes that run held in the [N, K] layout,
//    which has no skew (256 x 768 x 32896: the FFN takes 68 us there, 81 on
//    skewed tall tiles; [K, N] 78 without the skew, 80 with it).
//  - held: more tiles than CUs, unsplit, of a [N, K] B.
//  - big: likewise by time (the FFN of 1024 rows x 8192 x 28672: 783 us with it
//    against 846 on tall tiles; 512 rows, 224 tiles: 487 against 512).
struct GemmPlan {
  bool big;    // the 256-tile kernel
  int bm;      // else rows per tile of ffn_gemm_tile_kernel
  int slices;
  int skew;    // its tile columns start their slices a step apart
  bool held;   // ffn_gemm_held_kernel
};
constexpr int kGemmCus = 256;
constexpr int kMaxSlices = 16;
// Time of `units` tiles of `steps` 64-wide K-steps, from 1024-row products:
// 0.45 us a step and 6 us beside them for a 128-row tile (0.6 us where two
// share a CU), 0.85 and 8.4 us for a 256-row one, 1.55 and 10 us for the
// 256-tile kernel's.
inline double flat_us(int64_t units, int64_t steps) {
  const int64_t rounds = (units + kGemmCus - 1) / kGemmCus;
  return rounds * (steps * (rounds > 1 ? 0.6 : 0.45) + 6.0);
}
inline double tall_us(int64_t units, int64_t steps) {
  return (units + kGemmCus - 1) / kGemmCus * (steps * 0.85 + 8.4);
}
inline double big_us(int64_t units, int64_t steps) {
  return (units + kGemmCus - 1) / kGemmCus * (steps * 1.55 + 10.0);
}
// More units than CUs on ffn_gemm_held_kernel: 0.6 us a step for each of a
// CU's tiles and the 6 us once (600 tiles of 28 steps 56, measured 55; 736 of 16
// 35, 33; 1125 of 50 156, 158).
inline double held_us(int64_t units, int64_t steps) {
  return (units + kGemmCus - 1) / kGemmCus * (steps * 0.6) + 6.0;
}
// LDS that a launch of the held kernel asks for beside its own 36 KiB, to keep a
// third workgroup off each CU: 769 to 1024 tiles are two rounds of three to a
// CU, the second nearly empty, and two even rounds of two (962 tiles of 84 steps
// 247 us at three, 215 at two).  Not where the third workgroup's cover of short
// K loops is worth more, nor where rounds come out otherwise (the FFN with GEMM1
// of 825 tiles of 56 steps 306 and 296, 918 of 36 217.5 and 216, 840 of 12 78.6
// and 80.9; 736 of 16 76 and 80; 1650 of 28 249 and 253).
inline int held_extra_lds(int64_t tiles, int64_t steps) {
  return tiles > 3 * kGemmCus && tiles <= 4 * kGemmCus && steps >= 32 ? 24 << 10 : 0;
}
constexpr int64_t kSlabBytes = int64_t{64} << 20;  // most fp32 partial sums of one product

// Whether the held kernel can run an unsplit product of a [N, K] B, whichever
// of its sides is called M.
inline bool held_fits(int64_t M, int64_t N) {
  return (M / 128) * (N / 128) > kGemmCus && M > 128 && N > 128;
}

inline int gemm_slices(int64_t M, int64_t N, int64_t K) {
  constexpr double kReduceUs = 4.0, kReduceGBs = 4000.0;
  const int64_t tiles = (M / 128) * (N / 128), steps = K / kBigK;
  int best = 1;
  double best_us = 1e30;
  for (int s = 1; s <= kMaxSlices && steps / s >= 8; ++s) {
    if (s > 1 && s * M * N * 4 > kSlabBytes) break;
    double us = flat_us(tiles * s, (steps + s - 1) / s);
    if (s == 1 && held_fits(M, N) && held_us(tiles, steps) < us) us = held_us(tiles, steps);
    if (s > 1) us += kReduceUs + s * M * N * 8.0 / (kReduceGBs * 1e3);
    if (us < best_us * 0.95) {
      best = s;
      best_us = us;
    }
  }
  return best;
}

// Shapes the 256-tile kernel can take: M and N multiples of 256, K of 128, a
// tile count that is a multiple of the 8 XCDs, and operand tiles (256 * K * 2
// bytes; a [K, N] B's (K - 1) * N * 2 + 512, which every accepted shape keeps
// below 2^32) and the epilogue's R tile ((255 * N + 256) * 2 bytes) that fit
// a buffer resource.  A GEMM that scales its A rows (RMSNorm) multiplies the
// fp32 sums by rstd on these shapes and rounds x * rstd to bf16 first on every
// other one, whichever kernel runs.
inline bool big_shape(int64_t M, int64_t N, int64_t K) {
  return M % kBig == 0 && N % kBig == 0 && K % (2 * kBigK) == 0 &&
         ((M / kBig) * (N / kBig)) % 8 == 0 && K <= (1 << 22) && N <= (1 << 22);
}

inline GemmPlan gemm_plan(int64_t M, int64_t N, int64_t K, bool kn) {
  GemmPlan p{false, 128, gemm_slices(M, N, K), 0, false};
  const int64_t steps = K / kBigK / p.slices, tiles = (M / 128) * (N / 128) * p.slices;
  double us = flat_us(tiles, steps);
  if (M % 256 == 0 && K <= (1 << 22) && tall_us(tiles / 2, steps) < us) {
    p.bm = 256;
    us = tall_us(tiles / 2, steps);
  }
  const bool held = p.slices == 1 && held_fits(M, N) && held_us(tiles, steps) < us;
  p.skew = M == p.bm && !held;
  if (held && !kn) {
    p.held = true;
    us = held_us(tiles, steps);
  }
  if (p.slices == 1 && big_shape(M, N, K) && big_us(tiles / 4, steps) < us) {
    p.big = true;
    p.held = false;
  }
  return p;
}

// Bytes of a product's partial sums.
inline size_t part_bytes(int64_t M, int64_t N, int64_t K) {
  const int64_t slices = gemm_slices(M, N, K);
  return slices > 1 ? static_cast<size_t>(slices * M * N) * sizeof(float) : 0;
}

}  // namespace ffn
}  // namespace credit
