// The choice among the tiled GEMM's tilings (gemm.hip); host code only, so that
// the rule can be tested without a GPU.
#pragma once
#include <cmath>

namespace pa {

// The tilings, and the time each would take: rounds of workgroups over the
// 256 CUs, each round `us` plus `ns_per_k` for every unit of K.  The constants
// are fitted to the measured times of full rounds (us; K 896, 4096 or 4864,
// 12288; tiles in brackets):
//   256 x 256  1 workgroup per CU   29.5 [228]  111.7 a round [768]
//   256 x 128  1 per CU             19.9 [252]   74.6 [196]  199.5 [256]
//   128 x 128  2 per CU, 2 buffers 134.6 [4256]  69.3 [392]
//   128 x 128  1 per CU, K groups   11.6 [228]   40.6 [240]  103.6 [256]
//    64 x 128  1 per CU, K groups    8.3 [216]   26.8 [168]   64.7 [224]
//    64 x  64  1 per CU, K groups    5.3 [28]    15.7 [84]    35.1 [192]
// (taken with the integer rounding in the epilogue; without it all are up to
// 7% faster).
// Over 37 shapes timed in every tiling (M 65 to 8000, N 896 to 151936, K 896
// to 12288) the smallest estimate is the fastest tiling or within a few
// percent of it.
enum Tiling { k256x256, k256x128, k128x128Pair, k128x128, k64x128, k64x64 };
inline Tiling choose_tiling(int M, int wrows, int K, bool silu) {
  constexpr int kCUs = 256;
  struct Cost {
    Tiling t;
    int bm, bn;
    float us, ns_per_k;
  };
  static constexpr Cost costs[] = {{k256x256, 256, 256, 6.5f, 25.7f}, {k256x128, 256, 128, 5.5f, 15.f},
                                   {k128x128, 128, 128, 3.4f, 8.2f},  {k64x128, 64, 128, 4.f, 4.9f},
                                   {k64x64, 64, 64, 3.1f, 2.6f}};
  auto tiles = [&](int bm, int bn) {
    return (double)((M + bm - 1) / bm) * ((wrows + bn - 1) / bn);
  };
  Tiling best = k128x128;
  double best_us = 1e30;
  // More 128 x 128 tiles than CUs: two workgroups share a CU, and whichever
  // finishes is replaced.  The last round runs one tile per CU where it is at
  // most half full (540 tiles, K 896, with bias: 30.7 us against 20 for 504 and
  // 26 in 256 x 256).  (SwiGLU stores half as many outputs per tile: 134.6 us
  // against 256 x 256's 137.9 at 7160 x 9728, where the plain epilogue loses,
  // 236.7 against 202.0 at 640 x 151936 x 896.)
  const double pair = (silu ? 3. : 4.) + 15.5e-3 * K, alone = 3. + 8.4e-3 * K;
  if (const double n = tiles(128, 128); n > kCUs) {
    const double full = std::floor(n / (2 * kCUs)), rest = n - full * 2 * kCUs;
    best = k128x128Pair;
    best_us = 3.5 + full * pair +
              (rest == 0. ? 0.
               : rest <= kCUs ? alone
                              : std::max(rest / (2 * kCUs), full > 0. ? 0. : 0.85) * pair);
  }
  for (const Cost& c : costs) {
    const double us = std::ceil(tiles(c.bm, c.bn) / kCUs) * (c.us + c.ns_per_k * 1e-3 * K);
    if (us < best_us) {
      best_us = us;
      best = c.t;
    }
  }
  return best;
}

}  // namespace pa
