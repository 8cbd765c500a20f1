// How many workgroups share a context of the decode kernels (decode.hip); host
// code only, so that the rule can be tested without a GPU.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstddef>

namespace pa {

// Workgroups per (kv head, sequence) whose results the reduce kernel merges,
// for launches whose wavefronts merge in LDS.  One workgroup streams at most
// about 43 GB/s (bf16; FP8, with one step in flight per wavefront, 36; 36 / 31
// with 32 of them running, 29 / 25 with 128), so few (kv head, sequence) pairs leave the
// chip idle, and a number of them that does not fill whole rounds of the 256
// CUs leaves it idle in the last.  More workgroups cost the reduce launch with
// its load chain (bf16 4.2 us more than the LDS merge, FP8 3.2) and 1.4% of the
// stream each.  Estimated over `ctx`
// tokens for every sequence: the launch's longest context (the others' are on
// the device), or less where that is only a bound.  The least wins, one
// workgroup where they tie.  Measured, us, one workgroup / chosen:
// bf16, 8 kv heads x 128: 1 x 2000 tokens 27.0 / 10.0, 1 x 500 9.8 / 7.5, 4 x
// 2000 32.1 / 11.3, 16 x 200-2000 27.3 / 19.6, 48 x 4096 157 / 132, 37 x
// 500-8000 120 / 91, 64 x 4096 170 / 170 (one; two workgroups 175); FP8: 37 x
// 500-8000 69 / 56, 16 x 8000 78 / 50, 1 x 2000 19 / 9.
// (With 3.2 us in bf16 too, 32 x 768 tokens over 2 kv heads x 64 were split four
// ways, 8.0 us against 7.4 in one workgroup; with 4.5, 8 x 512 over 8 kv heads x
// 128 were not, 10.4 against 8.6.)
inline int choose_splits(int num_seqs, int num_heads, int num_kv_heads, int head_dim, int ctx,
                         int elem_bytes, size_t workspace_bytes) {
  constexpr double kCUs = 256;
  const double pairs = (double)num_seqs * num_kv_heads;
  const double pair_us = 2e-3 * ctx * head_dim * elem_bytes;  // bytes / 1000: us at 1 GB/s
  const double all = elem_bytes == 1 ? 6200. : 6500.;
  auto one = [&](double wgs) {
    return (elem_bytes == 1 ? 36. : 43.) * (wgs <= 16 ? 1. : wgs <= 64 ? 0.85 : 0.68);
  };
  int best = 1;
  double best_us = 0.;
  for (int s : {1, 2, 3, 4, 6, 8, 12, 16, 24, 32}) {
    const double wgs = pairs * s;
    if (s > 1 && (ctx < 64 * s || wgs > 4096. ||
                  (size_t)num_seqs * num_heads * s * (head_dim + 2) * sizeof(float) >
                      workspace_bytes))
      break;
    const double rounds = wgs <= kCUs ? 1. : std::ceil(wgs / kCUs) * kCUs / wgs;
    double us = std::max(pairs * pair_us / all * rounds, wgs <= kCUs ? pair_us / s / one(wgs) : 0.);
    if (s > 1) us = us * (1. + 0.014 * s) + (elem_bytes == 1 ? 3.2 : 4.2);
    if (s == 1 || us < best_us) {
      best = s;
      best_us = us;
    }
  }
  return best;
}

}  // namespace pa
