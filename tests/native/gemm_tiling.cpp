// Prints the tiling that the many-rows GEMM takes for each "rows, weight rows,
// K, SwiGLU" read from stdin (vllm-lite_amd/csrc/gemm_tiling.hpp).
#include <cstdio>

#include "gemm_tiling.hpp"

int main() {
  static const char* names[] = {"256x256", "256x128", "128x128 pair", "128x128", "64x128", "64x64"};
  int m, n, k, silu;
  while (std::scanf("%d %d %d %d", &m, &n, &k, &silu) == 4)
    std::printf("%s\n", names[pa::choose_tiling(m, n, k, silu != 0)]);
}
