// Prints choose_splits (vllm-lite_amd/csrc/decode_splits.hpp) for each
// "sequences, heads, kv heads, head_dim, context, element bytes, workspace
// bytes" read from stdin.
#include <cstdio>

#include "decode_splits.hpp"

int main() {
  int b, hq, hkv, d, ctx, es;
  unsigned long long ws;
  while (std::scanf("%d %d %d %d %d %d %llu", &b, &hq, &hkv, &d, &ctx, &es, &ws) == 7)
    std::printf("%d\n", pa::choose_splits(b, hq, hkv, d, ctx, es, (size_t)ws));
}
