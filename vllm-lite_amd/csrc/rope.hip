// Fused rotary position embedding + KV-cache write (pa_rope_reshape_and_cache)
// and the host inverse-frequency table (pa_rope_inv_freq).
//
// The reference applies RoPE to Q and K, then writes the expanded K/V into
// the cache token by token (crates/model/src/components/attention/
// rope_gqa.rs:283-302 -> paged_gqa.rs:29-63).  Here one kernel reads each
// token's Q, K and V once: Q is rotated in place, K is rotated on the way
// into the K cache, V is copied into the token-minor V cache.
#include <algorithm>
#include <cmath>

#include "pa_common.hpp"

namespace pa {
namespace {

// One workgroup per token.  Thread i of a head handles the pair
// (x[i], x[i + D/2]); heads are strided over the workgroup.
template <typename T>
__global__ __launch_bounds__(256) void rope_cache_kernel(
    T* __restrict__ q, int64_t q_stride, const T* __restrict__ key, int64_t key_stride,
    const T* __restrict__ value, int64_t value_stride, T* __restrict__ k_cache,
    T* __restrict__ v_cache, const int64_t* __restrict__ slots,
    const int64_t* __restrict__ positions, const float* __restrict__ inv_freq, int Hq, int Hkv,
    int D, int64_t num_slots) {
  const int t = blockIdx.x;
  const int half = D / 2;
  const float pos = (float)positions[t];
  const int64_t slot = slots[t];
  const bool write = slot >= 0 && slot < num_slots;
  const int64_t blk = write ? slot / kBlock : 0;
  const int off = write ? (int)(slot % kBlock) : 0;
  // Q rotation, all query heads.
  for (int e = threadIdx.x; e < Hq * half; e += blockDim.x) {
    const int h = e / half, i = e % half;
    float s, c;
    sincosf(pos * inv_freq[i], &s, &c);
    T* row = q + t * q_stride + (int64_t)h * D;
    const float x1 = Elem<T>::load(row + i), x2 = Elem<T>::load(row + half + i);
    Elem<T>::store(row + i, x1 * c - x2 * s);
    Elem<T>::store(row + half + i, x2 * c + x1 * s);
  }
  if (!write) return;
  // K rotation into the cache, V copy into the token-minor V cache.
  for (int e = threadIdx.x; e < Hkv * half; e += blockDim.x) {
    const int h = e / half, i = e % half;
    float s, c;
    sincosf(pos * inv_freq[i], &s, &c);
    const T* krow = key + t * key_stride + (int64_t)h * D;
    const float x1 = Elem<T>::load(krow + i), x2 = Elem<T>::load(krow + half + i);
    T* kd = k_cache + ((blk * Hkv + h) * kBlock + off) * (int64_t)D;
    Elem<T>::store(kd + i, x1 * c - x2 * s);
    Elem<T>::store(kd + half + i, x2 * c + x1 * s);
    const T* vrow = value + t * value_stride + (int64_t)h * D;
    T* vd = v_cache + ((blk * Hkv + h) * (int64_t)D) * kBlock + off;
    vd[(int64_t)i * kBlock] = vrow[i];
    vd[(int64_t)(half + i) * kBlock] = vrow[half + i];
  }
}

// Tiled form, for D a multiple of 16 up to 256 and 16-byte aligned rows: a
// workgroup takes 16 tokens [16 g, 16 g + 16).  Workgroups of column y < rot_cols
// rotate query and key heads: the angles of the 16 tokens' D / 2 pairs are
// formed once in LDS (a sincosf per head and pair was most of the one-token
// kernel's time), then a thread keeps the 8 pairs (8 u .. and D / 2 + 8 u ..)
// of one token in registers and rotates them head after head, 16 bytes per
// load and store.  The other workgroups copy value heads: where the tokens
// cover a whole cache block in order (a prompt's run of slots, as in
// cache_write_kernel) the token-minor block goes through LDS and leaves in
// 32-byte dim rows, else element by element.
// HBM-bound: (2 Hq + 4 Hkv) D elements per token.  7569 tokens, 14 / 2 heads x
// 64, bf16: 18.2 us (one workgroup per token, an angle per head and pair) -> 9.8; 618 tokens, 32 / 8 x
// 128: 13.4 -> 7.7.
constexpr int kTileTokens = kBlock;
template <typename T>
__global__ __launch_bounds__(256) void rope_cache_tiled_kernel(
    T* __restrict__ q, int64_t q_stride, const T* __restrict__ key, int64_t key_stride,
    const T* __restrict__ value, int64_t value_stride, T* __restrict__ k_cache,
    T* __restrict__ v_cache, const int64_t* __restrict__ slots,
    const int64_t* __restrict__ positions, const float* __restrict__ inv_freq, int T_, int Hq,
    int Hkv, int D, int64_t num_slots, int rot_cols) {
  struct __attribute__((aligned(16))) Unit {
    T v[8];
  };
  __shared__ __attribute__((aligned(16))) uint8_t lds[16 * 256 * 4];
  const int tid = threadIdx.x, t0 = blockIdx.x * kTileTokens;
  if ((int)blockIdx.y < rot_cols) {
    const int half = D / 2, units = half / 8, per_head = kTileTokens * units;
    float2* cs = reinterpret_cast<float2*>(lds);  // [16][D / 2]
    for (int e = tid; e < kTileTokens * half; e += 256) {
      const int j = e / half, i = e % half;
      float s, c;
      sincosf((float)positions[min(t0 + j, T_ - 1)] * inv_freq[i], &s, &c);
      cs[e] = float2{c, s};
    }
    __syncthreads();
    const int heads_at_once = 256 / per_head, sub = tid / per_head, e = tid % per_head;
    const int j = e / units, u = e % units, t = t0 + j;
    if (sub >= heads_at_once || t >= T_) return;
    float c[8], s[8];
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      const float2 a = cs[j * half + 8 * u + x];
      c[x] = a.x;
      s[x] = a.y;
    }
    const int64_t slot = slots[t];
    const bool write = slot >= 0 && slot < num_slots;
    const int64_t blk = write ? slot / kBlock : 0;
    const int off = write ? (int)(slot % kBlock) : 0;
    for (int h = blockIdx.y * heads_at_once + sub; h < Hq + Hkv; h += rot_cols * heads_at_once) {
      const bool is_q = h < Hq;
      if (!is_q && !write) continue;
      const T* src = (is_q ? q + t * q_stride + (int64_t)h * D
                           : key + t * key_stride + (int64_t)(h - Hq) * D) + 8 * u;
      T* dst = is_q ? q + t * q_stride + (int64_t)h * D + 8 * u
                    : k_cache + ((blk * Hkv + (h - Hq)) * kBlock + off) * (int64_t)D + 8 * u;
      const Unit a = *reinterpret_cast<const Unit*>(src);
      const Unit b = *reinterpret_cast<const Unit*>(src + half);
      Unit x, y;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float x1 = Elem<T>::load(a.v + i), x2 = Elem<T>::load(b.v + i);
        // the contraction the one-token kernel compiles to
        Elem<T>::store(x.v + i, __builtin_fmaf(x1, c[i], -(x2 * s[i])));
        Elem<T>::store(y.v + i, __builtin_fmaf(x2, c[i], x1 * s[i]));
      }
      *reinterpret_cast<Unit*>(dst) = x;
      *reinterpret_cast<Unit*>(dst + half) = y;
    }
    return;
  }
  // Value heads.  range[0] / range[1]: first token of the whole-block range that
  // begins in this workgroup's tokens' block / in the next one's, or -1.
  __shared__ int range[2];
  if (tid < 64) {
    const int h2 = (tid >> 4) & 1, j = tid & 15, tb = t0 + kTileTokens * h2;
    int start = -1;
    bool ok = false;
    if (tid < 32 && tb < T_) {
      const int64_t s0 = slots[tb];
      if (s0 >= 0 && s0 < num_slots) {
        start = tb - (int)(s0 % kBlock);
        if (start >= 0 && start + kBlock <= T_)
          ok = slots[start + j] == s0 - s0 % kBlock + j;
      }
    }
    const uint64_t bal = __builtin_amdgcn_ballot_w64(ok);
    if (tid == 0) range[0] = (bal & 0xFFFFull) == 0xFFFFull ? start : -1;
    if (tid == 16) range[1] = ((bal >> 16) & 0xFFFFull) == 0xFFFFull ? start : -1;
  }
  __syncthreads();
  const int r0 = range[0], r1 = range[1];
  const int units = D / 8, cols = gridDim.y - rot_cols;
  T* vt = reinterpret_cast<T*>(lds);  // [16 tokens][D]
  for (int h = blockIdx.y - rot_cols; h < Hkv; h += cols) {
    if (r0 >= 0) {
      const int64_t blk = slots[r0] / kBlock;
      for (int i = tid; i < kBlock * units; i += 256) {
        const int j = i / units, u = i % units;
        *reinterpret_cast<Unit*>(vt + j * D + 8 * u) = *reinterpret_cast<const Unit*>(
            value + (int64_t)(r0 + j) * value_stride + (int64_t)h * D + 8 * u);
      }
      __syncthreads();
      T* vd = v_cache + (blk * Hkv + h) * (int64_t)D * kBlock;
      for (int d = tid; d < D; d += 256) {
        Unit row[2];
#pragma unroll
        for (int j = 0; j < kBlock; ++j) row[j / 8].v[j % 8] = vt[j * D + d];
        *reinterpret_cast<Unit*>(vd + d * kBlock) = row[0];
        *reinterpret_cast<Unit*>(vd + d * kBlock + 8) = row[1];
      }
      __syncthreads();
    }
    for (int i = tid; i < kTileTokens * units; i += 256) {
      const int j = i / units, u = i % units, t = t0 + j;
      if (t >= T_) break;
      if ((r0 >= 0 && t >= r0 && t < r0 + kBlock) || (r1 >= 0 && t >= r1 && t < r1 + kBlock))
        continue;
      const int64_t slot = slots[t];
      if (slot < 0 || slot >= num_slots) continue;
      const Unit x = *reinterpret_cast<const Unit*>(value + (int64_t)t * value_stride +
                                                    (int64_t)h * D + 8 * u);
      T* vd = v_cache + ((slot / kBlock * Hkv + h) * (int64_t)D + 8 * u) * kBlock + slot % kBlock;
#pragma unroll
      for (int i2 = 0; i2 < 8; ++i2) vd[i2 * kBlock] = x.v[i2];
    }
  }
}

}  // namespace
}  // namespace pa

using namespace pa;

extern "C" int32_t pa_rope_inv_freq(int32_t head_dim, float theta, int32_t rope_type,
                                    float factor, int32_t original_max_position,
                                    int32_t cur_seq_len, const float* short_factor,
                                    const float* long_factor, float* out) {
  clear_error();
  PA_REQUIRE(head_dim > 0 && head_dim % 2 == 0, PA_ERR_INVALID_ARG,
             "pa_rope_inv_freq: head_dim %d must be even and positive", head_dim);
  PA_REQUIRE(rope_type >= PA_ROPE_DEFAULT && rope_type <= PA_ROPE_SU, PA_ERR_INVALID_ARG,
             "pa_rope_inv_freq: unknown rope type %d", rope_type);
  PA_REQUIRE(out, PA_ERR_INVALID_ARG, "pa_rope_inv_freq: null output");
  const int half = head_dim / 2;
  const bool near_one = std::fabs(factor - 1.0f) < 1.1920929e-07f;  // f32 epsilon
  const float d = (float)head_dim;
  float th = theta;
  if (rope_type == PA_ROPE_YARN && !near_one) {
    th = theta * std::pow(factor, d / (d - 2.0f));
  } else if (rope_type == PA_ROPE_DYNAMIC && original_max_position > 0 &&
             cur_seq_len > original_max_position && !near_one) {
    const float scale =
        std::fma(factor, (float)cur_seq_len / (float)original_max_position, -(factor - 1.0f));
    th = theta * std::pow(scale, d / (d - 2.0f));
  }
  for (int i = 0; i < half; ++i) out[i] = std::pow(th, -2.0f * (float)i / d);
  if (rope_type == PA_ROPE_LINEAR && !near_one)
    for (int i = 0; i < half; ++i) out[i] = out[i] / factor;
  if (rope_type == PA_ROPE_SU && original_max_position > 0) {
    int boundary = half;
    for (int i = 0; i < half; ++i)
      if (2.0f * 3.14159265358979323846f / out[i] > (float)original_max_position) {
        boundary = i;
        break;
      }
    for (int i = 0; i < half; ++i) {
      const float* f = i < boundary ? short_factor : long_factor;
      out[i] = out[i] / (f ? f[i] : 1.0f);
    }
  }
  return PA_OK;
}

extern "C" int32_t pa_rope_reshape_and_cache(void* q, int64_t q_stride, const void* key,
                                             int64_t key_stride, const void* value,
                                             int64_t value_stride, void* k_cache, void* v_cache,
                                             const int64_t* slot_mapping, const int64_t* positions,
                                             const float* inv_freq, int32_t num_tokens,
                                             int32_t num_heads, int32_t num_kv_heads,
                                             int32_t head_dim, int32_t num_blocks, int32_t dtype,
                                             pa_stream_t stream) {
  clear_error();
  PA_REQUIRE(dtype_ok(dtype), PA_ERR_INVALID_ARG, "pa_rope_reshape_and_cache: unknown dtype %d",
             dtype);
  PA_REQUIRE(num_tokens >= 0 && num_heads > 0 && num_kv_heads > 0 && head_dim > 0 &&
                 head_dim % 2 == 0 && num_blocks > 0,
             PA_ERR_INVALID_ARG, "pa_rope_reshape_and_cache: bad sizes");
  if (num_tokens == 0) return PA_OK;
  PA_REQUIRE(q && key && value && k_cache && v_cache && slot_mapping && positions && inv_freq,
             PA_ERR_INVALID_ARG, "pa_rope_reshape_and_cache: null pointer");
  if (q_stride == 0) q_stride = (int64_t)num_heads * head_dim;
  if (key_stride == 0) key_stride = (int64_t)num_kv_heads * head_dim;
  if (value_stride == 0) value_stride = (int64_t)num_kv_heads * head_dim;
  PA_REQUIRE(q_stride >= (int64_t)num_heads * head_dim &&
                 key_stride >= (int64_t)num_kv_heads * head_dim &&
                 value_stride >= (int64_t)num_kv_heads * head_dim,
             PA_ERR_INVALID_ARG, "pa_rope_reshape_and_cache: token stride too small");
  const int64_t num_slots = (int64_t)num_blocks * kBlock;
  hipStream_t s = (hipStream_t)stream;
  // 16-byte pieces of every row: aligned bases and strides.  Few tokens of at
  // most 512 rotation pairs (two per thread) stay with the one-token kernel:
  // us, one-token / tiled, bf16, 8 / 2 heads x 48: 1 token 2.5 / 3.4, 300 3.1 /
  // 3.6, 1000 3.7 / 3.8; 14 / 2 x 64: 1 token 3.0 / 3.2, 300 3.6 / 3.4, 1000 4.5 /
  // 3.7; more heads, 32 / 8 x 80 (1600 pairs): 1 token 4.8 / 3.6.
  const int es = (int)dtype_size(dtype);
  const bool few = num_tokens < 512 && (num_heads + num_kv_heads) * (int64_t)head_dim <= 1024;
  const bool tiled = !few && head_dim % 16 == 0 && head_dim <= 256 &&
                     ((uintptr_t)q | (uintptr_t)key | (uintptr_t)value | (uintptr_t)k_cache |
                      (uintptr_t)v_cache) % 16 == 0 &&
                     (q_stride * es) % 16 == 0 && (key_stride * es) % 16 == 0 &&
                     (value_stride * es) % 16 == 0;
  if (tiled) {
    // columns of workgroups over the heads: about four workgroups per CU, at
    // least one head pass each
    const int tiles = (num_tokens + kTileTokens - 1) / kTileTokens;
    const int at_once = 256 / (kTileTokens * head_dim / 16);
    const int rot = (num_heads + num_kv_heads + at_once - 1) / at_once;
    const int want = std::max(1, 1024 / tiles);
    const int rot_cols = std::min(rot, want), v_cols = std::min(num_kv_heads, want);
    const dim3 grid(tiles, rot_cols + v_cols);
    if (dtype == PA_DTYPE_BF16)
      rope_cache_tiled_kernel<uint16_t><<<grid, 256, 0, s>>>(
          (uint16_t*)q, q_stride, (const uint16_t*)key, key_stride, (const uint16_t*)value,
          value_stride, (uint16_t*)k_cache, (uint16_t*)v_cache, slot_mapping, positions, inv_freq,
          num_tokens, num_heads, num_kv_heads, head_dim, num_slots, rot_cols);
    else
      rope_cache_tiled_kernel<float><<<grid, 256, 0, s>>>(
          (float*)q, q_stride, (const float*)key, key_stride, (const float*)value, value_stride,
          (float*)k_cache, (float*)v_cache, slot_mapping, positions, inv_freq, num_tokens,
          num_heads, num_kv_heads, head_dim, num_slots, rot_cols);
  } else if (dtype == PA_DTYPE_BF16)
    rope_cache_kernel<uint16_t><<<num_tokens, 256, 0, s>>>(
        (uint16_t*)q, q_stride, (const uint16_t*)key, key_stride, (const uint16_t*)value,
        value_stride, (uint16_t*)k_cache, (uint16_t*)v_cache, slot_mapping, positions, inv_freq,
        num_heads, num_kv_heads, head_dim, num_slots);
  else
    rope_cache_kernel<float><<<num_tokens, 256, 0, s>>>(
        (float*)q, q_stride, (const float*)key, key_stride, (const float*)value, value_stride,
        (float*)k_cache, (float*)v_cache, slot_mapping, positions, inv_freq, num_heads,
        num_kv_heads, head_dim, num_slots);
  return check_launch("pa_rope_reshape_and_cache");
}
