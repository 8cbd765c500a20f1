// Prefill-sized linear layer: Y[M, N] = X[M, K] · W[N, K]ᵀ (bf16, f32
// accumulation) for batches of many rows (prompt chunks, mixed steps), the
// tiled MFMA GEMM behind pa_linear.
#include <algorithm>

#include "gemm_tiling.hpp"
#include "pa_common.hpp"
#include "pa_internal.hpp"

namespace pa {
namespace {

// A wavefront's copy HBM -> LDS of 16 bytes per lane: lane l's bytes come
// from base + off (off per lane) and land at LDS address lds + 16 l.  Written
// out in assembly: with the builtin the compiler cannot tell that the operand
// reads which follow use another LDS buffer, and makes them wait for the copy
// (vmcnt(0) right after every copy).  The kernel orders copies and reads
// itself (wait_copies and a barrier at the top of every step).  A load to LDS
// needs one wait state after the write of m0, which the compiler does not add
// inside assembly: the s_nop.
#pragma clang diagnostic ignored "-Winline-asm"  // m0 as a clobber
__device__ inline void lds_copy16(const uint8_t* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(off), "s"(base), "s"(lds)
               : "memory", "m0");
}
__device__ inline void lds_copy16(const uint8_t* base, uint64_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               :
               : "v"(base + off), "s"(lds)
               : "memory", "m0");
}
// Round to nearest even with the conversion instruction.
__device__ inline uint16_t to_bf16(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
// Waits until at most N of this wavefront's copies are in flight and its LDS
// reads and writes are done.
template <int N>
__device__ inline void wait_copies() {
  static_assert(N <= 63, "vmcnt range");
  __builtin_amdgcn_s_waitcnt(0x0070 | (N & 0xF) | ((N >> 4) << 14));
}

// Workgroup = KG groups of WM x WN wavefronts.  Wavefront (wm, wn) of a group
// computes TM x TN tiles of 32 x 32 (v_mfma_f32_32x32x16_bf16), so the
// workgroup tile is BM = 32 WM TM rows of X by BN = 32 WN TN rows of W.  K
// goes in steps of BK; group kg takes the kg-th part of every step, and the
// groups' sums meet in LDS at the end.  A step's X and W rows are copied
// HBM -> LDS (no register staging) into one of S buffers, S - 1 steps ahead
// of use, one barrier per step.
//
// What bounds it: a step waits for nothing as long as S - 1 steps of copies
// cover the memory latency; then the LDS operand reads (one KB per 32 rows
// and 16 of K) and the MFMAs share the time, so large tiles (each read feeds
// TM or TN MFMAs) are best where there are enough of them for every CU, and
// small outputs take small tiles, deep buffers and K groups instead (a
// long serial K over few workgroups is latency-bound).  The two-buffer
// 128 x 128 kernel this replaces ran one step of copies ahead of the compute,
// stored 8 bytes per lane straight from the accumulators and rounded to bf16
// in integer arithmetic; measured, us before -> after (M x N x K): 333 x 896
// x 4864 70.6 -> 15.9, 618 x 6144 x 4096 77.8 -> 39.1, 618 x 4096 x 4096 61.5
// -> 31.4, 7160 x 1152 x 896 with bias 28.5 -> 19.8, 7160 x 896 x 4864 87.5
// -> 62.5 (996 TFLOP/s), gate|up 333 x 9728 x 896 16.8 -> 12.1, 7160 x 9728
// x 896 146.6 -> 124.2, 2048 x 24576 x 4096 376 -> 326 (1264 TFLOP/s).
//
// LDS rows hold their 16-byte k chunks XOR-swizzled by the row's position
// above the rows that share 256 bytes, so the 16 rows an operand read serves
// at once hit 16 distinct bank slots.  The MFMAs compute the transposed tile
// (A = W, B = X): lane (n, g) = (lane % 32, lane / 32) holds X row n and, in
// register r, output column 8 (r / 4) + 4 g + r % 4.
//
// Epilogues (EPI): 0 none; 1 + bias[n]; 2 SwiGLU over a fused gate|up weight
// [2 N, K]: the tile's BN weight rows are BN/2 gate rows, then the matching
// up rows, a wavefront takes TN/2 gate tiles and their up tiles, and
// out[m][a] = silu(bf16(g)) * bf16(u).  The bf16 tile goes through LDS so
// that rows are stored (and, with add_out, the residual read) in whole
// 16-byte pieces.  Rows past M and weight rows past N are read clamped and
// not stored.
template <int EPI, int WM, int WN, int TM, int TN, int KG, int BK, int S, typename Off = uint32_t>
__global__ __launch_bounds__(64 * WM * WN * KG) void gemm_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
    const uint16_t* __restrict__ bias, int M, int N, int K, int add_out, int ntm, int ntn) {
  constexpr int NW = WM * WN * KG, NT = 64 * NW;
  constexpr int BM = 32 * WM * TM, BN = 32 * WN * TN, BNO = EPI == 2 ? BN / 2 : BN;
  constexpr int RB = BK * 2;          // bytes per tile row
  constexpr int RPC = 1024 / RB;      // rows per 1 KB copy chunk
  constexpr int LPR = RB / 16;        // lanes (16-byte chunks) per row
  constexpr int CA = BM / RPC / NW, CB = BN / RPC / NW, PER = CA + CB;  // chunks per wavefront
  static_assert(CA * NW * RPC == BM && CB * NW * RPC == BN && (EPI != 2 || TN % 2 == 0) &&
                    (EPI != 2 || (BN / 2) % RPC == 0) && (BK / 16) % KG == 0,
                "tiles");
  constexpr int STAGE = (BM + BN) * RB;
  constexpr int ORB = BNO * 2 + 16;   // bytes per row of the staged output tile
  constexpr int RED = BM * BN * 4 * (KG - 1);  // partial sums of groups 1 ..
  constexpr int SM0 = S * STAGE > BM * ORB ? S * STAGE : BM * ORB;
  constexpr int SM = SM0 > RED ? SM0 : RED;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[SM];
  __shared__ float sbias[EPI == 1 ? BN : 1];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wave / (WM * WN), wt = wave % (WM * WN);
  const int wm = wt / WN, wn = wt % WN;
  const int n = lane & 31, g = lane >> 5;
  // Tile order: workgroups are dealt round-robin to the 8 XCDs; XCD i takes
  // the i-th contiguous range of an order that goes through groups of row
  // tiles (all of them up to 8, so that W is streamed once; else 4), column
  // tiles outer within a group, so the tiles in flight on an XCD share X and
  // W rows in its L2.
  const int group_m = ntm <= 8 ? ntm : 4;
  const int total = ntm * ntn, per_xcd = (total + 7) / 8;
  const int tile = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
  if (tile >= total) return;
  const int first_m = tile / (group_m * ntn) * group_m;
  const int gsz = min(group_m, ntm - first_m), in_grp = tile % (group_m * ntn);
  const int m0 = (first_m + in_grp % gsz) * BM;
  const int c0 = in_grp / gsz * BNO;  // first output column
  auto swz = [](int r) -> int { return (r / (256 / RB)) % LPR; };
  // This wavefront's copy chunks: RPC rows each; lane l fills chunk position
  // l % LPR of row l / LPR, i.e. source chunk (l % LPR) ^ swz(row).  Scalar
  // base of the tile, lane offsets from it (Off: 32 bits, or 64 where the
  // tile's rows span more).  (A scalar base per chunk cost 5% of the
  // 256 x 256 tiling's rate.)
  const uint8_t* xb = reinterpret_cast<const uint8_t*>(x + (int64_t)m0 * K);
  const uint8_t* wb[CB];
  Off xo[CA], wo[CB];
#pragma unroll
  for (int u = 0; u < CA; ++u) {
    const int r = (CA * wave + u) * RPC + lane / LPR;
    xo[u] = (Off)min(r, M - 1 - m0) * (Off)(2 * (uint32_t)K) + ((lane % LPR) ^ swz(r)) * 16;
  }
#pragma unroll
  for (int u = 0; u < CB; ++u) {
    const int r0 = (CB * wave + u) * RPC, r = r0 + lane / LPR;
    // SwiGLU: rows BN/2 .. of the tile are up rows, N weight rows further on
    const bool up = EPI == 2 && r0 >= BN / 2;
    wb[u] = reinterpret_cast<const uint8_t*>(w + (int64_t)((up ? N : 0) + c0) * K);
    wo[u] = (Off)min(up ? r - BN / 2 : r, N - 1 - c0) * (Off)(2 * (uint32_t)K) +
            ((lane % LPR) ^ swz(r)) * 16;
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
  auto issue = [&](int kt, int buf) __attribute__((always_inline)) {
    const uint32_t la = __builtin_amdgcn_readfirstlane(lds0 + buf * STAGE + CA * wave * 1024);
    const uint32_t lb =
        __builtin_amdgcn_readfirstlane(lds0 + buf * STAGE + BM * RB + CB * wave * 1024);
#pragma unroll
    for (int u = 0; u < CA; ++u) lds_copy16(xb + (int64_t)kt * RB, xo[u], la + u * 1024);
#pragma unroll
    for (int u = 0; u < CB; ++u) lds_copy16(wb[u] + (int64_t)kt * RB, wo[u], lb + u * 1024);
  };
  // the tile's bias: loaded here, put into LDS after the steps (a wait for it
  // here would come before the first copy; older than the copies, it does not
  // disturb the steps' counts)
  static_assert(EPI != 1 || NT >= BN, "one bias value per thread");
  uint16_t bias_raw = 0;
  if (EPI == 1 && threadIdx.x < BN) bias_raw = bias[min(c0 + (int)threadIdx.x, N - 1)];
  // LDS rows of this wavefront's operand tiles (SwiGLU: gate tiles, then the
  // matching up tiles)
  int arow[TM], brow[TN];
#pragma unroll
  for (int t = 0; t < TM; ++t) arow[t] = (wm * TM + t) * 32 + n;
#pragma unroll
  for (int t = 0; t < TN; ++t)
    brow[t] = EPI == 2 ? (t < TN / 2 ? (wn * TN / 2 + t) * 32 + n
                                     : BN / 2 + (wn * TN / 2 + t - TN / 2) * 32 + n)
                       : (wn * TN + t) * 32 + n;
  f32x16 acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;
  const int nk = K / BK;
#pragma unroll
  for (int t = 0; t < S - 1; ++t)
    if (t < nk) issue(t, t);
  constexpr int SUB = BK / 16 / KG;  // MFMA steps per wavefront and K step
  for (int kt = 0, buf = 0, ibuf = S - 1; kt < nk; ++kt) {
    // this wavefront's copies of step kt have landed (near the end fewer
    // steps are in flight and all are waited for) ...
    if (nk - kt > S - 2)
      wait_copies<(S - 2) * PER>();
    else
      wait_copies<0>();
    // ... and after the barrier everyone's, and everyone is done with step
    // kt - 1, whose buffer the next copies fill
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (kt + S - 1 < nk) issue(kt + S - 1, ibuf);
    const uint8_t* at = lds + buf * STAGE;
    const uint8_t* bt = at + BM * RB;
#pragma unroll
    for (int s = 0; s < SUB; ++s) {
      bf16x8 af[TM], bfr[TN];
      const int ch = 2 * (kg * SUB + s) + g;
#pragma unroll
      for (int t = 0; t < TM; ++t)
        af[t] = *reinterpret_cast<const bf16x8*>(at + arow[t] * RB + ((ch ^ swz(arow[t])) * 16));
#pragma unroll
      for (int t = 0; t < TN; ++t)
        bfr[t] = *reinterpret_cast<const bf16x8*>(bt + brow[t] * RB + ((ch ^ swz(brow[t])) * 16));
#pragma unroll
      for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[b], af[a], acc[a][b], 0, 0, 0);
    }
    buf = buf == S - 1 ? 0 : buf + 1;
    ibuf = ibuf == S - 1 ? 0 : ibuf + 1;
  }
  if (EPI == 1 && threadIdx.x < BN) sbias[threadIdx.x] = bf16_bits_to_f32(bias_raw);
  __syncthreads();
  // the K groups' sums, in group order
  if constexpr (KG > 1) {
    float* red = reinterpret_cast<float*>(lds);
    auto slot = [&](int z, int a, int b, int q) __attribute__((always_inline)) {
      return red + (((z * WM * WN + wt) * TM * TN + a * TN + b) * 4 + q) * 256 + lane * 4;
    };
    if (kg > 0) {
#pragma unroll
      for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *reinterpret_cast<float4*>(slot(kg - 1, a, b, q)) =
                float4{acc[a][b][4 * q], acc[a][b][4 * q + 1], acc[a][b][4 * q + 2],
                       acc[a][b][4 * q + 3]};
    }
    __syncthreads();
    if (kg == 0) {
#pragma unroll
      for (int z = 0; z < KG - 1; ++z)
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
          for (int b = 0; b < TN; ++b)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const float4 v = *reinterpret_cast<const float4*>(slot(z, a, b, q));
              acc[a][b][4 * q] += v.x;
              acc[a][b][4 * q + 1] += v.y;
              acc[a][b][4 * q + 2] += v.z;
              acc[a][b][4 * q + 3] += v.w;
            }
    }
    __syncthreads();
  }
  // epilogue: the bf16 tile into LDS ...
  if (KG == 1 || kg == 0) {
    constexpr int TB = EPI == 2 ? TN / 2 : TN;
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int b = 0; b < TB; ++b)
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
          const int col = (wn * TB + b) * 32 + 8 * qd + 4 * g;
          uint16_t v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if constexpr (EPI == 2) {
              const float gg = (float)(__bf16)acc[a][b][4 * qd + e];
              const float uu = (float)(__bf16)acc[a][b + TB][4 * qd + e];
              v[e] = to_bf16(gg * __builtin_amdgcn_rcpf(1.0f + __expf(-gg)) * uu);
            } else {
              float y = acc[a][b][4 * qd + e];
              if constexpr (EPI == 1) y += sbias[col + e];
              v[e] = to_bf16(y);
            }
          }
          *reinterpret_cast<uint64_t*>(lds + arow[a] * ORB + col * 2) =
              *reinterpret_cast<const uint64_t*>(v);
        }
  }
  __syncthreads();
  // ... and from there to the output rows, 8 columns per thread at a time
  constexpr int CPRO = BNO / 8;
  for (int i = threadIdx.x; i < BM * CPRO; i += NT) {
    const int r = i / CPRO, cc = i % CPRO * 8;
    const int row = m0 + r, col = c0 + cc;
    if (row >= M || col >= N) continue;
    uint4 v = *reinterpret_cast<const uint4*>(lds + r * ORB + cc * 2);
    uint16_t* dst = out + (int64_t)row * N + col;
    auto add2 = [](uint32_t o, uint32_t y) -> uint32_t {
      return to_bf16(bf16_bits_to_f32((uint16_t)o) + bf16_bits_to_f32((uint16_t)y)) |
             (uint32_t)to_bf16(bf16_bits_to_f32((uint16_t)(o >> 16)) +
                               bf16_bits_to_f32((uint16_t)(y >> 16)))
                 << 16;
    };
    if (N % 8 == 0) {
      if (add_out) {
        const uint4 o = *reinterpret_cast<const uint4*>(dst);
        v = uint4{add2(o.x, v.x), add2(o.y, v.y), add2(o.z, v.z), add2(o.w, v.w)};
      }
      *reinterpret_cast<uint4*>(dst) = v;
    } else if (N % 4 == 0) {
      const uint2 half[2] = {uint2{v.x, v.y}, uint2{v.z, v.w}};
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        if (col + 4 * e >= N) continue;
        uint2 y = half[e];
        uint2* d = reinterpret_cast<uint2*>(dst + 4 * e);
        if (add_out) y = uint2{add2(d->x, y.x), add2(d->y, y.y)};
        *d = y;
      }
    } else {
      const uint32_t wd[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (col + e >= N) continue;
        uint16_t y = (uint16_t)(wd[e / 2] >> (16 * (e & 1)));
        if (add_out) y = to_bf16(bf16_bits_to_f32(dst[e]) + bf16_bits_to_f32(y));
        dst[e] = y;
      }
    }
  }
}

struct GemmCall {
  uint16_t* out;
  const uint16_t *x, *w, *bias;
  int M, N, K;
  bool silu, add;
  hipStream_t stream;
};

template <int WM, int WN, int TM, int TN, int KG, int BK, int S, typename Off = uint32_t>
int32_t launch(const GemmCall& c) {
  constexpr int BM = 32 * WM * TM, BN = 32 * WN * TN;
  const int bno = c.silu ? BN / 2 : BN;
  const int ntm = (c.M + BM - 1) / BM, ntn = (c.N + bno - 1) / bno;
  PA_REQUIRE((long long)ntm * ntn < (1ll << 30), PA_ERR_UNSUPPORTED, "pa_linear: %d rows", c.M);
  const dim3 grid(8 * ((ntm * ntn + 7) / 8));
  constexpr int NT = 64 * WM * WN * KG;
  if (c.silu)
    gemm_kernel<2, WM, WN, TM, TN, KG, BK, S, Off><<<grid, NT, 0, c.stream>>>(
        c.out, c.x, c.w, nullptr, c.M, c.N, c.K, 0, ntm, ntn);
  else if (c.bias)
    gemm_kernel<1, WM, WN, TM, TN, KG, BK, S, Off><<<grid, NT, 0, c.stream>>>(
        c.out, c.x, c.w, c.bias, c.M, c.N, c.K, c.add, ntm, ntn);
  else
    gemm_kernel<0, WM, WN, TM, TN, KG, BK, S, Off><<<grid, NT, 0, c.stream>>>(
        c.out, c.x, c.w, nullptr, c.M, c.N, c.K, c.add, ntm, ntn);
  return check_launch("pa_linear");
}

}  // namespace

int32_t launch_gemm(void* out, const void* x, const void* weight, const void* bias, int rows,
                    int out_features, int in_features, bool silu, bool add_out,
                    hipStream_t stream) {
  const GemmCall c{(uint16_t*)out, (const uint16_t*)x, (const uint16_t*)weight,
                   (const uint16_t*)bias, rows, out_features, in_features, silu, add_out, stream};
  const int wrows = silu ? 2 * out_features : out_features;
  const bool k128 = in_features % 128 == 0;
  // 255 rows below the 32-bit lane offsets' reach
  if (in_features >= 1 << 23) return launch<2, 1, 1, 2, 2, 64, 4, uint64_t>(c);
  switch (choose_tiling(rows, wrows, in_features, silu)) {
    case k256x256: return launch<4, 2, 2, 4, 1, 64, 2>(c);
    case k256x128: return launch<4, 2, 2, 2, 1, 64, 3>(c);
    case k128x128Pair: return launch<2, 2, 2, 2, 1, 64, 2>(c);
    case k128x128: return launch<2, 2, 2, 2, 2, 64, 4>(c);
    // K steps of 128 (one barrier per 128 of K) where K has whole ones
    case k64x128:
      return k128 ? launch<2, 2, 1, 2, 2, 128, 3>(c) : launch<2, 2, 1, 2, 1, 64, 3>(c);
    default:
      return k128 ? launch<2, 1, 1, 2, 4, 128, 4>(c) : launch<2, 1, 1, 2, 2, 64, 4>(c);
  }
}

}  // namespace pa
