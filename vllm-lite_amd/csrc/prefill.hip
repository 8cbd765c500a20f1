// Chunked causal prefill attention over the paged KV cache (pa_prefill).
//
// Query row i of sequence s sits at absolute position past[s] + i and
// attends keys 0 .. past[s] + i, all read through the block table.  One
// kernel covers fresh prefill (past = 0) and continuation (past > 0).
//
//  * prefill_mfma_kernel (bf16, D in {64, 128, 256}): each wavefront owns
//    NT * 16 consecutive query rows of one head and streams the keys two
//    16-token blocks at a time.  Sᵀ = K·Qᵀ and Oᵀ = Vᵀ·Pᵀ run on
//    v_mfma_f32_16x16x32_bf16 with the query rows as the N dimension; the
//    lane that receives score (key, row) from the first product is the lane
//    that feeds it to the second, so P never leaves registers.  Online
//    softmax per query row; the causal mask is only evaluated on steps that
//    straddle the diagonal.  Four wavefronts per workgroup cover adjacent
//    row ranges of the same head so their K/V reads share the L1/L2.
//  * prefill_f32_kernel (f32, D in {16 .. 256}): the same products on the f32
//    MFMA, with the keys split over wavefronts.
//  * prefill_generic_kernel (f32 or bf16, any D <= 512): one wavefront per
//    (query row, head), reference-grade.
#include <algorithm>
#include <type_traits>

#include "pa_common.hpp"
#include "pa_internal.hpp"

namespace pa {
namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNegBig = -1.0e30f;

__device__ inline float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ inline float shfl_xor_f(float x, int mask) { return __shfl_xor(x, mask, 64); }
// Max of three as one v_max3_f32.  fmaxf on values the compiler cannot prove
// canonical gets a quieting v_max_f32 x, x per operand first; MFMA results
// need none (their NaNs are quiet), and the IEEE-mode instruction returns the
// same value fmaxf does for them.  (Measured on the tiled prefill: the eight
// quieting instructions a step cost 1.1%.)
__device__ inline float max3_raw(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// A sequence's query rows and past length as the kernels use them.  The
// offsets are device data: they are clamped to the rows the call owns
// ([0, total_q)) and to max_q rows per sequence (the grid is sized for
// that), and a past outside [0, 2^30] is clamped into it, so inconsistent
// offsets (a caller error) never move a read or write outside q and out.
struct QRange {
  int begin, len, past;
};
__device__ inline QRange q_range(const int32_t* __restrict__ cu_q,
                                 const int32_t* __restrict__ past_lens, int seq, int total_q,
                                 int max_q) {
  const int b = min(max(cu_q[seq], 0), total_q);
  const int e = min(max(cu_q[seq + 1], b), total_q);
  return {b, min(e - b, max_q), min(max(past_lens[seq], 0), 1 << 30)};
}

constexpr int kWaves = 4;
template <int V>
using IC = std::integral_constant<int, V>;

// Lane layout as in decode_mfma_kernel (lane = 16 j + c):
//   QK:  A = K block (row = key c), B = Qᵀ (col = query row c of tile nt)
//        -> lane holds Sᵀ[key 4j + r][row c]
//   PV:  A = Vᵀ (row = dim 16 dt + c), B = Pᵀ, reduction slots 8j + r and
//        8j + 4 + r = key 4j + r of the step's first / second block
//        -> lane holds Oᵀ[dim 16 dt + 4j + r][row c]
template <int D, int NT>
__global__ __launch_bounds__(64 * kWaves) void prefill_mfma_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc,
    const uint16_t* __restrict__ vc, const int32_t* __restrict__ block_tables, int mbs,
    const int32_t* __restrict__ cu_q, const int32_t* __restrict__ past_lens, int Hq, int Hkv,
    int num_blocks, float scale_log2, int64_t q_row, int total_q, int max_q) {
  constexpr int KS = D / 32;
  constexpr int DT = D / 16;
  constexpr int ROWS = 16 * NT;  // query rows per wavefront
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 15, j = lane >> 4;
  const int h = blockIdx.y, seq = blockIdx.z;
  const int G = Hq / Hkv, kvh = h / G;
  const QRange qr = q_range(cu_q, past_lens, seq, total_q, max_q);
  const int q_begin = qr.begin;
  const int qlen = qr.len;
  const int row0 = (blockIdx.x * kWaves + wave) * ROWS;
  if (row0 >= qlen) return;
  const int past = qr.past;
  const int row_end = min(qlen, row0 + ROWS);
  const int kv_len = min(past + row_end, mbs * kBlock);  // keys this wavefront needs
  const int nblk = (kv_len + kBlock - 1) / kBlock;

  bf16x8 qv[NT][KS];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int row = row0 + 16 * nt + c;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if (row < qlen)
        qv[nt][s] = *reinterpret_cast<const bf16x8*>(
            q + (int64_t)(q_begin + row) * q_row + (int64_t)h * D + 32 * s + 8 * j);
      else
        qv[nt][s] = bf16x8{};
    }
  }

  f32x4 o[NT][DT];
  float m[NT], lsum[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    m[nt] = kNegBig;
    lsum[nt] = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[nt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  const int32_t* btab = block_tables + (int64_t)seq * mbs;
  const int64_t head_stride = (int64_t)kBlock * D;
  const int diag_key = past + row0;  // keys above this need the causal test

  for (int ib = 0; ib < nblk; ib += 2) {
    const int kb = ib * kBlock;
    int32_t b0 = btab[ib];
    const bool has1 = ib + 1 < nblk;
    int32_t b1 = has1 ? btab[ib + 1] : b0;
    const int rem = kv_len - kb;
    int lim0 = rem < kBlock ? rem : kBlock;
    int lim1 = has1 ? (rem - kBlock < kBlock ? rem - kBlock : kBlock) : 0;
    if (b0 < 0 || b0 >= num_blocks) { b0 = 0; lim0 = 0; }
    if (b1 < 0 || b1 >= num_blocks) { b1 = 0; lim1 = 0; }

    const uint16_t* k0 = kc + ((int64_t)b0 * Hkv + kvh) * head_stride + c * D + 8 * j;
    const uint16_t* k1 = kc + ((int64_t)b1 * Hkv + kvh) * head_stride + c * D + 8 * j;
    bf16x8 ka[KS], kb8[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      ka[s] = *reinterpret_cast<const bf16x8*>(k0 + 32 * s);
      kb8[s] = *reinterpret_cast<const bf16x8*>(k1 + 32 * s);
    }
    const uint16_t* v0 = vc + ((int64_t)b0 * Hkv + kvh) * head_stride + c * kBlock + 4 * j;
    const uint16_t* v1 = vc + ((int64_t)b1 * Hkv + kvh) * head_stride + c * kBlock + 4 * j;
    uint64_t va[DT], vb[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      va[dt] = *reinterpret_cast<const uint64_t*>(v0 + dt * 16 * kBlock);
      vb[dt] = *reinterpret_cast<const uint64_t*>(v1 + dt * 16 * kBlock);
    }
    const bool partial = lim0 < kBlock || lim1 < kBlock;
    if (partial) {
      const int n0 = min(max(lim0 - 4 * j, 0), 4), n1 = min(max(lim1 - 4 * j, 0), 4);
      const uint64_t mk0 = n0 >= 4 ? ~0ull : ((1ull << (16 * n0)) - 1);
      const uint64_t mk1 = n1 >= 4 ? ~0ull : ((1ull << (16 * n1)) - 1);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        va[dt] &= mk0;
        vb[dt] &= mk1;
      }
    }
    const bool diag = kb + 2 * kBlock - 1 > diag_key;  // wave-uniform

    bf16x8 pb[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[s], qv[nt][s], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kb8[s], qv[nt][s], s1, 0, 0, 0);
      }
      float x[8];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        x[r] = s0[r] * scale_log2;
        x[4 + r] = s1[r] * scale_log2;
      }
      if (partial || diag) {
        const int row_pos = past + row0 + 16 * nt + c;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int k_a = kb + 4 * j + r, k_b = k_a + kBlock;
          if (4 * j + r >= lim0 || k_a > row_pos) x[r] = -INFINITY;
          if (4 * j + r >= lim1 || k_b > row_pos) x[4 + r] = -INFINITY;
        }
      }
      float bm = x[0];
#pragma unroll
      for (int i = 1; i < 8; ++i) bm = fmaxf(bm, x[i]);
      bm = fmaxf(bm, shfl_xor_f(bm, 16));
      bm = fmaxf(bm, shfl_xor_f(bm, 32));
      if (__builtin_amdgcn_ballot_w64(bm > m[nt] + 8.0f)) {
        const float mn = fmaxf(m[nt], bm);
        const float a = fast_exp2(m[nt] - mn);
        m[nt] = mn;
        lsum[nt] *= a;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[nt][dt] *= a;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float p = fast_exp2(x[i] - m[nt]);
        lsum[nt] += p;
        pb[nt][i] = (__bf16)p;
      }
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const uint64_t pair[2] = {va[dt], vb[dt]};
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(pair);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        o[nt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pb[nt], o[nt][dt], 0, 0, 0);
    }
  }

#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    float l = lsum[nt];
    l += shfl_xor_f(l, 16);
    l += shfl_xor_f(l, 32);
    const int row = row0 + 16 * nt + c;
    if (row >= qlen) continue;
    const float inv = l != 0.f ? 1.f / l : 0.f;
    uint16_t* orow = out + ((int64_t)(q_begin + row) * Hq + h) * D + 4 * j;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      uint16_t w[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) w[r] = f32_to_bf16_bits(o[nt][dt][r] * inv);
      *reinterpret_cast<uint64_t*>(orow + 16 * dt) = *reinterpret_cast<const uint64_t*>(w);
    }
  }
}

// ---------------------------------------------------------------------------
// LDS-tiled MFMA prefill (bf16, D in {64, 128}).
//
// Workgroup = W wavefronts sharing one kv head.  Keys are streamed in tiles
// of 64 (4 cache blocks).  Each tile of K and V is copied HBM -> LDS once per
// workgroup with global_load_lds (no register staging) into one of three or
// four LDS buffers, two or three tiles ahead of use, and read by all
// wavefronts.  A wavefront owns 16 * NT query rows (NT MFMA column tiles) of
// one query head; with group size G the workgroup covers min(G, 4) heads of
// the group.  KG = 1: every wavefront works on whole tiles, the workgroup on
// 256 query rows (NT = 2, W = 8; a wavefront stays within 256 registers, so
// two share each SIMD and one's softmax overlaps the other's MFMAs), so
// every K/V byte brought into LDS feeds 256 rows.  KG = 2, for launches that
// would leave CUs idle: half the wavefronts take the first 32 keys of each
// tile and half the second, for 128 (NT = 2) or 64 (NT = 1) query rows, and
// the two groups' results meet in LDS at the end.
//
// Per wavefront the 32-key steps form a software pipeline: the Sᵀ = K·Qᵀ
// products of step n + 1 are issued in the same basic block as the
// exponentials and the Oᵀ += Vᵀ·Pᵀ products of step n, so the matrix core
// works while the VALU computes the softmax.  The row max is kept stale
// until a score exceeds it by 2^8; only then (rarely) is the exact max
// formed across lanes and the accumulator rescaled.  The softmax
// denominators are accumulated by one more MFMA per column tile with an
// all-ones operand, which keeps them off the VALU.
//
// LDS layouts (16-byte units, XOR-swizzled so the operand reads of 16 lanes
// hit distinct banks):
//   K tile [64 keys][D]: key row r, 16-byte chunk ch stored at chunk
//     position ch ^ (r % (D / 8)).
//   V tile [4 blocks][D][16]: the two 16-byte halves of a 32-byte dim row d
//     are swapped when bits 2 and 3 of d differ.
//
// Sequences whose tiles a launch numbers through (see the work items below).
constexpr int kMaxSeqs = 256;
template <int D, int NT, int W, int KG, typename TC>
__global__ __launch_bounds__(64 * W) void prefill_tiled_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ q, const TC* __restrict__ kc,
    const TC* __restrict__ vc, const int32_t* __restrict__ block_tables, int mbs,
    const int32_t* __restrict__ cu_q, const int32_t* __restrict__ past_lens, int Hq, int Hkv, int G,
    int num_blocks, float scale_log2, int B, int tiles_per_seq, int head_groups, int64_t q_row,
    int total_q, int max_q) {
  constexpr int KS = D / 32;   // QK reduction steps
  constexpr int DT = D / 16;   // PV output tiles
  // Cache elements: bf16 (TC = uint16_t) or FP8-E4M3 (TC = uint8_t), the
  // latter converted to bf16 (exactly) as operand fragments are read.
  constexpr bool FP8 = sizeof(TC) == 1;
  constexpr int ES = sizeof(TC);
  constexpr int CPR = D * ES / 16;  // 16-byte chunks per K row
  constexpr int KT = 64;       // keys per LDS tile
  // LDS tile buffers, and how many tiles ahead of use a tile is copied.  KG =
  // 2 has half the work per tile to cover a copy's latency.
  constexpr int NBUF = KG == 2 && !FP8 ? 4 : 3;
  constexpr int AHEAD = FP8 ? 3 : NBUF - 1;
  constexpr int TILE_BYTES = KT * D * ES;  // one K (or V) tile
  constexpr int NCH = TILE_BYTES / 1024;   // 1 KB copy chunks per tile
  constexpr int DMA_PER_WAVE = NCH >= W ? NCH / W : 1;
  constexpr int DMA_WAVES = NCH >= W ? W : NCH;  // wavefronts that copy
  constexpr int RPI = 64 / CPR;              // K rows per 1 KB chunk
  constexpr int CPB = D * kBlock * ES / 1024;  // 1 KB chunks per V block
  // 1 KB chunk i of a K tile and of a V tile lie in the same cache block
  // (i / CPB), and a wavefront's chunks stay within one block
  static_assert(RPI * CPB == kBlock && CPB % DMA_PER_WAVE == 0, "one block per wavefront copy");
  // Compute tiles are bf16 for both cache types: an FP8 tile is copied
  // into the staging area `stage` (its own layout, below) and converted to
  // bf16 once per workgroup at the tile boundary, so the per-step fragment
  // reads and the inner loop are those of the bf16 kernel.
  constexpr int CT_BYTES = KT * D * 2;  // one bf16 K (or V) compute tile
  __shared__ __attribute__((aligned(1024))) uint8_t smem[2][NBUF][CT_BYTES];
  __shared__ __attribute__((aligned(1024))) uint8_t stage[FP8 ? 2 : 1][2][FP8 ? TILE_BYTES : 16];

  const int lane = threadIdx.x & 63;
  const int wave_s = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
  const int c = lane & 15, j = lane >> 4;
  // G query heads per kv head, HW of them per workgroup, TT query tokens per
  // workgroup (a power of two; quotients by runtime values are kept out of
  // the way of a short launch, ~200 cycles each)
  const int HW = G < 4 ? G : 4;
  constexpr int TSH = NT * (W / KG / 4) == 4 ? 6 : NT * (W / KG / 4) == 2 ? 5 : 4;
  static_assert(16 * NT * (W / KG / 4) == 1 << TSH, "query tokens per workgroup");
  const int tsh = TSH + (HW == 1 ? 2 : HW == 2 ? 1 : 0), TT = 1 << tsh;
  auto tiles_of = [&](int len) -> int { return (len + TT - 1) >> tsh; };

  // Work items: a query tile (TT tokens) of a sequence for one kv head
  // (group).  Only tiles that hold query rows count: the sequences' tiles are
  // numbered through, sequences with the most keys first and within one the
  // later (longer) tiles first, by ranks and prefix sums that every workgroup
  // forms in LDS (up to kMaxSeqs sequences; beyond, in index order with the
  // empty tiles of the shorter sequences among them).
  // The items of one kv head group go to one XCD (workgroups are dealt
  // round-robin to the 8 XCDs, so workgroup g runs on XCD g % 8), whose L2
  // then holds its K/V: with fewer groups than XCDs, a group's items are dealt
  // in turn to its share of the XCDs.  The grid is persistent (about one
  // workgroup per CU): the XCD's workgroups take its items in rounds of
  // nslot, the workgroup in slot s taking item s of even rounds and item
  // nslot - 1 - s of odd rounds (longest first, so this pairs long and short
  // ones); the workgroups stay on neighbouring items (the same sequence's
  // K/V) and none waits for a CU behind a long-running one.
  // (Numbering max_q / TT tiles for every sequence instead, the single valid
  // tiles of short sequences met the same few workgroups in every round: 29
  // decode rows beside a 512-token chunk took 137 us; 32 prompts of 64 to 512
  // tokens over 2 kv heads, where a group's two XCDs also got its longer and
  // its shorter half, 47 us.  Other numbers of groups than 1, 2, 4 and 8 are
  // still cut into eight contiguous parts; 32 such prompts, heads of 128, four
  // per kv head, by kv heads: 5 73 us, 6 72, 8 85, 10 114, 12 136.)
  __shared__ int rank_seq[kMaxSeqs], rank_begin[kMaxSeqs], rank_len[kMaxSeqs],
      rank_past[kMaxSeqs], rank_tile0[kMaxSeqs], rank_of[kMaxSeqs], tile0_of[kMaxSeqs];
  __shared__ int tiles_in_all;
  const bool compact = B <= kMaxSeqs;
  if (compact) {
    // each wavefront compares its share of the sequences (held a lane each
    // and read lane by lane) with all of them; the counts meet in LDS
    for (int b = threadIdx.x; b < B; b += 64 * W) rank_of[b] = tile0_of[b] = 0;
    __syncthreads();
    for (int o0 = 0; o0 < B; o0 += 64) {
      const QRange ro = q_range(cu_q, past_lens, min(o0 + lane, B - 1), total_q, max_q);
      const int okey = ro.past + ro.len, otiles = tiles_of(ro.len), n = min(B - o0, 64);
      for (int b0 = 0; b0 < B; b0 += 64) {
        const int b = b0 + lane;
        int key = okey;
        if (b0 != o0) {
          const QRange r = q_range(cu_q, past_lens, min(b, B - 1), total_q, max_q);
          key = r.past + r.len;
        }
        int rank = 0, before = 0;
        for (int i = wave_s; i < n; i += W) {
          const int ko = __builtin_amdgcn_readlane(okey, i);
          const bool first = ko > key || (ko == key && o0 + i < b);
          rank += first;
          before += first ? __builtin_amdgcn_readlane(otiles, i) : 0;
        }
        if (b < B && rank > 0) {
          atomicAdd(&rank_of[b], rank);
          atomicAdd(&tile0_of[b], before);
        }
      }
    }
    __syncthreads();
    for (int b = threadIdx.x; b < B; b += 64 * W) {
      const QRange r = q_range(cu_q, past_lens, b, total_q, max_q);
      const int rank = rank_of[b], before = tile0_of[b];
      rank_seq[rank] = b;
      rank_begin[rank] = r.begin;
      rank_len[rank] = r.len;
      rank_past[rank] = r.past;
      rank_tile0[rank] = before;
      if (rank == B - 1) tiles_in_all = before + tiles_of(r.len);
    }
    __syncthreads();
  }
  const int nq = compact ? tiles_in_all : B * tiles_per_seq;  // tiles per kv head group
  const int nkg = Hkv * head_groups;
  const int xcd = (int)(blockIdx.x % 8), nslot = (int)(gridDim.x / 8), slot = (int)(blockIdx.x / 8);
  // the XCD's items: item i is tile (t0 + i * dt) % nq of group g0 + (t0 + i * dt) / nq
  // (the quotient is 0 where the XCD has one group)
  int g0 = 0, t0 = 0, dt = 1, items;
  if (nkg == 1 || nkg == 2 || nkg == 4 || nkg == 8) {
    const int sh = nkg == 1 ? 3 : nkg == 2 ? 2 : nkg == 4 ? 1 : 0;
    dt = 1 << sh;
    g0 = xcd >> sh;
    t0 = xcd & (dt - 1);
    items = t0 < nq ? (nq - t0 + dt - 1) >> sh : 0;
  } else {
    const int total = nkg * nq, per_xcd = (total + 7) / 8;
    t0 = min(total, xcd * per_xcd);
    items = min(total, t0 + per_xcd) - t0;
  }

  // One work item: attention for one (kv head group, sequence, query tile).
  auto process = [&](int item) {
  int kvhg = g0, qt = t0 + item * dt;
  if (qt >= nq) {
    kvhg += qt / nq;
    qt %= nq;
  }
  // every wavefront is done with the previous item's LDS tiles
  __syncthreads();
  int seq, tile;
  QRange qr;
  if (compact) {
    // the last rank whose tiles begin at or before this one
    int r = -1;
    for (int b0 = 0; b0 < B; b0 += 64)
      r += __builtin_popcountll(__builtin_amdgcn_ballot_w64(
          b0 + lane < B && rank_tile0[min(b0 + lane, B - 1)] <= qt));
    seq = __builtin_amdgcn_readfirstlane(rank_seq[r]);
    qr.begin = __builtin_amdgcn_readfirstlane(rank_begin[r]);
    qr.len = __builtin_amdgcn_readfirstlane(rank_len[r]);
    qr.past = __builtin_amdgcn_readfirstlane(rank_past[r]);
    tile = tiles_of(qr.len) - 1 - (qt - __builtin_amdgcn_readfirstlane(rank_tile0[r]));
  } else {
    seq = qt / tiles_per_seq;
    tile = tiles_per_seq - 1 - qt % tiles_per_seq;
    qr = q_range(cu_q, past_lens, seq, total_q, max_q);
  }
  int kvh = kvhg, hg = 0;
  if (head_groups > 1) {
    kvh = kvhg / head_groups;
    hg = kvhg % head_groups;
  }
  const int q_begin = qr.begin;
  const int qlen = qr.len;
  const int tok0 = tile * TT;
  if (tok0 >= qlen) return;  // uniform over the workgroup
  const int past = qr.past;
  const int key_end = min(past + min(qlen, tok0 + TT), mbs * kBlock);
  const int n_kt = (key_end + KT - 1) / KT;
  const int nblk = (key_end + kBlock - 1) / kBlock;

  // KG = 2: wavefronts W/2 .. take the second 32 keys of every tile
  const int kgrp = KG == 2 ? wave_s / (W / 2) : 0, wt = KG == 2 ? wave_s % (W / 2) : wave_s;
  const int tsub = (wt * (HW == 4 ? 8 : HW == 3 ? 11 : HW == 2 ? 16 : 32)) >> 5;  // wt / HW
  const int hl = wt - tsub * HW;
  const int head_in_group = hg * 4 + hl;
  const bool wave_active = tsub < (TT / (16 * NT)) && head_in_group < G;
  const int head = kvh * G + head_in_group;
  const int r0 = tok0 + tsub * 16 * NT;  // first query row of this wavefront
  const bool rows_active = wave_active && r0 < qlen;

  // Block ids.  Each wavefront's HBM -> LDS copies of a tile all read one
  // cache block (block `wblk` of the tile's 4), so a wavefront needs just
  // that id per tile: lane t of `ids` holds it for tile ids_base + t, loaded
  // for 64 tiles at a time with one vector load (at the item's start, then
  // every 64 tiles), and each tile takes it with a lane read.  (A scalar load
  // per tile, through the same counter as the LDS reads, made the step wait
  // for all its LDS reads at the load.)  The index is clamped to
  // the sequence's last block (keys past key_end are masked and their V
  // zeroed) and an id outside the pool reads block 0.  Whether any id of the
  // item's table lies outside the pool is found once per item (`bad_ids`);
  // only then are a tile's per-block validity bits needed (slow path).
  const int32_t* btab = block_tables + (int64_t)seq * mbs;
  const int64_t head_stride = (int64_t)kBlock * D;
  const int wblk = (wave_s * DMA_PER_WAVE) / CPB;
  auto load_ids = [&](int base) -> int32_t {
    const int t = base + lane;
    if (t >= n_kt) return 0;
    const int32_t id = btab[min(t * (KT / kBlock) + wblk, max(nblk - 1, 0))];
    return (id >= 0 && id < num_blocks) ? id : 0;
  };
  int ids_base = 0;
  int32_t ids = load_ids(0);
  // The query rows (clamped: unconditional loads, all in flight together
  // with the ids; converted after the first tiles' copies are issued) and
  // the check of the table's ids.
  bf16x8 qv[NT][KS];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int row = min(r0 + 16 * nt + c, qlen - 1);
    const uint16_t* qp = q + (int64_t)(q_begin + row) * q_row +
                         (int64_t)(kvh * G + min(head_in_group, G - 1)) * D + 8 * j;
#pragma unroll
    for (int s = 0; s < KS; ++s) qv[nt][s] = *reinterpret_cast<const bf16x8*>(qp + 32 * s);
  }
  int bad = 0;
  for (int b = threadIdx.x; b < nblk; b += 64 * W) {
    const int32_t id = btab[b];
    bad |= (id < 0 || id >= num_blocks) ? 1 : 0;
  }
  bool bad_ids = false;  // set after the first copies are issued
  auto fetch_id = [&](int kt) -> int32_t {
    if (kt - ids_base >= 64) {  // wavefront-uniform
      ids_base = kt & ~63;
      ids = load_ids(ids_base);
    }
    return __builtin_amdgcn_readlane(ids, kt - ids_base);
  };
  auto tile_valid = [&](int kt) -> int {
    if (!bad_ids) return (1 << (KT / kBlock)) - 1;
    int v = 0;
#pragma unroll
    for (int b = 0; b < KT / kBlock; ++b) {
      const int bi = kt * (KT / kBlock) + b;
      const int32_t id = bi < nblk ? btab[bi] : -1;
      v |= (id >= 0 && id < num_blocks) ? (1 << b) : 0;
    }
    return v;
  };
  // K row swizzle: 16-byte chunk ch of tile row r sits at chunk position
  // ch ^ kswz(r).  The rows one QK operand read touches (see qk) differ in
  // bits 0-1 and 3-4, which kswz spreads over distinct chunk positions.
  auto kswz = [](int r) -> int {
    constexpr int CPR2 = D * 2 / 16;  // 16-byte chunks per bf16 K row
    return CPR2 >= 16 ? (r & 3) | (((r >> 3) & 3) << 2) : (r & 3) | (((r >> 3) & 1) << 2);
  };
  // V row swizzle: the two 16-byte halves of dim row d are swapped when
  // bit 2 of d is set.  (Measured read rates of the operand pattern, per CU:
  // ~175 B/clk with this swizzle or none, ~100 B/clk when bit 3 takes part.)
  auto vswz = [](int d) -> int { return (d >> 2) & 1; };
  // FP8 K rows (D bytes) are read in 8-byte units (one MFMA fragment); unit
  // u of row r sits at unit position u ^ fsw(r).  Bit 0 is never flipped,
  // so an aligned 16-byte pair of units stays contiguous (one copy lane),
  // and the 32 lanes served together hit distinct bank pairs.  FP8 V dim
  // rows are 16 bytes and need no swizzle.
  auto fsw = [](int r) -> int {
    return D >= 128 ? (((r >> 1) & 1) << 1) | (((r >> 3) & 3) << 2) : ((r >> 3) & 3) << 1;
  };
  // Per-lane element offsets of this wavefront's HBM -> LDS copies (the
  // same for every tile).
  int koff[DMA_PER_WAVE], voff[DMA_PER_WAVE];
#pragma unroll
  for (int i0 = 0; i0 < DMA_PER_WAVE; ++i0) {
    const int i = wave_s * DMA_PER_WAVE + i0;  // 1 KB chunk of the tile
    const int r = i * RPI + lane / CPR;
    if constexpr (FP8) {
      koff[i0] = (r % kBlock) * D + ((lane % CPR) ^ (fsw(r) >> 1)) * 16;
      voff[i0] = ((i % CPB) * 64 + lane) * kBlock;
    } else {
      koff[i0] = (r % kBlock) * D + ((lane % CPR) ^ kswz(r)) * 8;
      const int d = (i % CPB) * 32 + lane / 2;
      voff[i0] = d * kBlock + ((lane & 1) ^ vswz(d)) * 8;
    }
  }
  // Issues this wavefront's share of the HBM -> LDS copies of a key tile
  // into LDS buffer `buf`; `id` is the cache block those copies read.
  auto issue_tile = [&](int32_t id, int buf) {
    const int64_t boff = ((int64_t)id * Hkv + kvh) * head_stride;
    const TC* kbase = kc + boff;
    const TC* vbase = vc + boff;
    if (NCH < W && wave_s >= DMA_WAVES) return;  // the tile has fewer chunks than wavefronts
#pragma unroll
    for (int i0 = 0; i0 < DMA_PER_WAVE; ++i0) {
      const int i = wave_s * DMA_PER_WAVE + i0;
      __builtin_amdgcn_global_load_lds(
          (const void*)(kbase + koff[i0]),
          (__attribute__((address_space(3))) void*)(FP8 ? &stage[buf & 1][0][i * 1024]
                                                        : &smem[0][buf][i * 1024]),
          16, 0, 0);
      __builtin_amdgcn_global_load_lds(
          (const void*)(vbase + voff[i0]),
          (__attribute__((address_space(3))) void*)(FP8 ? &stage[buf & 1][1][i * 1024]
                                                        : &smem[1][buf][i * 1024]),
          16, 0, 0);
    }
  };
  // Waits until at most `n` (0 to 2) tiles' copies of this wavefront are in
  // flight.
  auto wait_tiles = [&](int n) __attribute__((always_inline)) {
    constexpr int P = 2 * DMA_PER_WAVE;
    static_assert(2 * P < 64, "vmcnt");
    if (n >= 2)
      __builtin_amdgcn_s_waitcnt(0x0F70 | ((2 * P) & 0xF) | (((2 * P) >> 4) << 14));
    else if (n == 1)
      __builtin_amdgcn_s_waitcnt(0x0F70 | (P & 0xF) | ((P >> 4) << 14));
    else
      __builtin_amdgcn_s_waitcnt(0x0F70);
  };
  // A tile that reaches past the last key, or holds a block id outside the
  // pool, has V entries that are not this sequence's data (any bits, NaN
  // included).  Zero them in LDS once, after the tile has landed, so P·V
  // needs no per-step masking (their P is 0 and 0 * 0 = 0).  Uniform over
  // the workgroup; ends with a barrier when it writes.  Returns whether the
  // tile needs key masking.
  auto zero_stale = [&](int kt, int buf, int valid) -> bool {
    const bool special = kt * KT + KT > key_end || valid != (1 << (KT / kBlock)) - 1;
    if (!special) return false;
    // one 32-byte dim row (16 keys of a block) per thread, in 16-byte halves
    for (int e = threadIdx.x; e < KT / kBlock * D; e += 64 * W) {
      const int b = e / D, d = e % D;
      const int lim = (valid >> b) & 1 ? key_end - kt * KT - b * kBlock : 0;  // keys to keep
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int n = lim - 8 * h;
        if (n >= 8) continue;
        uint4* half = reinterpret_cast<uint4*>(&smem[1][buf][e * 32 + (h ^ vswz(d)) * 16]);
        uint4 v = uint4{0, 0, 0, 0};
        if (n > 0) {
          v = *half;
          uint32_t* w = &v.x;
#pragma unroll
          for (int i = 0; i < 4; ++i)
            w[i] = n >= 2 * i + 2 ? w[i] : n == 2 * i + 1 ? w[i] & 0xFFFFu : 0u;
        }
        *half = v;
      }
    }
    __syncthreads();
    return true;
  };
  // FP8: converts the tile staged in slot `slot` (copy layout: K row r's
  // 8-byte unit u at unit position u ^ fsw(r), V dim rows of 16 bytes) into
  // bf16 compute buffer `buf` (the bf16 layouts and swizzles above), exactly
  // (every E4M3 value is a bf16 value).  All threads of the workgroup.
  // Tile t is staged in slot t % 2 (issue_tile's `buf` is the slot for FP8)
  // and converted one tile boundary before its first use.
  // A wavefront whose units hold a code the hardware conversion reads
  // differently from the reference (NaN / inf / off-OCP codes; never
  // produced from finite input) converts them with the exact integer
  // decode.  Each thread's units are read first, so their LDS reads are in
  // flight together.
  auto convert_tile = [&](int buf, int slot) {
    if constexpr (FP8) {
      constexpr int UPT = KT * D / 8 / (64 * W);  // 8-byte units per thread, K and V each
      static_assert(UPT * 64 * W == KT * D / 8, "tile units per thread");
      uint2 kw[UPT], vw[UPT];
      uint32_t ex = 0;
#pragma unroll
      for (int i = 0; i < UPT; ++i) {
        const int e = threadIdx.x + i * 64 * W;
        const int r = e / (D / 8), u = e % (D / 8);
        kw[i] = *reinterpret_cast<const uint2*>(&stage[slot][0][r * D + (u ^ fsw(r)) * 8]);
        vw[i] = *reinterpret_cast<const uint2*>(&stage[slot][1][e * 8]);  // V dim rows
      }
#pragma unroll
      for (int i = 0; i < UPT; ++i)
        ex |= fp8_exotic_bits(kw[i].x) | fp8_exotic_bits(kw[i].y) | fp8_exotic_bits(vw[i].x) |
              fp8_exotic_bits(vw[i].y);
      auto store = [&](auto exact_c) {
#pragma unroll
        for (int i = 0; i < UPT; ++i) {
          const int e = threadIdx.x + i * 64 * W;
          const int r = e / (D / 8), u = e % (D / 8);
          const int bd = e / 2, h = e % 2;  // V: bd = block * D + dim
          const int d = bd % D;
          *reinterpret_cast<bf16x8*>(&smem[0][buf][r * (D * 2) + (u ^ kswz(r)) * 16]) =
              decltype(exact_c)::value ? fp8x8_to_bf16_exact(kw[i].x, kw[i].y)
                                       : fp8x8_to_bf16(kw[i].x, kw[i].y);
          *reinterpret_cast<bf16x8*>(&smem[1][buf][bd * 32 + (h ^ vswz(d)) * 16]) =
              decltype(exact_c)::value ? fp8x8_to_bf16_exact(vw[i].x, vw[i].y)
                                       : fp8x8_to_bf16(vw[i].x, vw[i].y);
        }
      };
      if (__builtin_amdgcn_ballot_w64((ex & 0x80808080u) != 0))
        store(std::true_type{});
      else
        store(std::false_type{});
    }
  };
  // Sᵀ for the 32 keys of step ST of the tile in buffer `buf`.  MFMA tile
  // kk's row i holds key 8 (i / 4) + 4 kk + i % 4 of the step, so the lane
  // (c, j) that receives rows 4j .. 4j+3 of both tiles holds keys
  // 8j .. 8j+7: eight consecutive keys of block j / 2.
  auto qk_load = [&](int buf, int ST, bf16x8 (&ka)[2][KS]) __attribute__((always_inline)) {
    const uint8_t* ks = &smem[0][buf][0];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int r = ST * 32 + 8 * (c >> 2) + 4 * kk + (c & 3);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int ch = (4 * s + j) ^ kswz(r);
        ka[kk][s] = *reinterpret_cast<const bf16x8*>(ks + r * (D * 2) + ch * 16);
      }
    }
  };
  auto qk_mfma = [&](const bf16x8 (&ka)[2][KS], f32x4 (&S)[NT][2]) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      S[nt][0] = f32x4{0.f, 0.f, 0.f, 0.f};
      S[nt][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        S[nt][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[0][s], qv[nt][s], S[nt][0], 0, 0, 0);
        S[nt][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[1][s], qv[nt][s], S[nt][1], 0, 0, 0);
      }
    }
  };

  bool tile_special;        // current tile needs key masking
  int valid_cur;            // validity bits of the current tile's 4 blocks
  int32_t id_ahead = 0;     // this wavefront's block id of the tile AHEAD of this one
  // Prologue: tiles 0 and 1 in flight, wait for tile 0.  (FP8: tiles 0 and
  // 1 staged and converted, then tile 2 copied into slot 0.)
  issue_tile(fetch_id(0), 0);
  if (n_kt > 1) issue_tile(fetch_id(1), 1);
  if constexpr (AHEAD == 3 && !FP8)
    if (n_kt > 2) issue_tile(fetch_id(2), 2);
  f32x4 o[NT][DT];
  f32x4 lacc[NT];  // softmax denominators, accumulated on the matrix core
  float nm[NT];  // minus the rows' running maxima (the Sᵀ accumulators start at it)
  float raise = 8.0f;  // a score this far above its row's max raises the max
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const bool ok = rows_active && r0 + 16 * nt + c < qlen;
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int i = 0; i < 8; ++i)
        qv[nt][s][i] = (__bf16)(ok ? (float)qv[nt][s][i] * scale_log2 : 0.f);
    nm[nt] = 0.f;
    lacc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[nt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  bad_ids = __syncthreads_or(bad) != 0;
  if constexpr (FP8) {
    wait_tiles(0);
    __syncthreads();
    convert_tile(0, 0);
    if (n_kt > 1) convert_tile(1, 1);
    __syncthreads();
    if (n_kt > 2) issue_tile(fetch_id(2), 0);
  } else {
    wait_tiles(min(n_kt, AHEAD) - 1);
  }
  __syncthreads();
  valid_cur = tile_valid(0);
  tile_special = zero_stale(0, 0, valid_cur);

  bf16x8 ones;  // all-ones MFMA operand for the row sums
#pragma unroll
  for (int i = 0; i < 8; ++i) ones[i] = (__bf16)1.0f;
  f32x4 S0[NT][2], S1[NT][2];
  {
    bf16x8 ka[2][KS];
    qk_load(0, kgrp, ka);
    qk_mfma(ka, S0);
  }

  // One 32-key step (step ST of tile kt, held in LDS buffer `buf`):
  // softmax of S (already computed), then in one basic block the P·V
  // products of this step and the Sᵀ products of the next.
  auto step = [&](int buf, auto stc, int kt, f32x4 (&S)[NT][2], f32x4 (&Snext)[NT][2]) {
    // KG = 1: step STC of the tile; KG = 2: this group's one step of it, which
    // begins with the tile boundary as the second step does
    constexpr int STC = KG == 2 ? 1 : decltype(stc)::value;
    const int ST = KG == 2 ? kgrp : STC;
    const int next = buf == NBUF - 1 ? 0 : buf + 1;
    // the buffer of the tile before this one, free again at the boundary
    const int free_buf = buf == 0 ? NBUF - 1 : buf - 1;
    // This step's Vᵀ fragments (dims 16 dt + c, keys 8j .. 8j+7 = one
    // 16-byte half of the 32-byte row of block 2 ST + j / 2), read first so
    // the softmax covers their latency.
    bf16x8 va[DT];
    {
      const uint8_t* vrow = &smem[1][buf][0] + (2 * ST + (j >> 1)) * (D * 32) + c * 32;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const int d = 16 * dt + c;
        va[dt] = *reinterpret_cast<const bf16x8*>(vrow + dt * 16 * 32 + (((j & 1) ^ vswz(d)) * 16));
      }
    }
    // K fragments of the next step, read now so the softmax prep below
    // covers their LDS latency.
    bf16x8 ka[2][KS];
    if constexpr (KG == 2) {
      if (kt + AHEAD < n_kt) id_ahead = fetch_id(kt + AHEAD);
    }
    if constexpr (STC == 0) {
      qk_load(buf, 1, ka);
      // this wavefront's block of the tile two ahead, a step before its copy
      if (kt + AHEAD < n_kt) id_ahead = fetch_id(kt + AHEAD);
    } else {
      // Tile boundary, at the start of a tile's second step: the next tile
      // has landed (all waves), the previous tile's buffer is free again
      // (every wavefront has finished the tile before this one), and the
      // next tile's first K fragments are read now so this step's softmax
      // covers them.  Past the last tile they are read from a buffer of
      // stale data and the products are never used.
      if (kt + 1 < n_kt) {
        // tile kt + 1 has landed; with four buffers kt + 2 may be in flight
        wait_tiles(NBUF == 4 && kt + 2 < n_kt ? 1 : 0);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if constexpr (FP8) {
          // FP8: tile kt + 2 (staged since the last boundary) into the free
          // compute buffer, visible to all at the next boundary's barrier;
          // its staging slot's previous tile (kt + 1) was converted a tile
          // ago, so tile kt + 3 is copied into it
          if (kt + 2 < n_kt) convert_tile(free_buf, (kt + 2) & 1);
          if (kt + 3 < n_kt) issue_tile(id_ahead, (kt + 3) & 1);
        } else {
          if (kt + AHEAD < n_kt) issue_tile(id_ahead, free_buf);
        }
      }
      qk_load(next, kgrp, ka);
    }
    {
      const int kb = (2 * kt + ST) * 32;  // first key of this step; x[i] <-> key kb + 8j + i
      if (tile_special || kb + 31 > past + r0) {
        // keys past the end, in invalid blocks, or above a row's diagonal
        const int blk_lim = ((valid_cur >> (2 * ST + (j >> 1))) & 1) ? key_end : 0;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const int row_pos = past + r0 + 16 * nt + c;
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const int key = kb + 8 * j + i;
            if (key >= blk_lim || key > row_pos) S[nt][i >> 2][i & 3] = -INFINITY;
          }
        }
      }
      // S holds log2-domain scores already offset by the row's running
      // max m (the Sᵀ accumulators start at -m).
      float lm[NT];
      bool need = false;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const float t0 = max3_raw(S[nt][0][0], S[nt][0][1], S[nt][0][2]);
        const float t1 = max3_raw(S[nt][0][3], S[nt][1][0], S[nt][1][1]);
        lm[nt] = max3_raw(t0, t1, max3_raw(S[nt][1][2], S[nt][1][3], S[nt][1][3]));
        need |= lm[nt] > raise;
      }
      // Rows keep a stale max until one of their scores exceeds it by 2^8;
      // only then is the exact max formed across the four lanes of the row
      // and the accumulator rescaled.  A row's first step with keys always
      // sets the max (m starts at 0, which says nothing about the row's
      // scores): step 0 or, where ids outside the pool masked all of the row's
      // keys so far, the first with any score (the row's denominator is still
      // 0 there, and at least 1 from then on).
      const bool first = (KG == 2 || STC == 0) && kt == 0;
      if (__builtin_expect(first || __builtin_amdgcn_ballot_w64(need) != 0, 0)) {
        raise = 8.0f;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          float bm = lm[nt];
          bm = fmaxf(bm, shfl_xor_f(bm, 16));
          bm = fmaxf(bm, shfl_xor_f(bm, 32));
          const bool none = first || lacc[nt][0] == 0.f;
          const bool masked = !(bm > -INFINITY);
          if (none && masked) raise = -INFINITY;
          const float delta = none ? (masked ? 0.f : bm) : fmaxf(bm, 0.f);
          nm[nt] -= delta;
#pragma unroll
          for (int i = 0; i < 8; ++i) S[nt][i >> 2][i & 3] -= delta;
          if (!first) {
            const float a = none ? 1.f : fast_exp2(-delta);
            lacc[nt] *= a;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) o[nt][dt] *= a;
          }
        }
      }
    }

    {
      // The next step's Sᵀ is computed even past this wavefront's last
      // step (it is then unused): keeping it unconditional keeps this one
      // basic block.  Its MFMAs are interleaved by hand with this step's
      // exponentials, one MFMA then EPM exponentials, so the matrix core
      // and the VALU of this wavefront work at the same time.  Consecutive
      // MFMAs go to independent accumulators (s outer, (nt, kk) inner).
      constexpr int NQK = 2 * KS * NT;  // next-step Sᵀ MFMAs
      constexpr int NEXP = 8 * NT;      // exponentials per lane
      constexpr int EPM = NEXP / NQK > 0 ? NEXP / NQK : 1;
      float pv[NT][8];
#pragma unroll
      for (int g = 0; g < NQK; ++g) {
        const int s_ = g / (2 * NT), q_ = g % (2 * NT), nt_ = q_ / 2, kk = q_ % 2;
        Snext[nt_][kk] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            ka[kk][s_], qv[nt_][s_], s_ == 0 ? f32x4{nm[nt_], nm[nt_], nm[nt_], nm[nt_]}
                                             : Snext[nt_][kk],
            0, 0, 0);
#pragma unroll
        for (int e = 0; e < EPM; ++e) {
          const int x = g * EPM + e;
          if (x < NEXP) {
            const int nt = x / 8, i = x % 8;
            pv[nt][i] = fast_exp2(S[nt][i >> 2][i & 3]);
          }
        }
      }
#pragma unroll
      for (int x = NQK * EPM; x < NEXP; ++x) {
        const int nt = x / 8, i = x % 8;
        pv[nt][i] = fast_exp2(S[nt][i >> 2][i & 3]);
      }
      // The interleave is imposed on the machine scheduler (compiler passes
      // before it may reorder the exponentials freely): groups of one MFMA
      // then EPM transcendental instructions, in this order.
#pragma unroll
      for (int g = 0; g < NQK; ++g) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);    // MFMA
        __builtin_amdgcn_sched_group_barrier(0x400, EPM, 0);  // transcendental
      }
      bf16x8 pb[NT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i = 0; i < 8; ++i) pb[nt][i] = (__bf16)pv[nt][i];
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          o[nt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[dt], pb[nt], o[nt][dt], 0, 0, 0);
      // Row sums of P: an all-ones operand makes every output row the sum
      // over the 32 keys, from the same bf16 P the numerator uses.
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        lacc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb[nt], lacc[nt], 0, 0, 0);
    }
    if constexpr (STC == 1) {
      if (kt + 1 < n_kt) {
        valid_cur = tile_valid(kt + 1);
        tile_special = zero_stale(kt + 1, next, valid_cur);
      }
    }
  };

  // Tile kt sits in LDS buffer kt % NBUF.  (Unrolling this loop over the
  // buffers, which would make every LDS address an immediate offset, costs
  // register spills.)
  for (int kt = 0, buf = 0; kt < n_kt; ++kt, buf = buf == NBUF - 1 ? 0 : buf + 1) {
    if constexpr (KG == 2) {
      step(buf, IC<1>{}, kt, S0, S1);
      if (++kt == n_kt) break;
      buf = buf == NBUF - 1 ? 0 : buf + 1;
      step(buf, IC<1>{}, kt, S1, S0);
    } else {
      step(buf, IC<0>{}, kt, S0, S1);
      step(buf, IC<1>{}, kt, S1, S0);
    }
  }

  if constexpr (KG == 2) {
    // The two groups' results meet in LDS (the tiles' space): log-sum-exp
    // merge by the first group's wavefronts.  A group that saw no key of a
    // row (l = 0) drops out.
    static_assert(W / 2 * NT * (DT * 1024 + 512) <= 2 * NBUF * CT_BYTES, "merge space");
    float* mo = reinterpret_cast<float*>(&smem[0][0][0]);
    float* mml = mo + W / 2 * NT * DT * 256;
    __syncthreads();
    if (kgrp == 1) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          *reinterpret_cast<f32x4*>(mo + ((wt * NT + nt) * DT + dt) * 256 + lane * 4) = o[nt][dt];
        *reinterpret_cast<float2*>(mml + ((wt * NT + nt) * 64 + lane) * 2) =
            float2{-nm[nt], lacc[nt][0]};
      }
    }
    __syncthreads();
    if (kgrp == 1) return;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const float2 ml = *reinterpret_cast<const float2*>(mml + ((wt * NT + nt) * 64 + lane) * 2);
      const float ma = lacc[nt][0] != 0.f ? -nm[nt] : kNegBig;
      const float mb = ml.y != 0.f ? ml.x : kNegBig;
      const float mx = fmaxf(ma, mb);
      const float fa = fast_exp2(ma - mx), fb = fast_exp2(mb - mx);
      lacc[nt] = lacc[nt] * fa + ml.y * fb;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        o[nt][dt] = o[nt][dt] * fa +
                    *reinterpret_cast<const f32x4*>(mo + ((wt * NT + nt) * DT + dt) * 256 + lane * 4) * fb;
    }
  }

  if (!rows_active) return;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const float l = lacc[nt][0];
    const int row = r0 + 16 * nt + c;
    if (row >= qlen) continue;
    const float inv = l != 0.f ? 1.f / l : 0.f;
    uint16_t* orow = out + ((int64_t)(q_begin + row) * Hq + head) * D + 4 * j;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      uint16_t w[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) w[r] = __builtin_bit_cast(uint16_t, (__bf16)(o[nt][dt][r] * inv));
      *reinterpret_cast<uint64_t*>(orow + 16 * dt) = *reinterpret_cast<const uint64_t*>(w);
    }
  }
  };
  for (int r = 0; r * nslot < items; ++r) {
    const int item = r * nslot + ((r & 1) ? nslot - 1 - slot : slot);
    if (item < items) process(item);
  }
}

// f32 caches (plain, or int8-in-f32 with one scale per block), D in {16, 32,
// 64, 128, 256}, on v_mfma_f32_16x16x4_f32 (full f32 products and sums).
//
// Workgroup = 8 wavefronts on 16 query tokens: min(G, 4) heads of one kv head
// x 8 / that many key splits; a wavefront takes every KS-th step (NB blocks of
// 16 keys) for the 16 tokens of its head, and the splits' results meet in LDS.
// Operand lane layout (lane = 16 j + c; the MFMA contracts over j):
//   Sᵀ = K·Qᵀ: a lane loads 4 consecutive dims 16 t + 4 j .. of key row c and
//     query row c (16 bytes each) and feeds them to 4 MFMAs -> the lane holds
//     Sᵀ[key 4 j + r][query c];
//   Oᵀ = Vᵀ·Pᵀ: a lane loads keys 4 j .. 4 j + 3 of dim 16 dt + c (16 bytes of
//     the token-minor block), whose P it already holds.
// K and V go straight from the cache to operand registers; the heads of a
// workgroup read the same blocks at the same time through the L1.
// Bound: the f32 matrix rate (157 TFLOP/s) where there are enough tokens, else
// the serial steps of the longest row tile, which the key splits shorten.
// 511, 129, 300 and 64 tokens on 0, 256, 0 and 33, 14 / 2 heads x 64:
// 492 us a call with one wavefront per (row, head) on the VALU, 27.7 here.
template <int D>
__global__ __launch_bounds__(512) void prefill_f32_kernel(
    float* __restrict__ out, const float* __restrict__ q, const float* __restrict__ kc,
    const float* __restrict__ vc, const int32_t* __restrict__ block_tables, int mbs,
    const int32_t* __restrict__ cu_q, const int32_t* __restrict__ past_lens, int Hq, int Hkv, int G,
    int num_blocks, float scale_log2, const float* __restrict__ kv_scales, int64_t q_row,
    int total_q, int max_q) {
  constexpr int NB = D <= 64 ? 2 : 1;  // cache blocks per step
  constexpr int DT = D / 16;
  __shared__ __attribute__((aligned(16))) float mo[8][DT][64][4];
  __shared__ float mml[8][64][2];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, j = lane >> 4;
  const int seq = blockIdx.z, head_groups = (G + 3) / 4;
  const QRange qr = q_range(cu_q, past_lens, seq, total_q, max_q);
  const int tok0 = 16 * (int)(gridDim.x - 1 - blockIdx.x);  // the longest tiles first
  if (tok0 >= qr.len) return;
  const int HW = min(G, 4), KS = HW == 1 ? 8 : HW == 2 ? 4 : 2;
  const int ks = wave / HW, hl = wave - ks * HW;
  const int kvh = blockIdx.y / head_groups, hig = (blockIdx.y - kvh * head_groups) * 4 + hl;
  const bool active = ks < KS && hig < G;  // HW = 3 leaves two wavefronts, G % 4 heads over
  const int head = kvh * G + min(hig, G - 1);
  const int row_pos = qr.past + tok0 + c;  // this lane's query row
  const int key_end = min(qr.past + min(qr.len, tok0 + 16), mbs * kBlock);
  const int nblk = active ? (key_end + kBlock - 1) / kBlock : 0;

  float4 qv[DT];
  const float* qp = q + (int64_t)(qr.begin + min(tok0 + c, qr.len - 1)) * q_row +
                    (int64_t)head * D + 4 * j;
#pragma unroll
  for (int t = 0; t < DT; ++t) qv[t] = *reinterpret_cast<const float4*>(qp + 16 * t);
  f32x4 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = kNegBig, l = 0.f;
  const int32_t* btab = block_tables + (int64_t)seq * mbs;
  const int64_t head_stride = (int64_t)kBlock * D;

  for (int ib = NB * ks; ib < nblk; ib += NB * KS) {
    const float* vb[NB];
    int lim[NB];  // keys of the block that count
    float bscale[NB];
    float4 kx[NB][DT], vx[NB][DT];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      int32_t id = btab[min(ib + b, nblk - 1)];
      lim[b] = min(max(key_end - (ib + b) * kBlock, 0), kBlock);
      if (id < 0 || id >= num_blocks) {
        id = 0;
        lim[b] = 0;
      }
      const int64_t off = ((int64_t)id * Hkv + kvh) * head_stride;
      vb[b] = vc + off;
      const float* kp = kc + off + c * D + 4 * j;
#pragma unroll
      for (int t = 0; t < DT; ++t) kx[b][t] = *reinterpret_cast<const float4*>(kp + 16 * t);
      bscale[b] = kv_scales ? kv_scales[id] : 1.0f;
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        vx[b][dt] = *reinterpret_cast<const float4*>(vb[b] + (16 * dt + c) * kBlock + 4 * j);
    f32x4 S[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) S[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        S[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kx[b][t].x, qv[t].x, S[b], 0, 0, 0);
        S[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kx[b][t].y, qv[t].y, S[b], 0, 0, 0);
        S[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kx[b][t].z, qv[t].z, S[b], 0, 0, 0);
        S[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kx[b][t].w, qv[t].w, S[b], 0, 0, 0);
      }
    // keys past the end, in invalid blocks or above a row's diagonal
    const bool diag = (ib + NB) * kBlock - 1 > qr.past + tok0;  // wavefront-uniform
    bool partial = false;
    float x[NB][4], bm = -INFINITY;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      partial |= lim[b] < kBlock;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        x[b][r] = S[b][r] * (bscale[b] * scale_log2);
        const int t = 4 * j + r;
        if (t >= lim[b] || (ib + b) * kBlock + t > row_pos) x[b][r] = -INFINITY;
        bm = fmaxf(bm, x[b][r]);
      }
    }
    // the max is kept until a score exceeds it by 2^8 (see decode)
    if (__builtin_amdgcn_ballot_w64(bm > m + 8.0f)) {
      bm = fmaxf(bm, shfl_xor_f(bm, 16));
      bm = fmaxf(bm, shfl_xor_f(bm, 32));
      const float mn = fmaxf(m, bm);
      const float a = exp2f(m - mn);
      m = mn;
      l *= a;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[dt] *= a;
    }
    float p[NB][4];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        p[b][r] = exp2f(x[b][r] - m);
        l += p[b][r];
        p[b][r] *= bscale[b];
      }
    float odd_scale = 0.f;
    if (kv_scales)
#pragma unroll
      for (int b = 0; b < NB; ++b) odd_scale += bscale[b] - bscale[b];
    if (odd_scale != 0.f) {
      // A masked key's probability stays 0 also where its block's scale is not
      // finite (0 * inf would reach the rows below the block).
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int t = 4 * j + r;
          if (t >= lim[b] || (ib + b) * kBlock + t > row_pos) p[b][r] = 0.f;
        }
    }
    if (partial) {
      // cache contents past the context may be any bits
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          const int n = lim[b] - 4 * j;
          vx[b][dt] = float4{n > 0 ? vx[b][dt].x : 0.f, n > 1 ? vx[b][dt].y : 0.f,
                             n > 2 ? vx[b][dt].z : 0.f, n > 3 ? vx[b][dt].w : 0.f};
        }
    }
    if (diag) {
      // A value that is not finite above a row's diagonal must not reach it
      // through 0 * v: such a step goes key by key.
      float odd = 0.f;
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          odd += (vx[b][dt].x - vx[b][dt].x) + (vx[b][dt].y - vx[b][dt].y) +
                 (vx[b][dt].z - vx[b][dt].z) + (vx[b][dt].w - vx[b][dt].w);
      if (__builtin_amdgcn_ballot_w64(odd != 0.f)) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            for (int jj = 0; jj < 4; ++jj) {
              const float pk = __shfl(p[b][r], 16 * jj + c, 64);
              const int t = 4 * jj + r;
              if (t >= lim[b] || (ib + b) * kBlock + t > row_pos) continue;
#pragma unroll
              for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                  o[dt][e] += pk * vb[b][(16 * dt + 4 * j + e) * kBlock + t];
            }
        continue;
      }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(vx[b][dt].x, p[b][0], o[dt], 0, 0, 0);
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(vx[b][dt].y, p[b][1], o[dt], 0, 0, 0);
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(vx[b][dt].z, p[b][2], o[dt], 0, 0, 0);
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(vx[b][dt].w, p[b][3], o[dt], 0, 0, 0);
      }
  }
  l += shfl_xor_f(l, 16);
  l += shfl_xor_f(l, 32);
  // the key splits' results: log-sum-exp merge by the first split's wavefront
  // of each head (a split that saw no key of a row has m = kNegBig, l = 0, o = 0)
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<f32x4*>(&mo[wave][dt][lane][0]) = o[dt];
  mml[wave][lane][0] = m;
  mml[wave][lane][1] = l;
  __syncthreads();
  if (ks != 0 || !active || tok0 + c >= qr.len) return;
  float mx = m;
  for (int z = 1; z < KS; ++z) mx = fmaxf(mx, mml[z * HW + hl][lane][0]);
  const float f0 = exp2f(m - mx);
  l *= f0;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] *= f0;
  for (int z = 1; z < KS; ++z) {
    const float f = exp2f(mml[z * HW + hl][lane][0] - mx);
    l += mml[z * HW + hl][lane][1] * f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      o[dt] += *reinterpret_cast<const f32x4*>(&mo[z * HW + hl][dt][lane][0]) * f;
  }
  const float inv = l != 0.f ? 1.f / l : 0.f;
  float* orow = out + ((int64_t)(qr.begin + tok0 + c) * Hq + head) * D + 4 * j;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
    *reinterpret_cast<f32x4*>(orow + 16 * dt) = o[dt] * inv;
}

// Generic: one wavefront per (query row, head); keys in chunks of 64 with
// an online softmax; lane d accumulates output dims d, d + 64, ...
template <typename T, typename TC = T>
__global__ __launch_bounds__(64) void prefill_generic_kernel(
    T* __restrict__ out, const T* __restrict__ q, const TC* __restrict__ kc,
    const TC* __restrict__ vc, const int32_t* __restrict__ block_tables, int mbs,
    const int32_t* __restrict__ cu_q, const int32_t* __restrict__ past_lens, int Hq, int Hkv,
    int D, int num_blocks, float scale_log2, const float* __restrict__ kv_scales, int64_t q_row,
    int total_q, int max_q) {
  // kv_scales: per-block scales of a quantised (int8-in-f32) cache, or null
  __shared__ float qs[512];
  __shared__ float ps[64];
  __shared__ int32_t bids[64];
  const int row = blockIdx.x, h = blockIdx.y, seq = blockIdx.z, lane = threadIdx.x;
  const QRange qr = q_range(cu_q, past_lens, seq, total_q, max_q);
  const int q_begin = qr.begin;
  if (row >= qr.len) return;
  const int G = Hq / Hkv, kvh = h / G;
  const int pos = qr.past + row;
  const int64_t qoff = (int64_t)(q_begin + row) * q_row + (int64_t)h * D;
  for (int d = lane; d < D; d += 64) qs[d] = Elem<T>::load(q + qoff + d);
  float acc[8];
  for (int i = 0; i < 8; ++i) acc[i] = 0.f;
  float m = kNegBig, l = 0.f;
  for (int k0 = 0; k0 <= pos; k0 += 64) {
    __syncthreads();
    if (lane < 4) {
      const int bi = k0 / kBlock + lane;
      int32_t b = (bi < mbs) ? block_tables[(int64_t)seq * mbs + bi] : -1;
      bids[lane] = (b >= 0 && b < num_blocks) ? b : -1;
    }
    __syncthreads();
    const int key = k0 + lane;
    float s = -INFINITY;
    const int32_t b = bids[lane / kBlock];
    if (key <= pos && b >= 0) {
      const TC* kr = kc + (((int64_t)b * Hkv + kvh) * kBlock + key % kBlock) * D;
      const float ks = kv_scales ? kv_scales[b] : 1.0f;
      float a = 0.f;
      for (int d = 0; d < D; ++d) a += qs[d] * (Elem<TC>::load(kr + d) * ks);
      s = a * scale_log2;
    }
    float bm = s;
    for (int w = 32; w > 0; w >>= 1) bm = fmaxf(bm, __shfl_xor(bm, w, 64));
    const float mn = fmaxf(m, bm);
    const float alpha = exp2f(m - mn);
    m = mn;
    const float p = exp2f(s - m);
    float ls = p;
    for (int w = 32; w > 0; w >>= 1) ls += __shfl_xor(ls, w, 64);
    l = l * alpha + ls;
    ps[lane] = p;
    __syncthreads();
    const int nk = min(64, pos + 1 - k0);
    for (int i = 0; i * 64 + lane < D; ++i) {
      const int d = i * 64 + lane;
      float a = acc[i] * alpha;
      for (int t = 0; t < nk; ++t) {
        const int32_t bt = bids[t / kBlock];
        if (bt < 0) continue;
        const float vs = kv_scales ? kv_scales[bt] : 1.0f;
        a += ps[t] * (Elem<TC>::load(vc + (((int64_t)bt * Hkv + kvh) * D + d) * kBlock +
                                     (k0 + t) % kBlock) *
                      vs);
      }
      acc[i] = a;
    }
  }
  const float inv = l != 0.f ? 1.f / l : 0.f;
  for (int i = 0; i * 64 + lane < D; ++i)
    Elem<T>::store(out + ((int64_t)(q_begin + row) * Hq + h) * D + i * 64 + lane, acc[i] * inv);
}

}  // namespace
}  // namespace pa

using namespace pa;



namespace {
// Compute units of the current device (cached per device).
int compute_units() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cached[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        n <= 0)
      n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}

int32_t prefill_impl(void* out, const void* q, const void* k_cache, const void* v_cache,
                     const float* kv_scales, const int32_t* block_tables,
                     int32_t max_blocks_per_seq, const int32_t* cu_q_lens,
                     const int32_t* past_lens, int32_t num_seqs, int32_t total_q,
                     int32_t max_q_len, int32_t num_heads, int32_t num_kv_heads,
                     int32_t head_dim, int32_t num_blocks, float scale, int32_t dtype,
                     pa_stream_t stream, int64_t q_row = 0) {
  clear_error();
  PA_REQUIRE(dtype_ok(dtype) || dtype == PA_DTYPE_FP8_E4M3, PA_ERR_INVALID_ARG,
             "pa_prefill: unknown dtype %d", dtype);
  PA_REQUIRE(num_seqs >= 0 && total_q >= 0 && max_q_len >= 0 && num_heads > 0 &&
                 num_kv_heads > 0 && head_dim > 0 && num_blocks > 0 && max_blocks_per_seq > 0,
             PA_ERR_INVALID_ARG, "pa_prefill: bad sizes");
  PA_REQUIRE(num_heads % num_kv_heads == 0, PA_ERR_INVALID_ARG,
             "pa_prefill: num_heads %d not a multiple of num_kv_heads %d", num_heads,
             num_kv_heads);
  PA_REQUIRE(head_dim <= 512, PA_ERR_UNSUPPORTED, "pa_prefill: head_dim %d > 512", head_dim);
  if (num_seqs == 0 || total_q == 0 || max_q_len == 0) return PA_OK;
  PA_REQUIRE(out && q && k_cache && v_cache && block_tables && cu_q_lens && past_lens,
             PA_ERR_INVALID_ARG, "pa_prefill: null pointer");
  if (q_row == 0) q_row = (int64_t)num_heads * head_dim;
  PA_REQUIRE(q_row >= (int64_t)num_heads * head_dim, PA_ERR_INVALID_ARG,
             "pa_prefill: q row stride %lld below num_heads * head_dim", (long long)q_row);
  const float scale_log2 = scale * kLog2e;
  hipStream_t s = (hipStream_t)stream;
  const bool fp8 = dtype == PA_DTYPE_FP8_E4M3;
  const bool tiled = !kv_scales && (dtype == PA_DTYPE_BF16 || fp8) &&
                     (head_dim == 64 || head_dim == 128);
  const bool mfma = !kv_scales && dtype == PA_DTYPE_BF16 && head_dim == 256;
  // 16-byte operand loads: rows of q and cache rows from 16-byte aligned
  // bases (a strided view of q may start anywhere), and a grid within limits
  const bool f32_mfma = dtype == PA_DTYPE_F32 && head_dim >= 16 && 256 % head_dim == 0 &&
                        ((uintptr_t)q | (uintptr_t)out | (uintptr_t)k_cache |
                         (uintptr_t)v_cache) % 16 == 0 &&
                        q_row % 4 == 0 && num_seqs <= 65535 &&
                        (long long)num_kv_heads * ((num_heads / num_kv_heads + 3) / 4) <= 65535;
  if (tiled) {
    const int G = num_heads / num_kv_heads;
    const int HW = G < 4 ? G : 4;
    const int head_groups = (G + 3) / 4;
    auto* o = (uint16_t*)out;
    auto* qq = (const uint16_t*)q;
    auto launch = [&](auto dc, auto ntc, auto wc, auto kgc, auto cache) -> int32_t {
      constexpr int DD = decltype(dc)::value, NT = decltype(ntc)::value, W = decltype(wc)::value;
      constexpr int KG = decltype(kgc)::value;
      using TC = decltype(cache);
      const int TT = 16 * NT * (W / KG / 4) * (4 / HW);
      const int tiles_per_seq = (max_q_len + TT - 1) / TT;
      const long long total = (long long)num_seqs * num_kv_heads * head_groups * tiles_per_seq;
      PA_REQUIRE(total < (1ll << 31) / 8, PA_ERR_UNSUPPORTED, "pa_prefill: launch too large");
      const int per_xcd = (int)((total + 7) / 8);
      // persistent grid: about one workgroup per CU (a multiple of the 8 XCDs)
      const dim3 grid(8 * std::max(1, std::min(per_xcd, compute_units() / 8)));
      prefill_tiled_kernel<DD, NT, W, KG, TC><<<grid, 64 * W, 0, s>>>(
          o, qq, (const TC*)k_cache, (const TC*)v_cache, block_tables, max_blocks_per_seq,
          cu_q_lens, past_lens, num_heads, num_kv_heads, G, num_blocks, scale_log2, num_seqs,
          tiles_per_seq, head_groups, q_row, total_q, max_q_len);
      return PA_OK;
    };
    // Query tokens per workgroup.  An item's time is its keys times the
    // workgroup's time per key tile (1 for 256 query rows, 0.7 for 128 rows
    // with two key groups, 0.53 for 64), and the items of a launch share the
    // CUs, their average about 0.65 of the longest; the lengths are on the
    // device, so the items are counted from the totals.  Measured, us (256 /
    // 128 / 64 rows): 512 tokens on 1024 cached, 32 / 8 heads x 128: 46 / 35
    // / 26; 701, 123 and 411 on 3001, 0 and 517: 98 / 71 / 87 (FP8 115 / 85 /
    // 119); 2 x 1024 on 0 and 1024: 61 / 54 / 71; 2048 on 2000 and 1000 on
    // 0: 115 / 136 / 181; 4 x 2048: 260 / 307 / 427; 14 / 2 heads x 64: 500,
    // 300, 222: 22 / 17 / 14, 2000, 1300, 1222: 45 / 55 / 75.
    auto cost = [&](int tokens, double per_tile) -> double {
      tokens *= HW == 1 ? 4 : HW == 2 ? 2 : 1;
      const double tiles =
          std::max((double)num_seqs, (double)total_q / tokens + 0.5 * num_seqs);
      return per_tile * std::max(1., 0.65 / 256 * tiles * num_kv_heads * head_groups);
    };
    const double c64 = cost(64, 1.), c32 = cost(32, 0.7), c16 = cost(16, 0.53);
    auto pick = [&](auto dc, auto cache) -> int32_t {
      if (c64 <= c32 && c64 <= c16) return launch(dc, IC<2>{}, IC<8>{}, IC<1>{}, cache);
      if (c32 <= c16) return launch(dc, IC<2>{}, IC<8>{}, IC<2>{}, cache);
      return launch(dc, IC<1>{}, IC<8>{}, IC<2>{}, cache);
    };
    const int32_t rc = fp8 ? (head_dim == 128 ? pick(IC<128>{}, uint8_t{}) : pick(IC<64>{}, uint8_t{}))
                           : (head_dim == 128 ? pick(IC<128>{}, uint16_t{})
                                              : pick(IC<64>{}, uint16_t{}));
    if (rc != PA_OK) return rc;
  } else if (mfma) {
    constexpr int NT = 2;
    const int rows_per_wg = 16 * NT * kWaves;
    const dim3 grid((max_q_len + rows_per_wg - 1) / rows_per_wg, num_heads, num_seqs);
    auto* o = (uint16_t*)out;
    auto* qq = (const uint16_t*)q;
    auto* kc = (const uint16_t*)k_cache;
    auto* vc = (const uint16_t*)v_cache;
#define PA_LAUNCH_PREFILL(DD)                                                                 \
  prefill_mfma_kernel<DD, NT><<<grid, 64 * kWaves, 0, s>>>(                                   \
      o, qq, kc, vc, block_tables, max_blocks_per_seq, cu_q_lens, past_lens, num_heads,       \
      num_kv_heads, num_blocks, scale_log2, q_row, total_q, max_q_len)
    PA_LAUNCH_PREFILL(256);
#undef PA_LAUNCH_PREFILL
  } else if (f32_mfma) {
    const int G = num_heads / num_kv_heads;
    const dim3 grid((max_q_len + 15) / 16, num_kv_heads * ((G + 3) / 4), num_seqs);
    auto launch = [&](auto dc) {
      prefill_f32_kernel<decltype(dc)::value><<<grid, 512, 0, s>>>(
          (float*)out, (const float*)q, (const float*)k_cache, (const float*)v_cache, block_tables,
          max_blocks_per_seq, cu_q_lens, past_lens, num_heads, num_kv_heads, G, num_blocks,
          scale_log2, kv_scales, q_row, total_q, max_q_len);
    };
    switch (head_dim) {
      case 16: launch(IC<16>{}); break;
      case 32: launch(IC<32>{}); break;
      case 64: launch(IC<64>{}); break;
      case 128: launch(IC<128>{}); break;
      default: launch(IC<256>{}); break;
    }
  } else {
    const dim3 grid(max_q_len, num_heads, num_seqs);
    if (dtype == PA_DTYPE_FP8_E4M3)
      prefill_generic_kernel<uint16_t, Fp8><<<grid, 64, 0, s>>>(
          (uint16_t*)out, (const uint16_t*)q, (const Fp8*)k_cache, (const Fp8*)v_cache,
          block_tables, max_blocks_per_seq, cu_q_lens, past_lens, num_heads, num_kv_heads,
          head_dim, num_blocks, scale_log2, nullptr, q_row, total_q, max_q_len);
    else if (dtype == PA_DTYPE_BF16)
      prefill_generic_kernel<uint16_t><<<grid, 64, 0, s>>>(
          (uint16_t*)out, (const uint16_t*)q, (const uint16_t*)k_cache, (const uint16_t*)v_cache,
          block_tables, max_blocks_per_seq, cu_q_lens, past_lens, num_heads, num_kv_heads,
          head_dim, num_blocks, scale_log2, nullptr, q_row, total_q, max_q_len);
    else
      prefill_generic_kernel<float><<<grid, 64, 0, s>>>(
          (float*)out, (const float*)q, (const float*)k_cache, (const float*)v_cache,
          block_tables, max_blocks_per_seq, cu_q_lens, past_lens, num_heads, num_kv_heads,
          head_dim, num_blocks, scale_log2, kv_scales, q_row, total_q, max_q_len);
  }
  return check_launch("pa_prefill");
}
}  // namespace

extern "C" int32_t pa_prefill(void* out, const void* q, const void* k_cache, const void* v_cache,
                              const int32_t* block_tables, int32_t max_blocks_per_seq,
                              const int32_t* cu_q_lens, const int32_t* past_lens,
                              int32_t num_seqs, int32_t total_q, int32_t max_q_len,
                              int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
                              int32_t num_blocks, float scale, int32_t dtype, pa_stream_t stream) {
  return prefill_impl(out, q, k_cache, v_cache, nullptr, block_tables, max_blocks_per_seq,
                      cu_q_lens, past_lens, num_seqs, total_q, max_q_len, num_heads, num_kv_heads,
                      head_dim, num_blocks, scale, dtype, stream);
}

extern "C" int32_t pa_prefill_quantized(void* out, const void* q, const float* k_cache,
                                        const float* v_cache, const float* block_scales,
                                        const int32_t* block_tables, int32_t max_blocks_per_seq,
                                        const int32_t* cu_q_lens, const int32_t* past_lens,
                                        int32_t num_seqs, int32_t total_q, int32_t max_q_len,
                                        int32_t num_heads, int32_t num_kv_heads,
                                        int32_t head_dim, int32_t num_blocks, float scale,
                                        pa_stream_t stream) {
  if (!block_scales) {
    clear_error();
    set_error("pa_prefill_quantized: null block_scales");
    return PA_ERR_INVALID_ARG;
  }
  return prefill_impl(out, q, k_cache, v_cache, block_scales, block_tables, max_blocks_per_seq,
                      cu_q_lens, past_lens, num_seqs, total_q, max_q_len, num_heads, num_kv_heads,
                      head_dim, num_blocks, scale, PA_DTYPE_F32, stream);
}

namespace pa {
int32_t prefill_strided(void* out, const void* q, int64_t q_row, const void* k_cache,
                        const void* v_cache, const int32_t* block_tables,
                        int32_t max_blocks_per_seq, const int32_t* cu_q_lens,
                        const int32_t* past_lens, int32_t num_seqs, int32_t total_q,
                        int32_t max_q_len, int32_t num_heads, int32_t num_kv_heads,
                        int32_t head_dim, int32_t num_blocks, float scale, int32_t dtype,
                        pa_stream_t stream) {
  return prefill_impl(out, q, k_cache, v_cache, nullptr, block_tables, max_blocks_per_seq,
                      cu_q_lens, past_lens, num_seqs, total_q, max_q_len, num_heads, num_kv_heads,
                      head_dim, num_blocks, scale, dtype, stream, q_row);
}
}  // namespace pa
