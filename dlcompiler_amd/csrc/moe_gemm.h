// Operands and small device helpers shared by the two grouped MoE GEMMs: the tiled one for many
// rows per expert (moe_fp8.hip, fp8) and the streaming one (moe_stream.hip).
#pragma once
#include <type_traits>

#include "common.h"
#include "moe_rules.h"

namespace dlb {

struct MoeGemmParams {
  const unsigned char* a;     // activations fp8 [rows, K] (or 16-bit: K = bytes per row)
  const float* a_scale;       // [rows, K / 128]
  const unsigned char* w;     // weights [E_local, N, K]
  const float* w_scale;       // [E_local, N / 128, K / 128]
  IdxArray sorted_ids;        // [num_mblocks * block_m] routing slots grouped by expert
  IdxArray counts;            // [num_experts] routed slots per (global) expert
  // launcher form of the routing (non-gated kernel only): the slot list is NOT padded per expert;
  // expert e owns its positions seg_start[e] .. counts[e] - 1 (counts then holds the segment ENDS)
  IdxArray seg_start;         // p == nullptr: block-aligned list
  int64_t a_rows;             // rows of `a` when it is read in sorted order (reads are clamped to it)
  int gather_a;               // non-gated kernel: rows of `a` are gathered by token (slot / topk)
  int scatter_c;              // non-gated kernel: output row = routing slot (else the sorted position)
  int num_experts;            // global expert count = length of counts
  int num_mblocks;            // capacity of sorted_ids in blocks
  int bm_shift;               // log2(block_m): 6 or 7
  int num_ntiles;
  int K, N, KC;               // K = bytes per activation / weight row, KC = K / 128
  int topk, numel;            // flat slots = tokens * topk (also the pad sentinel)
  int num_tokens;
  int expert_offset;          // weights hold experts [expert_offset, expert_offset + E_local)
  int num_local;              // E_local
  // gate_up flavour
  unsigned char* hq;          // [num_mblocks * block_m, I] fp8, or 16-bit when QT = 1
  float* hs;                  // [num_mblocks * block_m, I / 128]
  int I;
  // down flavour
  void* out;                  // [numel, N] bf16/f16
  const float* topk_w;        // [numel]
  int64_t lda;                // gated fp8, few rows: `a` is 16-bit, rows of lda bytes (0: quantised)
  uint32_t kc_rcp;            // 2^32 / KC, rounded down (KC > 1)
  uint32_t topk_rcp;          // 2^32 / topk, rounded down (topk 1: 2^32 - 1)
  // fp8, very few rows (see moe_hands_over_f32): the intermediate is [numel, I] fp32, by routing slot, which
  // gate_up leaves in h32 and the down GEMM, whose `a` it is, quantises as it loads it
  float* h32;
  int renorm;                 // weights are divided by the sum of their token's
  int summed;                 // the sum over the slots follows: fp8, many rows, `out` goes through the caches
};

// routing weight of a slot (1 without weights)
__device__ __forceinline__ float slot_weight(const MoeGemmParams& p, int slot) {
  if (!p.topk_w) return 1.0f;
  const float w = p.topk_w[slot];
  if (!p.renorm) return w;
  const uint32_t n = (uint32_t)slot, q = __umulhi(n, p.topk_rcp), token = n - q * p.topk >= (uint32_t)p.topk ? q + 1 : q;
  const float* mine = p.topk_w + token * (uint32_t)p.topk;
  float sum = 0.0f;
  // Four or eight weights on their way at once: one after the other is a chain of topk loads (fp8, us a layer: 64 experts of
  // 1024 x 512, 6000 tokens x 8, 196.9 -> 190.5; 32 of 2048 x 256, 2500 x 4, 77.0 -> 72.6).  Eight for two alone cost 1 %.
  auto add = [&](auto ahead) __attribute__((always_inline)) {
    constexpr int N = decltype(ahead)::value;
    for (int j0 = 0; j0 < p.topk; j0 += N) {
      float v[N];
#pragma unroll
      for (int j = 0; j < N; ++j) v[j] = mine[min(j0 + j, p.topk - 1)];
#pragma unroll
      for (int j = 0; j < N; ++j) sum += j0 + j < p.topk ? v[j] : 0.0f;
    }
  };
  if (p.topk <= 4) add(std::integral_constant<int, 4>{});
  else add(std::integral_constant<int, 8>{});
  return w / sum;
}

__device__ __forceinline__ i32x8 cat8(const u32x4& lo, const u32x4& hi) {
  return i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3],
               (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
}

// exchange between the two lane halves: afterwards lane half 0 holds (its a, the partner's a)
// and lane half 1 (the partner's b, its b), partner = the lane 32 away
__device__ __forceinline__ void swap_halves(unsigned int& a, unsigned int& b) {
  typedef __attribute__((ext_vector_type(2))) unsigned int u2;
  const u2 r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

// the tile of a workgroup
struct TileId {
  int e;     // local expert
  int row0;  // first position of the tile's rows in sorted_ids
  int nt;    // column tile
  int rows;  // real (unpadded) rows of the tile
};

// Do a layer's GEMMs hand the intermediate over in fp32 (fp8, up to kSmallMeanRows; see fp8_few_rows)?  up: of gate_up
bool moe_hands_over_f32(const MoeGemmParams& up);
// Launches the streaming kernel.  gated / quantised as the entry points; N_out checks are done.
int launch_moe_stream(const MoeGemmParams& p, bool gated, int quantised, int dtype, int w_layout, hipStream_t s);
// fp8: up to this many rows per expert, on average over the routed slots, the streaming kernel is the
// faster one (stream / tiled: 8 experts of 4096 x 4096, 22 rows 88.8 / 91.0 us, 36 rows 94.0 / 95.8; 64 of
// 2048 x 1408, 15 rows 110 / 112, 36 rows 119 / 116; 128 of 2048 x 768, 30 rows 134.7 / 135.6, 42 rows 147 / 140).
// 16-bit operands always take it.
constexpr int kStreamMeanRows = 32;
// While an expert mostly has one tile of up to 128 rows its weights are read once, and go past the caches: 64
// experts of 2048 x 1408, kept / not kept: 16 bit, 75 rows 234 / 210 us, 105 rows 254 / 224, 140 rows 316 / 387;
// fp8, 50 rows 125.7 / 119.7, 105 rows 145.2 / 140.9, 125 rows 176 / 187.  Not so weights that the 256 MB behind
// the L2s may still hold (fp8, 32 experts of 1024 x 512, 30 rows: 36.1 / 37.9).
inline bool weights_read_once(const MoeGemmParams& p) {
  return (int64_t)p.numel <= (int64_t)110 * p.num_experts && (int64_t)p.num_local * p.N * p.K > ((int64_t)128 << 20);
}

}  // namespace dlb
