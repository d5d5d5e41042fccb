// Router of one token on a DPP row (16 lanes): softmax over the experts, top-k by arg-max rounds.
// Shared by the stand-alone router and by the launches that also align the routing by expert.
#pragma once
#include "common.h"

namespace dlb {

// order-preserving map float -> uint32 (larger float <=> larger key); -0.0 < +0.0 there, so
// canonicalise zeros first to keep "equal logits -> lowest index".
__device__ __forceinline__ uint32_t orderable(float f) {
  f = (f == 0.0f) ? 0.0f : f;
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// inverse of orderable (zeros come back as +0)
__device__ __forceinline__ float from_orderable(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

template <int CTRL>
__device__ __forceinline__ uint32_t row_step_max(uint32_t v) {
  return max(v, dpp_u32<CTRL>(v));
}
__device__ __forceinline__ uint32_t row16_max_u32(uint32_t v) {
  v = row_step_max<kDppQuadXor1>(v);
  v = row_step_max<kDppQuadXor2>(v);
  v = row_step_max<kDppRowHalfMirror>(v);
  return row_step_max<kDppRowMirror>(v);
}

// The logits of one token, VPL consecutive experts per lane of its DPP row (-inf past E and for
// dead rows).  LT = element type of the logits (fp32, or bf16 / fp16 converted on the way in: the
// reference's fused gate kernel takes 16-bit logits and computes in fp32,
// python/dlBLAS/dlblas/kernels/topk_gating_fwd_part1.py:44-46).
template <int VPL, int LT>
__device__ __forceinline__ void load_token_logits(const void* __restrict__ logits_v, int64_t token,
                                                  bool live, int E, int64_t ld, int vec_ok,
                                                  float (&v)[VPL]) {
  const int lane16 = threadIdx.x & 15;
  // every lane of a row takes the same branch; DPP rows never straddle tokens
  const float NEG_INF = -__builtin_inff();
  const int e0 = lane16 * VPL;
  if constexpr (LT == DLB_DTYPE_F32) {
    const float* logits = (const float*)logits_v;
    if (live && vec_ok) {
      const f32x4* p = reinterpret_cast<const f32x4*>(logits + token * ld + e0);
#pragma unroll
      for (int q = 0; q < VPL / 4; ++q) {
        const f32x4 t = p[q];
        v[4 * q + 0] = t[0];
        v[4 * q + 1] = t[1];
        v[4 * q + 2] = t[2];
        v[4 * q + 3] = t[3];
      }
    } else {
#pragma unroll
      for (int j = 0; j < VPL; ++j)
        v[j] = (live && e0 + j < E) ? logits[token * ld + e0 + j] : NEG_INF;
    }
  } else {
    const unsigned short* logits = (const unsigned short*)logits_v;
    if (live && vec_ok) {
      const unsigned short* p = logits + token * ld + e0;
      unsigned int w[VPL / 2];
      if constexpr (VPL == 4) {
        const u32x2 t = *reinterpret_cast<const u32x2*>(p);
        w[0] = t[0];
        w[1] = t[1];
      } else {
#pragma unroll
        for (int q = 0; q < VPL / 8; ++q) {
          const u32x4 t = reinterpret_cast<const u32x4*>(p)[q];
#pragma unroll
          for (int i = 0; i < 4; ++i) w[4 * q + i] = t[i];
        }
      }
#pragma unroll
      for (int q = 0; q < VPL / 2; ++q) {
        v[2 * q] = Elem<LT>::lo(w[q]);
        v[2 * q + 1] = Elem<LT>::hi(w[q]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < VPL; ++j)
        v[j] = (live && e0 + j < E) ? Elem<LT>::load1(logits, token * ld + e0 + j) : NEG_INF;
    }
  }
}

// Routes one token, whose logits the calling DPP row holds: lane r < K of the row stores the
// r-th selected probability and expert and gets that expert back (other lanes and dead rows: -1).
// probs / masks (either may be null) are the outputs in the form of the reference's fused gate
// kernel (python/dlBLAS/dlblas/kernels/topk_gating_fwd_part1.py:47-60): the full softmax row
// gates[token, :] and, for every selection round r, the one-hot row masks[r, token, :] (int64).
//
// The K rounds are the kernel's serial chain, so a round is kept to the arg-max itself: keys of
// taken experts become 0, and a lane that keeps a result remembers its key, from which its
// logit (hence its probability) follows once, after the rounds.  A 16-bit logit and its expert
// share one 32-bit key (one row maximum per round); an fp32 logit takes two (the largest key,
// then the lowest expert that has it).  Carrying (key, expert) pairs and the probability
// through every round took three times the instructions.
template <int VPL, int LT>
__device__ __forceinline__ int32_t route_token(const float (&v)[VPL], float* __restrict__ weights,
                                               int32_t* __restrict__ ids, int64_t token, bool live,
                                               int E, int K, int renorm,
                                               float* __restrict__ probs = nullptr,
                                               int64_t* __restrict__ masks = nullptr, int64_t T = 0) {
  const int lane16 = threadIdx.x & 15;
  const int e0 = lane16 * VPL;

  // softmax statistics: p_e = exp(l_e - max) / sum
  float mx = v[0];
#pragma unroll
  for (int j = 1; j < VPL; ++j) mx = fmaxf(mx, v[j]);
  mx = row16_max(mx);
  float sum = 0.0f;
#pragma unroll
  for (int j = 0; j < VPL; ++j) sum += expf(v[j] - mx);  // exp(-inf) = 0 for the padding experts
  sum = row16_sum(sum);
  if (probs && live) {
#pragma unroll
    for (int j = 0; j < VPL; ++j)
      if (e0 + j < E) probs[token * E + e0 + j] = expf(v[j] - mx) / sum;  // = a selected expert's weight
  }

  // K rounds of arg-max over (orderable(logit), lowest index first); key 0 = no candidate
  constexpr bool k16 = LT != DLB_DTYPE_F32;
  uint32_t key[VPL];
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    // (16-bit logits are exact in the upper bits an fp32 key of theirs needs: 16 for bf16; an
    // fp16 value is ordered by its own 16 bits)
    if constexpr (k16) {
      const uint32_t h = Elem<LT>::pack(v[j] == 0.0f ? 0.0f : v[j], 0.0f) & 0xffffu;
      const uint32_t o = (h & 0x8000u) ? (h ^ 0xffffu) : (h | 0x8000u);
      key[j] = (o << 16) | (uint32_t)(256 - (e0 + j));
    } else {
      key[j] = max(orderable(v[j]), 1u);
    }
    if (e0 + j >= E) key[j] = 0u;
  }
  uint32_t my_key = 0u;  // lane r keeps the r-th selection
  int32_t my_id = 0;
  for (int r = 0; r < K; ++r) {
    uint32_t m = key[0];
#pragma unroll
    for (int j = 1; j < VPL; ++j) m = max(m, key[j]);
    m = row16_max_u32(m);
    int sel;
    if constexpr (k16) {
      sel = 256 - (int)(m & 0xffffu);
#pragma unroll
      for (int j = 0; j < VPL; ++j) key[j] = key[j] == m ? 0u : key[j];
    } else {
      uint32_t tag = 0u;
#pragma unroll
      for (int j = VPL - 1; j >= 0; --j) tag = key[j] == m ? (uint32_t)(256 - (e0 + j)) : tag;
      sel = 256 - (int)row16_max_u32(tag);
#pragma unroll
      for (int j = 0; j < VPL; ++j) key[j] = e0 + j == sel ? 0u : key[j];
    }
    if (masks && live) {
#pragma unroll
      for (int j = 0; j < VPL; ++j)
        if (e0 + j < E) masks[((int64_t)r * T + token) * E + e0 + j] = (e0 + j == sel) ? 1 : 0;
    }
    if (lane16 == r) {
      my_key = m;
      my_id = sel;
    }
  }
  float logit;
  if constexpr (k16) {
    const uint32_t o = my_key >> 16;
    logit = Elem<LT>::lo((o & 0x8000u) ? (o & 0x7fffu) : (o ^ 0xffffu));
  } else {
    logit = from_orderable(my_key);
  }
  const bool mine = live && lane16 < K;
  float w = mine ? expf(logit - mx) / sum : 0.0f;
  if (renorm) w = w / row16_sum(w);
  if (mine) {
    weights[token * K + lane16] = w;
    ids[token * K + lane16] = my_id;
    return my_id;
  }
  return -1;
}

// whole-row vector loads of the logits: 16-byte aligned base, rows a whole number of 16-byte pieces
inline bool logits_vector_ok(const void* logits, int dtype, int64_t ld) {
  return aligned16(logits) && ld % (dtype == DLB_DTYPE_F32 ? 4 : 8) == 0;
}

}  // namespace dlb
