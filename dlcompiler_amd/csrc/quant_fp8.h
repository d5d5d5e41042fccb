// fp8 (OCP e4m3fn) per-token-group quantisation of activations, shared by the stand-alone
// quantiser and by the launch that runs it beside the expert alignment.
// Rule: per group of 128 consecutive elements of a row, scale = max(absmax, 1e-10) / 448 and
// q = rne_e4m3(clamp(x / scale, +-448)); a NaN stays NaN and does not count for the absmax.
#pragma once
#include "common.h"

namespace dlb {

constexpr float kFp8Max = 448.0f;
constexpr float kQuantEps = 1e-10f;

__device__ __forceinline__ unsigned int pack4_fp8(float a, float b, float c, float d) {
  // v_cvt_pk_fp8_f32 rounds to nearest even.  The scale is the group's own maximum / 448, so a finite
  // quotient is at most 448 and a rounding, which rounds to 448 (only beyond 464 would it become NaN):
  // there is nothing to clamp, and fminf / fmaxf would turn a NaN into -448.
  int r = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
  r = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, r, true);
  return (unsigned int)r;
}

// f / scale, rounded as the division rounds (Markstein: one residual step from the rounded reciprocal), for
// |f| <= 448 scale, up to a rounding, and a finite scale; +0 for -0, whose residual is +0 as the sum then is.
__device__ __forceinline__ float finite_quotient(float f, float scale, float inv) {
  const float q = f * inv;
  return fmaf(fmaf(-q, scale, f), inv, q);
}
// ... with the sign of a zero, and `by` for the scale, 0 if that is infinite: 0 for a finite f then, else NaN.
__device__ __forceinline__ float divide_by_scale(float f, float by, float inv) {
  return __builtin_copysignf(finite_quotient(f, by, inv), f);
}

constexpr int kQuantThreads = 256;
constexpr int kQuantUnroll = 4;  // groups per DPP row and workgroup pass (loads issued together)
constexpr int kQuantGroupsPerBlock = (kQuantThreads / 16) * kQuantUnroll;

// One group by a DPP row, eight 16-bit values a lane: the lane's eight bytes, and the group's scale in every lane.
template <int DT>
__device__ __forceinline__ u32x2 quantise_group(const u32x4& raw, float& scale) {
  float v[8];
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    v[2 * w] = Elem<DT>::lo(raw[w]);
    v[2 * w + 1] = Elem<DT>::hi(raw[w]);
  }
  float amax = 0.0f;
#pragma unroll
  for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[j]));
  amax = row16_max(amax);
  scale = fmaxf(amax, kQuantEps) / kFp8Max;
  const float inv = 1.0f / scale, by = scale == __builtin_inff() ? 0.0f : scale;
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = divide_by_scale(v[j], by, inv);
  return u32x2{pack4_fp8(v[0], v[1], v[2], v[3]), pack4_fp8(v[4], v[5], v[6], v[7])};
}

// ... of eight fp32 values a lane, to the bytes that the epilogue of the gate_up GEMM gives
__device__ __forceinline__ u32x2 quantise_group_f32(const u32x4& lo, const u32x4& hi, float& scale) {
  float v[8], amax = 0.0f;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    v[j] = __uint_as_float(j < 4 ? lo[j] : hi[j - 4]);
    amax = fmaxf(amax, fabsf(v[j]));
  }
  scale = fmaxf(row16_max(amax), kQuantEps) / kFp8Max;
  const float inv = __builtin_amdgcn_rcpf(scale);  // the stored scale stays exact
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] *= inv;
  return u32x2{pack4_fp8(v[0], v[1], v[2], v[3]), pack4_fp8(v[4], v[5], v[6], v[7])};
}

struct QuantParams {
  const unsigned short* x;
  unsigned char* xq;
  float* xs;
  int64_t total_groups;
  int groups_per_row;
  int64_t ldx, ldq, lds;
};

// the work of thread `tid` of block `block` (kQuantThreads threads): one DPP row (16 lanes x 8 elements) per
// 128-element group, kQuantUnroll groups per row
template <int DT>
__device__ __forceinline__ void quant_fp8_group128_block(const QuantParams& q, int64_t block, int tid) {
  const int lane16 = tid & 15;
  int64_t row[kQuantUnroll];
  int gc[kQuantUnroll];
  bool live[kQuantUnroll];
  u32x4 raw[kQuantUnroll];
  const int64_t first = block * kQuantGroupsPerBlock;
  if (first >= q.total_groups) return;
  // One division for the block, in as many bits as it needs; its groups follow in 32 bits.  The loads go out without
  // a condition: groups past the last are the last one again, and are not stored.  (Four 64-bit divisions per lane
  // and loads behind branches: 4096 x 2048 bf16 8.2 us, so 8.05, on inputs from memory; its bytes take 4.)
  const uint32_t per_row = (uint32_t)q.groups_per_row;
  const int64_t row0 =
      q.total_groups <= 0xffffffff ? (int64_t)((uint32_t)first / per_row) : first / q.groups_per_row;
  const uint32_t gc0 = (uint32_t)(first - row0 * q.groups_per_row);
  const int left = (int)min(q.total_groups - first, (int64_t)kQuantGroupsPerBlock);
#pragma unroll
  for (int u = 0; u < kQuantUnroll; ++u) {
    const int local = 16 * u + (tid >> 4);
    live[u] = local < left;
    const uint32_t at = gc0 + (uint32_t)min(local, left - 1), r = at / per_row;
    row[u] = row0 + r;
    gc[u] = (int)(at - r * per_row);
    raw[u] = __builtin_nontemporal_load((const u32x4*)(q.x + row[u] * q.ldx + gc[u] * 128 + lane16 * 8));
  }
#pragma unroll
  for (int u = 0; u < kQuantUnroll; ++u) {
    float scale;
    const u32x2 o = quantise_group<DT>(raw[u], scale);
    if (live[u]) {
      *(u32x2*)(q.xq + row[u] * q.ldq + gc[u] * 128 + lane16 * 8) = o;
      if (lane16 == 0) q.xs[row[u] * q.lds + gc[u]] = scale;
    }
  }
}

// argument checks of the quantiser (shared by its two entry points); fills `q` on DLB_OK
inline int fill_quant_params(QuantParams& q, const void* x, void* xq, float* xs, int64_t M, int K,
                             int64_t ld_x, int64_t ld_q, int64_t ld_s, int dtype) {
  if (M < 0 || K < 0 || ld_x < K || ld_q < K || ld_s < K / 128) return DLB_ERR_BAD_ARG;
  if (M > 0 && K > 0 && (!x || !xq || !xs)) return DLB_ERR_BAD_ARG;
  if (dtype != DLB_DTYPE_BF16 && dtype != DLB_DTYPE_F16) return DLB_ERR_UNSUPPORTED;
  if (K % 128 != 0 || ld_x % 8 != 0 || ld_q % 8 != 0 || !aligned16(x) ||
      (reinterpret_cast<uintptr_t>(xq) & 7u) != 0)
    return DLB_ERR_UNSUPPORTED;
  q.x = (const unsigned short*)x;
  q.xq = (unsigned char*)xq;
  q.xs = xs;
  q.groups_per_row = K / 128;
  q.total_groups = M * (int64_t)(K / 128);
  q.ldx = ld_x;
  q.ldq = ld_q;
  q.lds = ld_s;
  return DLB_OK;
}

}  // namespace dlb
