// MoE router for gfx950: softmax over experts, top-k selection, optional renormalisation.
//
// Semantics follow the router the reference's fused_moe is fed with
// (python/dlBLAS/tests/kernels/test_fused_moe.py:213-216: softmax in fp32, then top-k;
// python/dlBLAS/dlblas/kernels/fused_moe.py:322-323: weights / weights.sum(-1)), with the two
// points the reference leaves open fixed here: selection runs on the logits (the softmax is
// monotone, so this is the same order without depending on exp rounding) and equal logits
// resolve to the lowest expert index.  The fused softmax + K x argmax structure is that of
// python/dlBLAS/dlblas/kernels/topk_gating_fwd_part1.py:24-60; indices are written directly, and
// that kernel's own outputs (the full softmax and the [K, S, E] int64 one-hot masks) on request.
//
// Mapping: a token is owned by one DPP row (16 lanes); every lane holds VPL consecutive
// experts (VPL = 4 covers E <= 64 with one 128-bit load per lane), so a wave processes four
// tokens and every reduction (max, sum, K argmax rounds) is four DPP steps with no LDS.
#include "moe_route.h"

namespace dlb {
namespace {

template <int VPL, int LT>
__global__ __launch_bounds__(256) void moe_topk_softmax_kernel(
    const void* __restrict__ logits, float* __restrict__ weights, int32_t* __restrict__ ids,
    int64_t T, int E, int K, int64_t ld, int renorm, int vec_ok, float* __restrict__ probs,
    int64_t* __restrict__ masks) {
  const int64_t token = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
  float v[VPL];
  load_token_logits<VPL, LT>(logits, token, token < T, E, ld, vec_ok, v);
  route_token<VPL, LT>(v, weights, ids, token, token < T, E, K, renorm, probs, masks, T);
}

}  // namespace
}  // namespace dlb

extern "C" int dlb_moe_topk_softmax_f32(const void* logits, float* weights, int32_t* ids,
                                        float* probs, int64_t* masks, int64_t T, int E, int K,
                                        int64_t ld_logits, int logits_dtype, int renormalize,
                                        void* stream) {
  using namespace dlb;
  if (T < 0 || E < 1 || K < 1 || K > E || ld_logits < E) return DLB_ERR_BAD_ARG;
  if (K > 16 || E > 256) return DLB_ERR_UNSUPPORTED;
  if (logits_dtype != DLB_DTYPE_F32 && logits_dtype != DLB_DTYPE_BF16 && logits_dtype != DLB_DTYPE_F16)
    return DLB_ERR_UNSUPPORTED;
  if (T == 0) return DLB_OK;
  if (!logits || !weights || !ids) return DLB_ERR_BAD_ARG;
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid((uint32_t)ceil_div(T, 16)), block(256);
  const bool a16 = logits_vector_ok(logits, logits_dtype, ld_logits);
#define DLB_LAUNCH_ROUTE(LT_)                                                                      \
  do {                                                                                             \
    if (E <= 64)                                                                                   \
      launch((moe_topk_softmax_kernel<4, LT_>), grid, block, s, logits, weights, ids, \
                         T, E, K, ld_logits, renormalize, (int)(a16 && E == 64), probs, masks);    \
    else if (E <= 128)                                                                             \
      launch((moe_topk_softmax_kernel<8, LT_>), grid, block, s, logits, weights, ids, \
                         T, E, K, ld_logits, renormalize, (int)(a16 && E == 128), probs, masks);   \
    else                                                                                           \
      launch((moe_topk_softmax_kernel<16, LT_>), grid, block, s, logits, weights,   \
                         ids, T, E, K, ld_logits, renormalize, (int)(a16 && E == 256), probs,      \
                         masks);                                                                   \
  } while (0)
  if (logits_dtype == DLB_DTYPE_F32) DLB_LAUNCH_ROUTE(DLB_DTYPE_F32);
  else if (logits_dtype == DLB_DTYPE_BF16) DLB_LAUNCH_ROUTE(DLB_DTYPE_BF16);
  else DLB_LAUNCH_ROUTE(DLB_DTYPE_F16);
#undef DLB_LAUNCH_ROUTE
  return launch_status();
}
