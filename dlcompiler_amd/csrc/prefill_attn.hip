// Prefill attention: how a launch is cut, the merge of split rows, the C entry points.  The kernel,
// prefill_attn_kernel, is in prefill_attn.h.
#include <cmath>

#include "prefill_attn.h"
#include "prefill_rules.h"

namespace dlb {
namespace {

// Merge of the partial rows of every (query, head) of a sequence (blockIdx.y): half a wave per row (at most
// 128 dims), four rows per workgroup.  Rows without a visible key in any part become 0; rows in one part
// are written already.  A chain of memory latencies: the lengths, all the (maximum, denominator) pairs of
// a row in one load, then the parts eight at a time (3200 rows of 5 parts: 5.1 -> 4.5 us).
constexpr int kCombineRows = 4;
template <int DT>
__global__ __launch_bounds__(32 * kCombineRows) void prefill_combine_kernel(const PrefillParams p) {
  const int seq = blockIdx.y;
  const int idx = blockIdx.x * kCombineRows + (threadIdx.x >> 5);
  const int qrow = idx / p.Hq, head = idx - qrow * p.Hq;
  const int lane = threadIdx.x & 31;
  const int L = p.seq_len[seq], kv_total = p.kv_len[seq], hist = kv_total - L;
  const int64_t tok = p.start_loc[seq] + qrow;
  if (qrow >= L || hist < 0) return;
  const int block_q = 128 >> p.pack_shift;
  const TileRun run = visible_tiles(kv_total, hist, qrow / block_q * block_q, block_q, p.window);
  const int per = tiles_per_part(run, p.nsplit), parts = (run.end - run.first + per - 1) / per;
  if (parts < 2) return;
  const int64_t rows = p.tokens * p.Hq, row = tok * p.Hq + head;
  const float NONE = -__builtin_inff();
  typedef __attribute__((ext_vector_type(2))) float f32x2;
  // (loads are clamped, not conditional: behind a branch each would be waited for before the next)
  auto pair_of = [&](int s) {
    const f32x2 ml = *(const f32x2*)(p.ws_ml + 2 * (min(s, parts - 1) * rows + row));
    return s < parts ? ml : f32x2{NONE, 0.0f};
  };
  f32x2 first = pair_of(lane);  // parts 0 .. 31; the rest below
  float m = first[0];
  for (int s0 = 32; s0 < parts; s0 += 32) m = fmaxf(m, pair_of(s0 + lane)[0]);
#pragma unroll
  for (int d = 16; d >= 1; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, 32));
  float den = 0.0f;
  f32x4 acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const float* mine = p.ws_o + row * p.ws_d + min(4 * lane, p.ws_d - 4);
  for (int s0 = 0; s0 < parts; s0 += 32) {
    const f32x2 ml = s0 == 0 ? first : pair_of(s0 + lane);
    const float w = ml[0] == NONE ? 0.0f : __builtin_amdgcn_exp2f(ml[0] - m);
    den += w * ml[1];
    const int n = min(parts - s0, 32);
    for (int s = 0; s < n; s += 8) {
      f32x4 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        v[u] = *(const f32x4*)(mine + min(s0 + s + u, parts - 1) * rows * p.ws_d);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float wu = __shfl(w, s + u, 32);  // (past the last part: 0)
        if (wu > 0.0f) acc += wu * v[u];
      }
    }
  }
#pragma unroll
  for (int d = 16; d >= 1; d >>= 1) den += __shfl_xor(den, d, 32);
  const float inv = den > 0.0f ? 1.0f / den : 0.0f;
  if (4 * lane < p.dv)
    *(u32x2*)((unsigned short*)p.o + tok * p.o_st + head * p.o_sh + 4 * lane) =
        u32x2{Mma32<DT>::pack2(acc[0] * inv, acc[1] * inv), Mma32<DT>::pack2(acc[2] * inv, acc[3] * inv)};
}

}  // namespace
}  // namespace dlb

namespace dlb {
namespace {

// How a paged launch is cut.
// Query runs that fill a fraction of 128 rows share a workgroup by heads of their KV group.  Where that
// leaves few workgroups (up to half as many as CUs; the chip holds two per CU) their key tiles are split, from 32
// tiles on, eight tiles per part at least; with more workgroups or fewer tiles the partial rows cost
// more than the split saves (256 workgroups, 34 tiles: 43 us, split in two 49; 129 tiles: 156
// against 110).  Where nothing is split, heads share a workgroup only while every CU still has one.
// 32 heads (8 kv) of 128, neither -> both: 32 queries over 16000 keys 254 -> 25.5 us, 2 x 100 over 10000
// 166 -> 56, 16 x 8 - 32 over up to 8000 175 -> 95.
struct PackPlan {
  int pack_shift, nsplit;
  bool use;
};
PackPlan pack_plan(int B, int Hq, int Hkv, int D, int max_len, int64_t max_keys, int window) {
  PackPlan plan = {0, 1, false};
  if (D > 128) return plan;
  const int group = Hq / Hkv;
  const int64_t cus = current_device_cu_count();
  const int64_t reach = (int64_t)window + max_len;  // (windows of up to 2^31 - 1 come as "none")
  const int64_t seen = window > 0 && reach < max_keys ? reach : max_keys;
  const int64_t tiles = ceil_div(seen, kTileN);
  auto workgroups = [&](int shift) { return (int64_t)(Hq >> shift) * ceil_div(max_len, 128 >> shift) * B; };
  while (group % (2 << plan.pack_shift) == 0 && (int64_t)max_len << (plan.pack_shift + 1) <= 128 &&
         (tiles >= 32 || workgroups(plan.pack_shift + 1) >= cus))
    ++plan.pack_shift;
  const int64_t wgs = workgroups(plan.pack_shift);
  if (2 * wgs <= cus ? tiles >= 32 : wgs <= cus && tiles >= 96) {
    const int64_t most = tiles / kPartTiles;
    plan.nsplit = (int)(2 * cus / wgs < most ? 2 * cus / wgs : most);
  }
  plan.use = plan.pack_shift > 0 || plan.nsplit > 1;
  return plan;
}
size_t split_ws_bytes(int64_t tokens, int Hq, int Dv, int nsplit) {
  return nsplit > 1 ? (size_t)tokens * Hq * nsplit * ((Dv + 3) / 4 * 4 + 2) * sizeof(float) : 0;
}

// 64-row workgroups (half the chain of key tiles, RW = 2) or 128-row ones?  Counted in steps, one wave on one
// key tile (about 0.95 us with D > 64, else 0.67 us): 128-row workgroups take the longest chain of key
// tiles.  64-row ones take half of it, or a CU's share of the work where that is more, then half a step to merge,
// and they wait for their turn.  With D > 64 a CU holds one of them (128 KB of LDS), and each further round puts
// first loads that nothing hides, seven steps, in front of the chain; else it holds two, which hide most
// of that and together take 1.7 times as long.  Host code knows the longest sequence and, if the caller
// says so, the tokens of all: a batch's other histories count as 0.6 of the longest.
// 64-row / 128-row us, D = 128: 32 heads x 512 tokens 11.2 / 13.8, 16 x 1536 22.0 / 28.4, 16 x 2560 49.3 / 46.7,
// 8 x 4096 50.3 / 63.8, 8 heads x 8 x 300 15.4 / 10.7, 4 x 10 x 640 21.8 / 16.8; D = 64: 16 x 2048 19.5 / 26.6,
// 32 x 1280 16.4 / 19.9, 8 x 8 x 300 8.5 / 7.8, paged 32 x 6 x up to 478 17.6 / 14.9, 40 x 14 x 29 over up to 3355
// 33.8 / 46.4.  Over 1100 random batches of up to 2000 128-row workgroups the choice is 0.8 % above the better one on
// average ("up to 240 128-row workgroups": 2.0 %), at worst 32 % (50 % has been seen), where all histories are long and equal.
bool small_tiles(int Hq, int B, int D, int max_len, int64_t max_keys, int64_t tokens) {
  if (D > 128) return false;
  const double cus = current_device_cu_count();
  const double rows = (double)ceil_div(max_len, 64), chain = (double)ceil_div(max_keys, kTileN);
  const double history = chain > rows ? (chain - rows) * (0.4 + 0.6 * B) / B : 0.0;
  double tiles = B * rows;  // row tiles of 64
  if (tokens > 0 && tokens / 64.0 + 0.7 * B < tiles) tiles = tokens / 64.0 + 0.7 * B;
  if (tiles < B) tiles = B;  // (32 heads, 9 x up to 14 tokens over 151, D = 128: 64-row 14.0 us, 128-row 9.1)
  const double wgs = Hq * tiles, rounds = ceil(wgs / cus);
  double share = 0.5 * rounds * history + 0.25 * (rows + 1.0) * wgs / cus, wait = 7.0 * (rounds - 1.0);
  if (D <= 64) {
    share /= 1.2;
    wait = (rounds > 1.0 ? 1.0 : 0.0) + ceil(wgs / (2.0 * cus)) - 1.0;
  }
  const double half = ceil(0.5 * chain);
  return chain > 2.0 && (share > half ? share : half) + 0.5 + wait < 0.95 * chain;
}

// Shared argument checks and launch of both entry points; the paged fields of `p` are already
// filled in (or zeroed) by the caller.  tokens: rows of q, 0 if the caller does not say.
int launch_prefill(PrefillParams& p, bool paged, int B, int Hq, int Hkv, int Dk, int Dv, int max_len, int64_t tokens,
                   int64_t max_keys, float sm_scale, int dtype, void* ws, size_t ws_bytes, void* stream) {
  if (Dk % 8 != 0 || Dv % 8 != 0 || Dk > 256 || Dv > 256) return DLB_ERR_UNSUPPORTED;
  // head size the kernel instance is built for; past 128 there is one instance, for 256, that
  // takes every size on its ragged path (one workgroup per CU, one wave per SIMD: the 128 output
  // accumulators and the 64 query registers of a lane leave no room for a second wave)
  const int Dm = Dk > Dv ? Dk : Dv;
  const int D = Dm <= 64 ? 64 : Dm <= 96 ? 96 : Dm <= 128 ? 128 : 256;
  const bool ragged = Dk != D || Dv != D || D == 256;
  p.dk = Dk;
  p.dv = Dv;
  if (dtype != DLB_DTYPE_BF16 && dtype != DLB_DTYPE_F16) return DLB_ERR_UNSUPPORTED;
  if (!aligned16(p.q) || !aligned16(p.k) || !aligned16(p.v) ||
      (reinterpret_cast<uintptr_t>(p.o) & 7u) != 0)
    return DLB_ERR_UNSUPPORTED;
  const int64_t in_strides[] = {p.q_st, p.q_sh, p.k_st, p.k_sh, p.v_st, p.v_sh, p.k_sp, p.v_sp};
  for (int64_t sd : in_strides)
    if (sd % 8 != 0) return DLB_ERR_UNSUPPORTED;
  if (p.o_st % 4 != 0 || p.o_sh % 4 != 0) return DLB_ERR_UNSUPPORTED;
  if (B > 65535) return DLB_ERR_UNSUPPORTED;
  if (!(sm_scale > 0.0f)) return DLB_ERR_BAD_ARG;  // the tile maximum is taken before scaling

  p.Hq = Hq;
  p.Hkv = Hkv;
  p.group = Hq / Hkv;
  p.scale_log2e = sm_scale * 1.4426950408889634f;
  p.sm_scale = sm_scale;

  hipStream_t s = (hipStream_t)stream;
  PackPlan plan = {0, 1, false};
  if (paged) plan = pack_plan(B, Hq, Hkv, D, max_len, max_keys, p.window);
  if (plan.nsplit > 1) {
    const size_t need = split_ws_bytes(p.tokens, Hq, Dv, plan.nsplit);
    if (!ws) plan.nsplit = 1;  // (a caller without scratch)
    else if (ws_bytes < need || !aligned16(ws)) return DLB_ERR_WORKSPACE;
    plan.use = plan.pack_shift > 0 || plan.nsplit > 1;
  }
  p.pack_shift = plan.pack_shift;
  p.nsplit = plan.nsplit;
  p.B = B;
  p.ws_d = (Dv + 3) / 4 * 4;
  p.ws_o = (float*)ws;
  p.ws_ml = p.ws_o ? p.ws_o + (size_t)p.tokens * Hq * p.nsplit * p.ws_d : nullptr;
  const int64_t seen = p.window > 0 && (int64_t)p.window + max_len < max_keys ? (int64_t)p.window + max_len : max_keys;
  const bool small = !plan.use && small_tiles(Hq, B, D, max_len, seen, p.tokens);
  // Heads of a KV group share workgroups where the KV heads fall on the XCDs by themselves and the row tiles fit the grid.
  const int row_waves = small ? 2 : 4;
  int64_t qtiles = ceil_div(ceil_div(max_len, 32) * p.group, row_waves);
  // (A soft-cap has kernels of its own, which have no such form.)
  // (A kernel of its own: where heads do not share, its longer start costs 1 %, 16 heads, 16 kv, of 64: 176.2 / 178.7.)
  const bool share = !plan.use && !small && (8 % Hkv == 0 || Hkv % 8 == 0) && qtiles <= 65535 && p.group > 1 &&
                     p.group <= 4096 && !(paged && p.softcap > 0.0f) &&
                     heads_share_workgroups(paged, D, B, Hq, max_len, tokens, current_device_cu_count());
  // (exact: numbers below 2^18, at most 2^12 heads)
  p.share_rcp = share ? (unsigned int)(0x100000000ull / p.group + 1) : 0;
  if (!share) qtiles = ceil_div(max_len, 32 * row_waves);
  if (plan.use) qtiles = ceil_div(max_len, 128 >> p.pack_shift);
  if (qtiles > 65535 || (int64_t)B * p.nsplit > 65535) return DLB_ERR_UNSUPPORTED;
  const int head_groups = plan.use ? Hq >> p.pack_shift : share ? Hkv : Hq;
  // workgroups are dealt round-robin to the 8 XCDs by linear id; with Hq % 8 == 0 the
  // remap in the kernel puts heads {x, x+8, ...} -> consecutive heads on one XCD so a KV
  // group's four query heads hit the same L2.
  p.xcd_heads = head_groups % 8 == 0 && head_groups >= 16 ? head_groups >> 3 : 0;
  const dim3 grid = dim3((uint32_t)head_groups, (uint32_t)qtiles, (uint32_t)(B * p.nsplit));
  // pages that hold whole 64-key tiles take the kernel with one page look-up per tile (the lane
  // offsets inside a page are 32-bit)
  const bool tile_pages = paged && p.page % kTileN == 0 &&
                          (int64_t)p.page * p.k_st * 2 <= 0x7fffffff && (int64_t)p.page * p.v_st * 2 <= 0x7fffffff;
  const PrefillForm form = {dtype, D, tile_pages ? 2 : paged ? 1 : 0, ragged, small, plan.use, share};
  if (paged && p.softcap > 0.0f) launch_prefill_capped(p, form, grid, s);
  else launch_prefill_kernel<false>(p, form, grid, s);
  if (p.nsplit > 1) {
    const dim3 rows((uint32_t)ceil_div((int64_t)max_len * Hq, kCombineRows), (uint32_t)B);
    if (dtype == DLB_DTYPE_BF16)
      launch(prefill_combine_kernel<DLB_DTYPE_BF16>, rows, dim3(32 * kCombineRows), s, p);
    else
      launch(prefill_combine_kernel<DLB_DTYPE_F16>, rows, dim3(32 * kCombineRows), s, p);
  }
  return launch_status();
}

}  // namespace
}  // namespace dlb

extern "C" int dlb_prefill_attn_varlen(const void* q, const void* k, const void* v, void* o,
                                       const void* start_loc, const void* seq_len,
                                       int index64_mask, int B, int Hq, int Hkv, int D, int max_len, int64_t q_stride_tok,
                                       int64_t q_stride_head, int64_t k_stride_tok,
                                       int64_t k_stride_head, int64_t v_stride_tok,
                                       int64_t v_stride_head, int64_t o_stride_tok,
                                       int64_t o_stride_head, float sm_scale, int dtype,
                                       void* stream) {
  return dlb_prefill_attn_varlen_tokens(q, k, v, o, start_loc, seq_len, index64_mask, B, Hq, Hkv, D, max_len, q_stride_tok,
                                        q_stride_head, k_stride_tok, k_stride_head, v_stride_tok, v_stride_head,
                                        o_stride_tok, o_stride_head, sm_scale, dtype, 0, stream);
}

extern "C" int dlb_prefill_attn_varlen_tokens(const void* q, const void* k, const void* v, void* o,
                                       const void* start_loc, const void* seq_len,
                                       int index64_mask, int B, int Hq, int Hkv, int D, int max_len, int64_t q_stride_tok,
                                       int64_t q_stride_head, int64_t k_stride_tok,
                                       int64_t k_stride_head, int64_t v_stride_tok,
                                       int64_t v_stride_head, int64_t o_stride_tok,
                                       int64_t o_stride_head, float sm_scale, int dtype, int64_t tokens,
                                       void* stream) {
  using namespace dlb;
  if (B < 0 || Hq < 1 || Hkv < 1 || D < 1 || max_len < 0) return DLB_ERR_BAD_ARG;
  if (Hq % Hkv != 0) return DLB_ERR_BAD_ARG;
  if (B == 0 || max_len == 0) return DLB_OK;
  if (!q || !k || !v || !o || !start_loc || !seq_len) return DLB_ERR_BAD_ARG;
  PrefillParams p = {};
  p.q = q;
  p.k = k;
  p.v = v;
  p.o = o;
  if (index64_mask & ~3) return DLB_ERR_BAD_ARG;
  p.start_loc = idx_array(start_loc, index64_mask, 0);
  p.seq_len = idx_array(seq_len, index64_mask, 1);
  p.q_st = q_stride_tok;
  p.q_sh = q_stride_head;
  p.k_st = k_stride_tok;
  p.k_sh = k_stride_head;
  p.v_st = v_stride_tok;
  p.v_sh = v_stride_head;
  p.o_st = o_stride_tok;
  p.o_sh = o_stride_head;
  p.page = 1;
  p.page_shift = 0;
  p.window = -1;
  p.softcap = -1.0f;
  return launch_prefill(p, false, B, Hq, Hkv, D, D, max_len, tokens, max_len, sm_scale, dtype, nullptr, 0, stream);
}

extern "C" size_t dlb_paged_prefill_ws_bytes(int64_t tokens, int B, int Hq, int Hkv, int D, int Dv, int page,
                                             int max_blocks, int max_q_len, int window_size) {
  using namespace dlb;
  if (tokens < 1 || B < 1 || Hq < 1 || Hkv < 1 || Hq % Hkv != 0 || page < 1 || max_blocks < 1 || max_q_len < 1 ||
      D < 1 || Dv < 1)
    return 0;
  const PackPlan plan =
      pack_plan(B, Hq, Hkv, D > Dv ? D : Dv, max_q_len, (int64_t)page * max_blocks, window_size);
  return split_ws_bytes(tokens, Hq, Dv, plan.nsplit);
}

extern "C" int dlb_paged_prefill_attn(const void* q, const void* k_cache, const void* v_cache, void* o,
                                      const void* block_table, const void* q_start_loc, const void* q_len,
                                      const void* kv_len, int index64_mask, int B, int Hq, int Hkv, int D, int Dv,
                                      int page, int max_blocks, int max_q_len, int64_t q_stride_tok,
                                      int64_t q_stride_head, int64_t k_stride_page, int64_t k_stride_tok,
                                      int64_t k_stride_head, int64_t v_stride_page, int64_t v_stride_tok,
                                      int64_t v_stride_head, int64_t o_stride_tok, int64_t o_stride_head,
                                      int64_t bt_stride, float sm_scale, int window_size, float logit_softcapping,
                                      int dtype, void* stream) {
  return dlb_paged_prefill_attn_ws(q, k_cache, v_cache, o, block_table, q_start_loc, q_len, kv_len, index64_mask, B,
                                   Hq, Hkv, D, Dv, page, max_blocks, max_q_len, q_stride_tok, q_stride_head,
                                   k_stride_page, k_stride_tok, k_stride_head, v_stride_page, v_stride_tok,
                                   v_stride_head, o_stride_tok, o_stride_head, bt_stride, sm_scale, window_size,
                                   logit_softcapping, dtype, 0, nullptr, 0, stream);
}

extern "C" int dlb_paged_prefill_attn_ws(const void* q, const void* k_cache, const void* v_cache, void* o,
                                         const void* block_table, const void* q_start_loc, const void* q_len,
                                         const void* kv_len, int index64_mask, int B, int Hq, int Hkv, int D, int Dv,
                                         int page, int max_blocks, int max_q_len, int64_t q_stride_tok,
                                         int64_t q_stride_head, int64_t k_stride_page, int64_t k_stride_tok,
                                         int64_t k_stride_head, int64_t v_stride_page, int64_t v_stride_tok,
                                         int64_t v_stride_head, int64_t o_stride_tok, int64_t o_stride_head,
                                         int64_t bt_stride, float sm_scale, int window_size,
                                         float logit_softcapping, int dtype, int64_t tokens, void* ws,
                                         size_t ws_bytes, void* stream) {
  using namespace dlb;
  if (B < 0 || Hq < 1 || Hkv < 1 || D < 1 || Dv < 1 || max_q_len < 0 || page < 1 || max_blocks < 0)
    return DLB_ERR_BAD_ARG;
  if (Hq % Hkv != 0) return DLB_ERR_BAD_ARG;
  if (B == 0 || max_q_len == 0) return DLB_OK;
  if (!q || !k_cache || !v_cache || !o || !block_table || !q_start_loc || !q_len || !kv_len)
    return DLB_ERR_BAD_ARG;
  PrefillParams p = {};
  p.q = q;
  p.k = k_cache;
  p.v = v_cache;
  p.o = o;
  if (index64_mask & ~15) return DLB_ERR_BAD_ARG;
  p.block_table = idx_array(block_table, index64_mask, 0);
  p.start_loc = idx_array(q_start_loc, index64_mask, 1);
  p.seq_len = idx_array(q_len, index64_mask, 2);
  p.kv_len = idx_array(kv_len, index64_mask, 3);
  p.bt_stride = bt_stride;
  p.tokens = tokens;
  p.q_st = q_stride_tok;
  p.q_sh = q_stride_head;
  p.k_sp = k_stride_page;
  p.k_st = k_stride_tok;
  p.k_sh = k_stride_head;
  p.v_sp = v_stride_page;
  p.v_st = v_stride_tok;
  p.v_sh = v_stride_head;
  p.o_st = o_stride_tok;
  p.o_sh = o_stride_head;
  p.page = page;
  p.page_shift = (page & (page - 1)) == 0 ? __builtin_ctz((unsigned)page) : -1;
  p.window = window_size;
  p.softcap = logit_softcapping;
  return launch_prefill(p, true, B, Hq, Hkv, D, Dv, max_q_len, tokens, (int64_t)page * max_blocks, sm_scale, dtype, ws,
                        ws_bytes, stream);
}
