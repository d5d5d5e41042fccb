// Expert alignment of MoE routing for gfx950: per-expert counts, expert-sorted flat slot ids
// padded per expert to a multiple of `block`, and the expert id of each block.
//
// The reference derives the same information with a full argsort of the flat id list plus a
// kernel that rescans that list once per expert
// (python/dlBLAS/dlblas/kernels/fused_moe.py:238-293, 314-320: exp_start/exp_end are the
// exclusive/inclusive cumulative sums of the per-expert counts).  Here it is a counting sort:
//   1. count:  every workgroup histograms its contiguous chunk of the flat id list in LDS and
//              writes one row of per-chunk counts (plain stores, so the result is reproducible);
//   2. scan:   one workgroup turns the [chunks, E] table into per-chunk start offsets, pads each
//              expert's total to `block`, and emits counts, block -> expert ids, the sentinel
//              pad slots and the padded total;
//      (for up to 256 chunks step 2 is folded into step 3: every workgroup reduces the small
//      count table itself, which saves a launch on the sizes a decoder layer produces)
//   3. place:  every workgroup re-reads its chunk in order and writes flat index i to
//              start[chunk][e] + (number of earlier i' in the chunk with the same e), the rank
//              coming from wave ballots, which makes the sort stable (ascending i per expert).
// Integer work only; no float or order-dependent atomics, so the output is bit-reproducible.
//
// Up to kOneSlots routing slots (a decode step) all of it runs in ONE workgroup and one launch,
// after the router itself where the caller asks for both.
#include <mutex>

#include "moe_route.h"
#include "quant_fp8.h"

namespace dlb {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
constexpr int kChunk = 2048;  // flat ids per workgroup (large inputs)
constexpr int kMaxE = 256;
constexpr int kFusedChunks = 256;  // rows of the count table the fused placement kernel reduces

// Flat ids per chunk (= per workgroup of the counting and the placement pass).  Inputs of up to
// kFusedChunks * kChunk ids are cut into as many chunks as the fused placement kernel takes (256),
// but not below one tile of 256 ids: a decoder layer's 25 k - 100 k routing slots then run on
// 96 - 256 workgroups with one or two tiles each instead of 12 - 48 workgroups that walk eight
// tiles one after the other.  Larger inputs use chunks of kChunk ids and the three-launch path.
__host__ __device__ inline int chunk_ids_for(int64_t numel) {
  if (numel > (int64_t)kFusedChunks * kChunk) return kChunk;
  const int64_t per = (numel + kFusedChunks - 1) / kFusedChunks;
  const int64_t rounded = (per + 63) / 64 * 64;
  return (int)(rounded < kThreads ? kThreads : rounded);
}
__host__ __device__ inline int64_t num_chunks(int64_t numel) {
  const int c = chunk_ids_for(numel);
  return numel > 0 ? (numel + c - 1) / c : 1;
}

// sets p[0 .. n) to v, as thread t of nt; 16 bytes per store where p is aligned
__device__ __forceinline__ void fill_words(int32_t* __restrict__ p, int64_t n, int32_t v, int64_t t, int64_t nt) {
  int64_t done = 0;
  if ((reinterpret_cast<uintptr_t>(p) & 15u) == 0) {
    typedef __attribute__((ext_vector_type(4))) int i32x4;
    const i32x4 q = {v, v, v, v};
    for (int64_t i = t; i < n / 4; i += nt) ((i32x4*)p)[i] = q;
    done = n / 4 * 4;
  }
  for (int64_t i = done + t; i < n; i += nt) p[i] = v;
}

// lanes of the wave holding the same expert, from ballots over the 9 key bits (bit 8 separates
// the dropped entries, e = -1 -> key 0x1ff)
__device__ __forceinline__ uint64_t same_expert(int32_t e) {
  const uint32_t key = (uint32_t)e & 0x1ffu;
  uint64_t peers = ~0ull;
#pragma unroll
  for (int b = 0; b < 9; ++b) {
    const bool bit = (key >> b) & 1u;
    const uint64_t m = __ballot(bit);
    peers &= bit ? m : ~m;
  }
  return peers;
}

// n / block by the block's reciprocal (2^32 / block, rounded down), whose estimate is at most one too small.  (A
// division by a number that only the host knows is 20 instructions, and a workgroup waits for these.)
__device__ __forceinline__ uint32_t blocks_of(uint32_t n, uint32_t block, uint32_t rcp) {
  const uint32_t q = __umulhi(n, rcp);
  return n - q * block >= block ? q + 1 : q;
}

// totals (0 past E, 16-byte aligned) -> padded expert bases base_s[0 .. E], by one wave: four
// experts per lane
__device__ __forceinline__ void scan_bases(const int32_t* total_s, int32_t* base_s, int E, int block, uint32_t rcp,
                                           int lane) {
  typedef __attribute__((ext_vector_type(4))) int i32x4;
  const i32x4 total = ((const i32x4*)total_s)[lane];
  int32_t pad[4], sum = 0;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    pad[c] = (int32_t)(blocks_of((uint32_t)total[c] + (uint32_t)block - 1u, block, rcp) * (uint32_t)block);
    sum += pad[c];
  }
  int32_t run = wave_inclusive_scan(sum) - sum;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    if (4 * lane + c < E) base_s[4 * lane + c] = run;
    run += pad[c];
  }
  if (lane == 63) base_s[E] = run;
}

struct AlignOut {
  int32_t* sorted_ids;
  int64_t sorted_cap;
  int32_t* expert_ids;
  int64_t expert_ids_cap;
  int32_t* counts;  // may be null
  int32_t* num_post_pad;
  int64_t numel;
  int E, block;
  uint32_t block_rcp;  // 2^32 / block, rounded down (block 1: 2^32 - 1)
};
uint32_t reciprocal_of(int block) { return block > 1 ? (uint32_t)(0x100000000ull / (uint32_t)block) : 0xffffffffu; }
// block -> expert ids (-1 past the last block) and the padded total, as thread t of nt (at least kMaxE): every thread
// takes blocks of one expert.  (Looking up a block's expert takes six or eight dependent reads of base_s.  With this
// and blocks_of, 48 tokens x 6 of 64 experts 5.58 -> 5.28 us a call, 64 x 8 of 256 10.9 -> 10.5, 16384 x 6 of 64
// 10.3 -> 10.05.)
__device__ __forceinline__ void write_block_experts(const AlignOut& o, const int32_t* base_s, int t, int nt) {
  const int32_t total_padded = base_s[o.E];
  if (t == 0) *o.num_post_pad = total_padded;
  // (no more threads than blocks: a workgroup without a share, which has a full chunk behind it where the first ones
  // have the short last one's, leaves at once; 1220 tokens x 8 of 64, 9.7 -> 9.5 us)
  if (o.expert_ids_cap < nt) nt = (int)(o.expert_ids_cap + kMaxE - 1) / kMaxE * kMaxE;
  if (t >= nt) return;
  const int shift = o.E > 1 ? 32 - __builtin_clz(o.E - 1) : 0;  // experts, rounded up to a power of two
  const int e = t & ((1 << shift) - 1);
  if (e < o.E) {
    const uint32_t first = blocks_of((uint32_t)base_s[e], o.block, o.block_rcp);
    const uint32_t end = blocks_of((uint32_t)base_s[e + 1], o.block, o.block_rcp);
    for (uint32_t b = first + (uint32_t)(t >> shift); b < end; b += (uint32_t)(nt >> shift)) o.expert_ids[b] = e;
  }
  for (int64_t b = blocks_of((uint32_t)total_padded, o.block, o.block_rcp) + t; b < o.expert_ids_cap; b += nt)
    o.expert_ids[b] = -1;
}

// ---- everything in one workgroup ------------------------------------------------------------
// A launch costs more than the work of a few thousand slots, so up to kOneSlots of them are
// counted, scanned and placed by one workgroup.  A wave takes consecutive slots, 64 at a time; its
// running per-expert counts give every slot its rank inside the wave, one scan over the waves and
// one over the experts turn ranks into positions.  The pad value is written everywhere first,
// while the ids are on their way.  Router and alignment of 48 tokens x 6 of 64 experts (block 128):
// 14.6 us a call in two launches, 5.8 us in this one; of 45 tokens x 8 of 256 experts, where the
// pads used to be written by one workgroup expert by expert, 35.7 -> 9.8 us.
constexpr int kOneThreads = 1024;
constexpr int kOneWaves = kOneThreads / kWave;
constexpr int kOneGroups = 4;  // slots per lane
constexpr int kOneSlots = kOneThreads * kOneGroups;

struct OneShared {
  int32_t wave_cnt[kOneWaves][kMaxE];  // running counts of a wave, then its exclusive prefix
  __attribute__((aligned(16))) int32_t total[kMaxE];
  int32_t base[kMaxE + 1];
};
__device__ __forceinline__ void align_one_begin(const AlignOut& o, OneShared& s) {
  fill_words(o.sorted_ids, o.sorted_cap, (int32_t)o.numel, threadIdx.x, kOneThreads);
  for (int i = threadIdx.x; i < kOneWaves * kMaxE; i += kOneThreads) (&s.wave_cnt[0][0])[i] = 0;
}
// slots of a wave
__device__ __forceinline__ int one_wave_slots(int numel) { return (numel + kOneThreads - 1) / kOneThreads * kWave; }
// get(g, i): expert of slot i, the lane's slot of group g, or -1.  Between align_one_begin and this call lies a
// barrier.
template <typename Get>
__device__ __forceinline__ void align_one_workgroup(const AlignOut& o, OneShared& s, Get get) {
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  const int numel = (int)o.numel, E = o.E;
  const int per = one_wave_slots(numel);
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  int32_t e[kOneGroups], rank[kOneGroups];
#pragma unroll
  for (int g = 0; g < kOneGroups; ++g) {
    const int i = wave * per + g * kWave + lane;
    e[g] = (g * kWave < per && i < numel) ? get(g, i) : -1;
    rank[g] = 0;
  }
#pragma unroll
  for (int g = 0; g < kOneGroups; ++g) {
    if (g * kWave < per) {
      const uint64_t peers = same_expert(e[g]);
      const int r = __popcll(peers & lt_mask);
      if (e[g] >= 0) {
        const int32_t before = s.wave_cnt[wave][e[g]];
        rank[g] = before + r;
        // (the wave's own row: its LDS operations complete in order)
        if (r == 0) s.wave_cnt[wave][e[g]] = before + __popcll(peers);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  }
  __syncthreads();
  if (tid < kMaxE) {  // (nothing was counted past E)
    int32_t run = 0;
#pragma unroll
    for (int w = 0; w < kOneWaves; ++w) {
      const int32_t c = s.wave_cnt[w][tid];
      s.wave_cnt[w][tid] = run;
      run += c;
    }
    s.total[tid] = run;
    if (tid < E && o.counts) o.counts[tid] = run;
  }
  __syncthreads();
  if (wave == 0) scan_bases(s.total, s.base, E, o.block, o.block_rcp, lane);
  __syncthreads();
#pragma unroll
  for (int g = 0; g < kOneGroups; ++g)
    if (e[g] >= 0)
      o.sorted_ids[s.base[e[g]] + s.wave_cnt[wave][e[g]] + rank[g]] = wave * per + g * kWave + lane;
  write_block_experts(o, s.base, tid, kOneThreads);
}

__device__ __forceinline__ void align_one_ids(const AlignOut& o, const IdxArray ids) {
  __shared__ OneShared s;
  // (requested before the pads are written; the last id again past the end, rather than a branch around a load)
  const int per = one_wave_slots((int)o.numel), at = threadIdx.x / kWave * per + (threadIdx.x & (kWave - 1));
  int32_t id[kOneGroups];
#pragma unroll
  for (int g = 0; g < kOneGroups; ++g) id[g] = o.numel > 0 ? ids[min(at + g * kWave, (int)o.numel - 1)] : -1;
  align_one_begin(o, s);
  __syncthreads();
  align_one_workgroup(o, s, [&](int g, int) { return (id[g] >= 0 && id[g] < o.E) ? id[g] : -1; });
}
__global__ __launch_bounds__(kOneThreads) void align_one_kernel(const AlignOut o, const IdxArray ids) {
  align_one_ids(o, ids);
}
// ... with the fp8 activation quantiser on the other workgroups (see align_place_quant_kernel)
static_assert(kOneThreads % kQuantThreads == 0, "whole quantiser blocks per workgroup");
constexpr int kOneQuantBlocks = kOneThreads / kQuantThreads;
template <int DT>
__global__ __launch_bounds__(kOneThreads) void align_one_quant_kernel(const AlignOut o, const IdxArray ids,
                                                                      const QuantParams q) {
  if (blockIdx.x == 0) align_one_ids(o, ids);
  else
    quant_fp8_group128_block<DT>(q, ((int64_t)blockIdx.x - 1) * kOneQuantBlocks + threadIdx.x / kQuantThreads,
                                 threadIdx.x % kQuantThreads);
}

// ---- router and alignment -------------------------------------------------------------------
struct RouteParams {
  const void* logits;
  float* weights;
  int32_t* ids;
  int64_t T;
  int E, K;
  int64_t ld;
  int renorm, vec_ok;
};

// Router, then the alignment of its own selections, in one workgroup: 64 tokens per pass.  A pass keeps
// the CU's SIMDs busy, so past some tokens the second launch, whose router has 16 of them on a CU, is the
// cheaper way (one / two launches, fp32, us: 64 experts, 80 tokens 6.8 / 7.3, 96 7.35 / 7.3, 128 9.0 / 7.4; 128
// experts, 48 tokens 7.6 / 8.1, 64 8.6 / 8.1; 256 experts, 32 tokens 9.2 / 10.0, 48 11.2 / 9.8).
constexpr int one_workgroup_tokens(int experts_per_lane) {
  return experts_per_lane == 4 ? 96 : experts_per_lane == 8 ? 56 : 36;
}
constexpr int kRouteSlots = one_workgroup_tokens(4) * 16;
static_assert(kRouteSlots <= kOneSlots, "the routed slots fit one workgroup's alignment");
template <int VPL, int LT>
__global__ __launch_bounds__(kOneThreads) void route_align_one_kernel(const RouteParams p, const AlignOut o) {
  __shared__ OneShared s;
  __shared__ int32_t ids_s[kRouteSlots];
  const int row = threadIdx.x >> 4;
  float v[VPL];
  load_token_logits<VPL, LT>(p.logits, row, row < p.T, p.E, p.ld, p.vec_ok, v);
  align_one_begin(o, s);
  // (a wave without a token leaves the SIMD to those that have one)
  for (int64_t first = 0; first + 4 * (threadIdx.x / kWave) < p.T; first += 64) {
    const int64_t token = first + row;
    float next[VPL];
    load_token_logits<VPL, LT>(p.logits, token + 64, token + 64 < p.T, p.E, p.ld, p.vec_ok, next);
    const int32_t e = route_token<VPL, LT>(v, p.weights, p.ids, token, token < p.T, p.E, p.K, p.renorm);
    if (e >= 0) ids_s[token * p.K + (threadIdx.x & 15)] = e;
#pragma unroll
    for (int j = 0; j < VPL; ++j) v[j] = next[j];
  }
  __syncthreads();
  align_one_workgroup(o, s, [&](int, int i) { return ids_s[i]; });
}

// More tokens: two launches.  First the router, THREADS / 16 * PASSES tokens per workgroup, which also
// writes a row of the [chunks, E] count table: the experts selected by exactly those tokens.  A
// token selects an expert at most once, so a count fits a byte, and the table the second launch
// reduces in every workgroup is a quarter of what 32-bit counts take.  The pad value goes
// everywhere meanwhile (the second launch scatters the slots over it).  Both launches are bound by
// latency: 16384 tokens x 6 of 64 experts 15.7 -> 12.8 us a call, 9336 x 8 of 256 43.9 -> 16.6 us.
template <int VPL, int THREADS, int PASSES, int LT>
__global__ __launch_bounds__(THREADS) void route_count_kernel(const RouteParams p, const AlignOut o,
                                                                  uint32_t* __restrict__ table) {
  constexpr int kRows = THREADS / 16;  // tokens per pass
  static_assert(kRows * PASSES < 256, "counts are bytes");
  static_assert(THREADS >= kMaxE, "a thread per expert");
  __shared__ int32_t hist[kMaxE];
  if (threadIdx.x < kMaxE) hist[threadIdx.x] = 0;
  const int64_t first = (int64_t)blockIdx.x * (kRows * PASSES);
  float v[PASSES][VPL];
#pragma unroll
  for (int pass = 0; pass < PASSES; ++pass) {  // all loads first: one memory round trip
    const int64_t token = first + pass * kRows + (threadIdx.x >> 4);
    load_token_logits<VPL, LT>(p.logits, token, token < p.T, p.E, p.ld, p.vec_ok, v[pass]);
  }
  fill_words(o.sorted_ids, o.sorted_cap, (int32_t)o.numel, (int64_t)blockIdx.x * THREADS + threadIdx.x,
             (int64_t)gridDim.x * THREADS);
  __syncthreads();
#pragma unroll
  for (int pass = 0; pass < PASSES; ++pass) {
    const int64_t token = first + pass * kRows + (threadIdx.x >> 4);
    const int32_t e = route_token<VPL, LT>(v[pass], p.weights, p.ids, token, token < p.T, p.E, p.K, p.renorm);
    if (e >= 0) atomicAdd(&hist[e], 1);  // integer add: order-insensitive
  }
  __syncthreads();
  const int words = (p.E + 3) / 4;
  if (threadIdx.x < words) {
    const int e = 4 * threadIdx.x;  // (entries past E are zero)
    table[(int64_t)blockIdx.x * words + threadIdx.x] = (uint32_t)hist[e] | (uint32_t)hist[e + 1] << 8 |
                                                       (uint32_t)hist[e + 2] << 16 | (uint32_t)hist[e + 3] << 24;
  }
}

// Second launch: every workgroup reduces the count table itself (expert totals and the part of
// them in earlier chunks) and places its chunk.  The ranks inside the chunk need nothing from the
// table, so they are worked out while its rows are on their way.
constexpr int kRouteGroups = 8;  // slots per lane: chunks of up to 128 tokens x 16
__global__ __launch_bounds__(kThreads) void route_place_kernel(const IdxArray ids, const AlignOut o,
                                                               const uint32_t* __restrict__ table, int chunks,
                                                               int chunk_ids) {
  __shared__ int32_t wave_cnt[kWaves][kMaxE];
  __shared__ __attribute__((aligned(16))) int32_t total_s[kMaxE];
  __shared__ int32_t before_s[kMaxE];
  __shared__ int32_t base_s[kMaxE + 1];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  const int E = o.E, me = blockIdx.x;
  const int64_t begin = (int64_t)me * chunk_ids;
  const int count = (int)(begin + chunk_ids < o.numel ? chunk_ids : o.numel - begin);
  const int per = (count + kThreads - 1) / kThreads * kWave;  // slots per wave
  int32_t e[kRouteGroups], rank[kRouteGroups];
#pragma unroll
  for (int g = 0; g < kRouteGroups; ++g) {
    const int i = wave * per + g * kWave + lane;
    e[g] = (g * kWave < per && i < count) ? ids[begin + i] : -1;
    rank[g] = 0;
  }
  // table columns of four experts: thread = (column tid % W, rows tid / W, + 256 / W, ...)
  const int words = (E + 3) / 4, W = words <= 16 ? 16 : words <= 32 ? 32 : 64;
  const int col = tid % W, slices = kThreads / W;
  const bool live = col < words;
  uint32_t tot_lo = 0, tot_hi = 0, bef_lo = 0, bef_hi = 0;  // 16-bit sums of experts 0, 2 and 1, 3 of the column
  constexpr int kRowsInFlight = 16;
  uint32_t n[kRowsInFlight];
  auto request = [&](int r0) {
#pragma unroll
    for (int u = 0; u < kRowsInFlight; ++u)
      n[u] = (live && r0 + u * slices < chunks) ? table[(int64_t)(r0 + u * slices) * words + col] : 0u;
  };
  auto collect = [&](int r0) {
#pragma unroll
    for (int u = 0; u < kRowsInFlight; ++u) {
      const uint32_t lo = n[u] & 0x00ff00ffu, hi = (n[u] >> 8) & 0x00ff00ffu;
      tot_lo += lo;
      tot_hi += hi;
      if (r0 + u * slices < me) {
        bef_lo += lo;
        bef_hi += hi;
      }
    }
  };
  request(tid / W);
  for (int i = tid; i < kWaves * kMaxE; i += kThreads) (&wave_cnt[0][0])[i] = 0;
  total_s[tid] = 0;
  before_s[tid] = 0;
  __syncthreads();
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
  for (int g = 0; g < kRouteGroups; ++g) {
    if (g * kWave < per) {
      const uint64_t peers = same_expert(e[g]);
      const int r = __popcll(peers & lt_mask);
      if (e[g] >= 0) {
        const int32_t before = wave_cnt[wave][e[g]];
        rank[g] = before + r;
        if (r == 0) wave_cnt[wave][e[g]] = before + __popcll(peers);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  }
  collect(tid / W);
  for (int r0 = tid / W + kRowsInFlight * slices; r0 < chunks; r0 += kRowsInFlight * slices) {
    request(r0);
    collect(r0);
  }
  if (live) {
    const int e0 = 4 * col;
    atomicAdd(&total_s[e0], (int)(tot_lo & 0xffffu));
    atomicAdd(&total_s[e0 + 1], (int)(tot_hi & 0xffffu));
    atomicAdd(&total_s[e0 + 2], (int)(tot_lo >> 16));
    atomicAdd(&total_s[e0 + 3], (int)(tot_hi >> 16));
    atomicAdd(&before_s[e0], (int)(bef_lo & 0xffffu));
    atomicAdd(&before_s[e0 + 1], (int)(bef_hi & 0xffffu));
    atomicAdd(&before_s[e0 + 2], (int)(bef_lo >> 16));
    atomicAdd(&before_s[e0 + 3], (int)(bef_hi >> 16));
  }
  __syncthreads();
  if (wave == 0) scan_bases(total_s, base_s, E, o.block, o.block_rcp, lane);
  __syncthreads();
  if (tid < E) {  // first position of each wave's slots of expert tid
    int32_t run = base_s[tid] + before_s[tid];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const int32_t c = wave_cnt[w][tid];
      wave_cnt[w][tid] = run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int g = 0; g < kRouteGroups; ++g)
    if (e[g] >= 0)
      o.sorted_ids[wave_cnt[wave][e[g]] + rank[g]] = (int32_t)(begin + wave * per + g * kWave + lane);
  // (the blocks' experts are shared out: by one workgroup, which looked up one after the other, they took longer than
  // all the rest, 16384 tokens x 6 of 64 experts, 1600 blocks, 13.3 us a call against 10.3.  The last chunk, which is
  // the shortest, has the first share, and few blocks need no other: behind the first one's full chunk, measured with
  // look-ups too, 147 tokens x 8 of 64 took 9.2 us, so 8.7, 1090 x 8 of 256 15.6 and 15.1, 8192 x 8 of 256 15.0 and 14.8)
  write_block_experts(o, base_s, (chunks - 1 - me) * kThreads + tid, chunks * kThreads);
  if (me == chunks - 1 && tid < E && o.counts) o.counts[tid] = total_s[tid];
}

__global__ __launch_bounds__(kThreads) void align_count_kernel(const IdxArray ids,
                                                               int64_t numel, int E, int chunk_ids,
                                                               int32_t* __restrict__ chunk_counts,
                                                               int32_t* __restrict__ sorted_ids,
                                                               int64_t sorted_cap) {
  __shared__ int32_t hist[kMaxE];
  // (the pad value goes everywhere here; the placement scatters the slots over it)
  fill_words(sorted_ids, sorted_cap, (int32_t)numel, (int64_t)blockIdx.x * kThreads + threadIdx.x,
             (int64_t)gridDim.x * kThreads);
  for (int e = threadIdx.x; e < E; e += kThreads) hist[e] = 0;
  __syncthreads();
  const int64_t begin = (int64_t)blockIdx.x * chunk_ids;
  const int64_t end = begin + chunk_ids < numel ? begin + chunk_ids : numel;
  for (int64_t i = begin + threadIdx.x; i < end; i += kThreads) {
    const int32_t e = ids[i];
    if (e >= 0 && e < E) atomicAdd(&hist[e], 1);  // integer add: order-insensitive
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += kThreads) chunk_counts[(int64_t)blockIdx.x * E + e] = hist[e];
}

// One workgroup of 1024 threads: sub-group q = tid / E' (E' = E rounded up to 64) scans a
// slice of the chunk rows for expert tid % E', the slices are combined through LDS, so the
// dependent chain per thread is chunks / groups long instead of chunks.
constexpr int kScanThreads = 1024;

__global__ __launch_bounds__(kScanThreads) void align_scan_kernel(
    int32_t* __restrict__ chunk_counts /* in: counts, out: start offsets */, int64_t chunks, const AlignOut o) {
  const int E = o.E, block = o.block;
  __shared__ int32_t part_s[kScanThreads];  // [group][expert'] slice totals -> slice bases
  __shared__ __attribute__((aligned(16))) int32_t total_s[kMaxE];
  __shared__ int32_t base_s[kMaxE + 1];
  const int tid = threadIdx.x;
  const int ep = (E + 63) & ~63;           // experts rounded up to a whole wave
  const int groups = kScanThreads / ep;     // >= 4 for E <= 256
  const int e = tid % ep, q = tid / ep;
  const bool live = (e < E) && (q < groups);
  const int64_t per = (chunks + groups - 1) / groups;
  const int64_t c0 = q * per, c1 = (c0 + per < chunks) ? c0 + per : chunks;

  int32_t slice = 0;
  if (live)
    for (int64_t c = c0; c < c1; ++c) slice += chunk_counts[c * E + e];
  part_s[tid] = slice;
  __syncthreads();
  if (tid < E) {  // exclusive scan over the groups of this expert, total
    int32_t run = 0;
    for (int g2 = 0; g2 < groups; ++g2) {
      const int32_t v = part_s[g2 * ep + tid];
      part_s[g2 * ep + tid] = run;
      run += v;
    }
    total_s[tid] = run;
  } else if (tid < kMaxE) {
    total_s[tid] = 0;
  }
  __syncthreads();
  if (tid < 64) scan_bases(total_s, base_s, E, block, o.block_rcp, tid);
  __syncthreads();
  if (live) {
    // chunk start offsets of this slice for the placement pass
    int32_t run = base_s[e] + part_s[q * ep + e];
    for (int64_t c = c0; c < c1; ++c) {
      const int32_t n = chunk_counts[c * E + e];
      chunk_counts[c * E + e] = run;
      run += n;
    }
  }
  if (tid < E && o.counts) o.counts[tid] = total_s[tid];
  write_block_experts(o, base_s, tid, kScanThreads);
}

__global__ __launch_bounds__(kThreads) void align_place_kernel(
    const IdxArray ids, int64_t numel, int E,
    const int32_t* __restrict__ chunk_start, int32_t* __restrict__ sorted_ids) {
  __shared__ int32_t cursor[kMaxE];           // next free slot per expert for this chunk
  __shared__ int32_t wave_cnt[kWaves][kMaxE];  // per-tile, per-wave counts
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  for (int e = threadIdx.x; e < E; e += kThreads) cursor[e] = chunk_start[(int64_t)blockIdx.x * E + e];
  for (int i = threadIdx.x; i < kWaves * kMaxE; i += kThreads) (&wave_cnt[0][0])[i] = 0;
  __syncthreads();

  const int64_t begin = (int64_t)blockIdx.x * kChunk;
  const int64_t end = begin + kChunk < numel ? begin + kChunk : numel;
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  for (int64_t tile = begin; tile < end; tile += kThreads) {  // uniform trip count
    const int64_t i = tile + threadIdx.x;
    int32_t e = -1;
    if (i < end) {
      e = ids[i];
      if (e < 0 || e >= E) e = -1;
    }
    const uint64_t peers = same_expert(e);
    const int rank_in_wave = __popcll(peers & lt_mask);
    const int peer_count = __popcll(peers);
    if (e >= 0 && rank_in_wave == 0) wave_cnt[wave][e] = peer_count;
    __syncthreads();
    if (e >= 0) {
      int32_t pos = cursor[e] + rank_in_wave;
      for (int w = 0; w < wave; ++w) pos += wave_cnt[w][e];
      sorted_ids[pos] = (int32_t)i;
    }
    __syncthreads();
    for (int x = threadIdx.x; x < E; x += kThreads) {
      int32_t add = 0;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        add += wave_cnt[w][x];
        wave_cnt[w][x] = 0;
      }
      cursor[x] += add;
    }
    __syncthreads();
  }
}

// Scan and placement in one launch, for inputs of up to kFusedChunks chunks: every workgroup
// reduces the (small) [chunks, E] count table itself -- expert totals, padded expert bases and
// the offsets of its own chunk -- instead of waiting for a separate one-workgroup scan kernel;
// one extra workgroup emits what the scan kernel emits (counts, block -> expert ids, padded total).  The table is only read here.
struct PlaceParams {
  IdxArray ids;  // int32 or int64 (the routing ids as torch.topk returns them)
  const int32_t* chunk_counts;
  int chunks, chunk_ids;
  AlignOut out;
};

// the work of workgroup `me` (0 .. chunks) of the fused scan + placement
__device__ __forceinline__ void align_place_fused_block(const PlaceParams& pp, const int me) {
  const IdxArray ids = pp.ids;
  const int64_t numel = pp.out.numel;
  const int E = pp.out.E, chunks = pp.chunks, chunk_ids = pp.chunk_ids;
  const int32_t* __restrict__ chunk_counts = pp.chunk_counts;
  int32_t* __restrict__ sorted_ids = pp.out.sorted_ids;
  __shared__ int32_t cursor[kMaxE];            // next free slot per expert for this chunk
  __shared__ int32_t wave_cnt[kWaves][kMaxE];  // per-tile, per-wave counts
  __shared__ __attribute__((aligned(16))) int32_t total_s[kMaxE];
  __shared__ int32_t base_s[kMaxE + 1];
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid / kWave;

  // this chunk's first ids are requested before the count table is reduced (they do not depend
  // on it), each later tile's while the tile before it is placed
  const int64_t begin = (int64_t)me * chunk_ids;  // chunk_ids flat ids per chunk (kChunk by default)
  const int64_t end = begin + chunk_ids < numel ? begin + chunk_ids : numel;
  auto load_expert = [&](int64_t tile) -> int32_t {
    const int64_t i = tile + tid;
    int32_t e = -1;
    if (i < end) {
      e = ids[i];
      if (e < 0 || e >= E) e = -1;
    }
    return e;
  };
  int32_t e_next = load_expert(begin);

  // totals and the part of them that lies in earlier chunks: sub-group q = tid / E' (E' = E
  // rounded up to a whole wave) sums a slice of the chunk rows for expert tid % E', the slices
  // meet in LDS (wave_cnt doubles as the scratch for that before it is cleared)
  const int ep = (E + 63) & ~63;
  const int groups = kThreads / ep;  // 4, 2 or 1
  {
    const int e = tid % ep, q = tid / ep;
    const int per = (chunks + groups - 1) / groups;
    const int c0 = q * per, c1 = min(c0 + per, chunks);
    int32_t total = 0, before_part = 0;
    if (e < E && q < groups) {
      // The table was written by the launch before this one, on other XCDs: every dependent batch
      // of loads is a full memory round trip.  All rows of the slice are therefore requested at
      // once (64 per thread cover 256 chunks of up to 64 experts; wider expert counts take a
      // second or fourth batch).
      constexpr int kRowsInFlight = 64;
      for (int cb = c0; cb < c1; cb += kRowsInFlight) {
        int32_t n[kRowsInFlight];
#pragma unroll
        for (int u = 0; u < kRowsInFlight; ++u)
          n[u] = (cb + u < c1) ? chunk_counts[(int64_t)(cb + u) * E + e] : 0;
#pragma unroll
        for (int u = 0; u < kRowsInFlight; ++u) {
          total += n[u];
          if (cb + u < me) before_part += n[u];
        }
      }
    }
    int32_t* part = &wave_cnt[0][0];  // [2][groups][ep] <= 2 * 256 entries
    if (q < groups) {
      part[q * ep + e] = total;
      part[kThreads + q * ep + e] = before_part;
    }
  }
  __syncthreads();
  int32_t before = 0;
  if (tid < E) {
    const int32_t* part = &wave_cnt[0][0];
    int32_t total = 0;
    for (int q = 0; q < groups; ++q) {
      total += part[q * ep + tid];
      before += part[kThreads + q * ep + tid];
    }
    total_s[tid] = total;
  } else {
    total_s[tid] = 0;
  }
  __syncthreads();
  for (int i = tid; i < kWaves * kMaxE; i += kThreads) (&wave_cnt[0][0])[i] = 0;
  __syncthreads();
  if (tid < 64) scan_bases(total_s, base_s, E, pp.out.block, pp.out.block_rcp, tid);
  __syncthreads();
  if (tid < E) cursor[tid] = base_s[tid] + before;
  if (me == chunks) {  // the extra workgroup: what the scan kernel emits besides offsets
    if (tid < E && pp.out.counts) pp.out.counts[tid] = total_s[tid];
    write_block_experts(pp.out, base_s, tid, kThreads);
    return;
  }
  __syncthreads();

  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  for (int64_t tile = begin; tile < end; tile += kThreads) {  // uniform trip count
    const int64_t i = tile + tid;
    const int32_t e = e_next;
    e_next = load_expert(tile + kThreads);
    const uint64_t peers = same_expert(e);
    const int rank_in_wave = __popcll(peers & lt_mask);
    const int peer_count = __popcll(peers);
    if (e >= 0 && rank_in_wave == 0) wave_cnt[wave][e] = peer_count;
    __syncthreads();
    if (e >= 0) {
      int32_t pos = cursor[e] + rank_in_wave;
      for (int w = 0; w < wave; ++w) pos += wave_cnt[w][e];
      sorted_ids[pos] = (int32_t)i;
    }
    __syncthreads();
    for (int x = tid; x < E; x += kThreads) {
      int32_t add = 0;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        add += wave_cnt[w][x];
        wave_cnt[w][x] = 0;
      }
      cursor[x] += add;
    }
    __syncthreads();
  }
}

__global__ __launch_bounds__(kThreads) void align_place_fused_kernel(const PlaceParams pp) {
  align_place_fused_block(pp, blockIdx.x);
}

// The fused scan + placement and the fp8 activation quantiser in ONE launch: workgroups
// 0 .. chunks run the placement, the ones after them quantise.  The two jobs share nothing; run
// side by side they cost one launch and the longer of the two instead of two launches.
static_assert(kQuantThreads == kThreads, "one workgroup size for both jobs");
template <int DT>
__global__ __launch_bounds__(kThreads) void align_place_quant_kernel(const PlaceParams pp,
                                                                     const QuantParams q) {
  const int nplace = pp.chunks + 1;
  if ((int)blockIdx.x < nplace) align_place_fused_block(pp, blockIdx.x);
  else quant_fp8_group128_block<DT>(q, (int64_t)blockIdx.x - nplace, threadIdx.x);
}

}  // namespace
}  // namespace dlb

extern "C" size_t dlb_moe_align_ws_bytes(int64_t numel, int E) {
  if (numel < 0 || E < 1) return 0;
  return (size_t)dlb::num_chunks(numel) * (size_t)E * sizeof(int32_t);
}

namespace dlb {
namespace {

// argument checks shared by the two alignment entry points (everything but the scratch)
int check_align_args(const void* topk_ids, int64_t numel, int E, int block,
                     const int32_t* sorted_ids, int64_t sorted_cap, const int32_t* expert_ids,
                     int64_t expert_ids_cap, const int32_t* num_post_pad) {
  if (numel < 0 || E < 1 || block < 1) return DLB_ERR_BAD_ARG;
  if (E > kMaxE) return DLB_ERR_UNSUPPORTED;
  if (numel + (int64_t)E * block >= (int64_t)0x7fffffff) return DLB_ERR_UNSUPPORTED;
  if (!sorted_ids || !expert_ids || !num_post_pad || (numel > 0 && !topk_ids))
    return DLB_ERR_BAD_ARG;
  if (sorted_cap < numel + (int64_t)E * (block - 1)) return DLB_ERR_BAD_ARG;
  if (expert_ids_cap < ceil_div(sorted_cap, block)) return DLB_ERR_BAD_ARG;
  return DLB_OK;
}

// the launches of the alignment; chunk_counts holds num_chunks(numel) x E int32, every word of
// which the counting pass overwrites before anything reads it (nothing has to start at zero)
int launch_align(const IdxArray topk_ids, int64_t numel, int E, int block, int32_t* sorted_ids,
                 int64_t sorted_cap, int32_t* expert_ids, int64_t expert_ids_cap, int32_t* counts,
                 int32_t* num_post_pad, int32_t* chunk_counts, hipStream_t s,
                 const QuantParams* quant = nullptr, int quant_dtype = DLB_DTYPE_BF16) {
  const AlignOut out = {sorted_ids, sorted_cap, expert_ids, expert_ids_cap, counts, num_post_pad, numel, E, block,
                      reciprocal_of(block)};
  if (numel <= kOneSlots) {
    if (quant && quant->total_groups > 0) {
      const uint32_t grid = (uint32_t)(1 + ceil_div(quant->total_groups, kQuantGroupsPerBlock * kOneQuantBlocks));
      if (quant_dtype == DLB_DTYPE_BF16)
        launch(align_one_quant_kernel<DLB_DTYPE_BF16>, dim3(grid), dim3(kOneThreads), s, out,
                           topk_ids, *quant);
      else
        launch(align_one_quant_kernel<DLB_DTYPE_F16>, dim3(grid), dim3(kOneThreads), s, out,
                           topk_ids, *quant);
    } else {
      launch(align_one_kernel, dim3(1), dim3(kOneThreads), s, out, topk_ids);
    }
    return launch_status();
  }
  const int64_t chunks = num_chunks(numel);
  const int chunk_ids = chunk_ids_for(numel);
  launch(align_count_kernel, dim3((uint32_t)chunks), dim3(kThreads), s, topk_ids,
                     numel, E, chunk_ids, chunk_counts, sorted_ids, sorted_cap);
  if (chunks <= kFusedChunks) {
    const PlaceParams pp = {topk_ids, chunk_counts, (int)chunks, chunk_ids, out};
    if (quant && quant->total_groups > 0) {
      const uint32_t grid = (uint32_t)(chunks + 1 + ceil_div(quant->total_groups, kQuantGroupsPerBlock));
      if (quant_dtype == DLB_DTYPE_BF16)
        launch(align_place_quant_kernel<DLB_DTYPE_BF16>, dim3(grid), dim3(kThreads), s, pp, *quant);
      else
        launch(align_place_quant_kernel<DLB_DTYPE_F16>, dim3(grid), dim3(kThreads), s, pp, *quant);
    } else {
      launch(align_place_fused_kernel, dim3((uint32_t)chunks + 1), dim3(kThreads), s, pp);
    }
    return launch_status();
  }
  if (quant) return DLB_ERR_UNSUPPORTED;  // (the caller launches the quantiser on its own then)
  launch(align_scan_kernel, dim3(1), dim3(kScanThreads), s, chunk_counts, chunks, out);
  launch(align_place_kernel, dim3((uint32_t)chunks), dim3(kThreads), s, topk_ids, numel, E,
                     chunk_counts, sorted_ids);
  return launch_status();
}

// ---- scratch of the entry point that allocates nothing --------------------------------------
// The per-chunk count table of up to kStaticChunks chunks x kMaxE experts (256 KB) lives in a
// file-scope device array: every GPU the library runs on holds one copy of it until the process
// ends.  In host code the array's name is only a handle, not a device address; the address on
// the current device comes from hipGetSymbolAddress, once per device, and is what the kernels
// receive.
constexpr int kStaticChunks = kFusedChunks;
constexpr int kMaxDevices = 64;
static __device__ __align__(256) int32_t scratch[kStaticChunks * kMaxE];

std::mutex scratch_mutex;
int32_t* scratch_ptr[kMaxDevices];  // per device, filled on the first call made on that device

int static_scratch(int32_t** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return DLB_ERR_LAUNCH;
  std::lock_guard<std::mutex> guard(scratch_mutex);
  if (!scratch_ptr[dev]) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) {
      (void)hipGetLastError();
      return DLB_ERR_LAUNCH;
    }
    scratch_ptr[dev] = (int32_t*)ptr;
  }
  *out = scratch_ptr[dev];
  return DLB_OK;
}

}  // namespace
}  // namespace dlb

extern "C" int dlb_moe_align_block_size(const void* topk_ids, int ids_int64, int64_t numel, int E, int block,
                                        int32_t* sorted_ids, int64_t sorted_cap,
                                        int32_t* expert_ids, int64_t expert_ids_cap,
                                        int32_t* counts, int32_t* num_post_pad, void* ws,
                                        size_t ws_bytes, void* stream) {
  using namespace dlb;
  const int st = check_align_args(topk_ids, numel, E, block, sorted_ids, sorted_cap, expert_ids,
                                  expert_ids_cap, num_post_pad);
  if (st != DLB_OK) return st;
  if (!ws || ws_bytes < dlb_moe_align_ws_bytes(numel, E)) return DLB_ERR_WORKSPACE;
  return launch_align(idx_array(topk_ids, ids_int64 ? 1 : 0, 0), numel, E, block, sorted_ids, sorted_cap,
                      expert_ids, expert_ids_cap, counts, num_post_pad, (int32_t*)ws,
                      (hipStream_t)stream);
}

extern "C" int dlb_moe_align_quant_fp8(const void* topk_ids, int ids_int64, int64_t numel, int E, int block,
                                       int32_t* sorted_ids, int64_t sorted_cap,
                                       int32_t* expert_ids, int64_t expert_ids_cap,
                                       int32_t* counts, int32_t* num_post_pad, void* ws,
                                       size_t ws_bytes, const void* x, void* xq, float* xs,
                                       int64_t M, int K, int64_t ld_x, int64_t ld_q, int64_t ld_s,
                                       int dtype, void* stream) {
  using namespace dlb;
  const int st = check_align_args(topk_ids, numel, E, block, sorted_ids, sorted_cap, expert_ids,
                                  expert_ids_cap, num_post_pad);
  if (st != DLB_OK) return st;
  if (!ws || ws_bytes < dlb_moe_align_ws_bytes(numel, E)) return DLB_ERR_WORKSPACE;
  QuantParams q;
  const int sq = fill_quant_params(q, x, xq, xs, M, K, ld_x, ld_q, ld_s, dtype);
  if (sq != DLB_OK) return sq;
  const IdxArray ids = idx_array(topk_ids, ids_int64 ? 1 : 0, 0);
  if (num_chunks(numel) <= kFusedChunks)
    return launch_align(ids, numel, E, block, sorted_ids, sorted_cap, expert_ids,
                        expert_ids_cap, counts, num_post_pad, (int32_t*)ws, (hipStream_t)stream, &q,
                        dtype);
  // more routing slots than the fused placement takes: the separate launches
  const int sa = launch_align(ids, numel, E, block, sorted_ids, sorted_cap, expert_ids,
                              expert_ids_cap, counts, num_post_pad, (int32_t*)ws, (hipStream_t)stream);
  if (sa != DLB_OK) return sa;
  return dlb_per_token_group_quant_fp8(x, xq, xs, M, K, ld_x, ld_q, ld_s, dtype, stream);
}

extern "C" int64_t dlb_moe_align_block_size_static_max_numel(void) {
  return (int64_t)dlb::kStaticChunks * dlb::kChunk;  // = kFusedChunks chunks of the largest size
}

extern "C" int dlb_moe_align_block_size_static(const void* topk_ids, int ids_int64, int64_t numel,
                                               int E, int block, int32_t* sorted_ids, int64_t sorted_cap,
                                               int32_t* expert_ids, int64_t expert_ids_cap,
                                               int32_t* counts, int32_t* num_post_pad,
                                               void* stream) {
  using namespace dlb;
  const int st = check_align_args(topk_ids, numel, E, block, sorted_ids, sorted_cap, expert_ids,
                                  expert_ids_cap, num_post_pad);
  if (st != DLB_OK) return st;
  // the static table holds kStaticChunks chunks: larger inputs must bring their own workspace
  if (numel > dlb_moe_align_block_size_static_max_numel()) return DLB_ERR_WORKSPACE;
  int32_t* chunk_counts = nullptr;
  const int sp = static_scratch(&chunk_counts);
  if (sp != DLB_OK) return sp;
  return launch_align(idx_array(topk_ids, ids_int64 ? 1 : 0, 0), numel, E, block, sorted_ids, sorted_cap,
                      expert_ids, expert_ids_cap, counts, num_post_pad, chunk_counts,
                      (hipStream_t)stream);
}

// ---------------------------------------------------------------------------------------
// Router and alignment as one pipeline: one workgroup up to one_workgroup_tokens, else the router with
// per-chunk expert counts (a chunk = the K routing slots of route_chunk_tokens consecutive
// tokens) and the placement.
// ---------------------------------------------------------------------------------------
namespace dlb {
namespace {

// Tokens per workgroup of the router.  Its arg-max rounds keep the SIMDs busy, so the fewer tokens a CU has the
// better, but every placing workgroup reduces the whole count table: 16 tokens while it reads that at once, 32
// while the table stays within kFusedChunks rows, as 64 (one pass) after that, else 128 (two passes).  64 / 32 / 16
// tokens, us in fp32: 256 experts, 8 each, 1024 tokens 14.9 / 10.9 / 10.2, 4096 15.4 / 12.3 / 13.7; 128 experts,
// 2048 tokens 11.1 / 8.9 / 8.7, 4096 11.4 / 9.3 / 9.9; 64 experts, 6 each, 200 tokens 8.5 / 7.4 / 7.3, 4096 9.1 / 7.9 /
// 7.9, 6000 9.1 / 8.0.
int route_chunk_tokens(int64_t T, int E) {
  const int at_once = 16 * kThreads / (E <= 64 ? 16 : E <= 128 ? 32 : 64);
  if (ceil_div(T, 16) <= at_once) return 16;
  for (int tokens = 32; tokens < 128; tokens *= 2)
    if (ceil_div(T, tokens) <= kFusedChunks) return tokens;
  return 128;
}
size_t route_ws_bytes(int64_t T, int E, int chunk_tokens) {
  return (size_t)(T > 0 ? ceil_div(T, chunk_tokens) : 1) * (size_t)((E + 3) / 4) * sizeof(uint32_t);
}

template <int VPL, int LT>
void launch_route_align(const RouteParams& p, const AlignOut& o, uint32_t* table, int chunk_tokens, hipStream_t s) {
  if (p.T <= one_workgroup_tokens(VPL)) {
    launch((route_align_one_kernel<VPL, LT>), dim3(1), dim3(kOneThreads), s, p, o);
    return;
  }
  const int chunks = (int)ceil_div(p.T, chunk_tokens);
  if (chunk_tokens == 16)
    launch((route_count_kernel<VPL, 256, 1, LT>), dim3(chunks), dim3(256), s, p, o, table);
  else if (chunk_tokens == 32)
    launch((route_count_kernel<VPL, 512, 1, LT>), dim3(chunks), dim3(512), s, p, o, table);
  else if (chunk_tokens == 64)
    launch((route_count_kernel<VPL, 1024, 1, LT>), dim3(chunks), dim3(1024), s, p, o, table);
  else
    launch((route_count_kernel<VPL, 1024, 2, LT>), dim3(chunks), dim3(1024), s, p, o, table);
  launch(route_place_kernel, dim3(chunks), dim3(kThreads), s, IdxArray{p.ids, 0}, o, table, chunks,
                     chunk_tokens * p.K);
}

}  // namespace
}  // namespace dlb

extern "C" size_t dlb_moe_topk_softmax_align_ws_bytes(int64_t T, int E) {
  if (T < 0 || E < 1) return 0;
  return dlb::route_ws_bytes(T, E, dlb::route_chunk_tokens(T, E));
}

extern "C" int dlb_moe_topk_softmax_align_f32(const void* logits, float* weights, int32_t* ids,
                                              int64_t T, int E, int K, int64_t ld_logits,
                                              int logits_dtype, int renormalize, int block,
                                              int32_t* sorted_ids,
                                              int64_t sorted_cap, int32_t* expert_ids,
                                              int64_t expert_ids_cap, int32_t* counts,
                                              int32_t* num_post_pad, void* ws, size_t ws_bytes,
                                              void* stream) {
  using namespace dlb;
  if (T < 0 || E < 1 || K < 1 || K > E || ld_logits < E || block < 1) return DLB_ERR_BAD_ARG;
  if (K > 16 || E > kMaxE) return DLB_ERR_UNSUPPORTED;
  if (logits_dtype != DLB_DTYPE_F32 && logits_dtype != DLB_DTYPE_BF16 && logits_dtype != DLB_DTYPE_F16)
    return DLB_ERR_UNSUPPORTED;
  const int64_t numel = T * K;
  if (numel + (int64_t)E * block >= (int64_t)0x7fffffff) return DLB_ERR_UNSUPPORTED;
  // larger inputs take the two separate entry points (their scan runs as its own launch)
  int chunk_tokens = route_chunk_tokens(T, E);
  if (T > (int64_t)kFusedChunks * chunk_tokens) return DLB_ERR_UNSUPPORTED;
  // (a scratch for chunks of 64 tokens is enough)
  while (chunk_tokens < 64 && ws_bytes < route_ws_bytes(T, E, chunk_tokens)) chunk_tokens *= 2;
  if (!sorted_ids || !expert_ids || !num_post_pad || (T > 0 && (!logits || !weights || !ids)))
    return DLB_ERR_BAD_ARG;
  if (sorted_cap < numel + (int64_t)E * (block - 1)) return DLB_ERR_BAD_ARG;
  if (expert_ids_cap < ceil_div(sorted_cap, block)) return DLB_ERR_BAD_ARG;
  if (!ws || ws_bytes < route_ws_bytes(T, E, chunk_tokens)) return DLB_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  const RouteParams p = {logits, weights, ids, T, E, K, ld_logits, renormalize,
                         (int)(logits_vector_ok(logits, logits_dtype, ld_logits) && (E == 64 || E == 128 || E == 256))};
  const AlignOut o = {sorted_ids, sorted_cap, expert_ids, expert_ids_cap, counts, num_post_pad, numel, E, block,
                      reciprocal_of(block)};
  uint32_t* table = (uint32_t*)ws;
#define DLB_LAUNCH_ROUTE_ALIGN(VPL_)                                                                   \
  do {                                                                                                 \
    if (logits_dtype == DLB_DTYPE_F32) launch_route_align<VPL_, DLB_DTYPE_F32>(p, o, table, chunk_tokens, s);        \
    else if (logits_dtype == DLB_DTYPE_BF16) launch_route_align<VPL_, DLB_DTYPE_BF16>(p, o, table, chunk_tokens, s); \
    else launch_route_align<VPL_, DLB_DTYPE_F16>(p, o, table, chunk_tokens, s);                                      \
  } while (0)
  if (E <= 64) DLB_LAUNCH_ROUTE_ALIGN(4);
  else if (E <= 128) DLB_LAUNCH_ROUTE_ALIGN(8);
  else DLB_LAUNCH_ROUTE_ALIGN(16);
#undef DLB_LAUNCH_ROUTE_ALIGN
  return launch_status();
}
