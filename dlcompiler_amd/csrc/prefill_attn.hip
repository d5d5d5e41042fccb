// Varlen causal flash-attention prefill for gfx950 (packed [tokens, heads, D] layout, GQA).
//
// Replaces context_attention_fwd + _fwd_kernel
// (python/dlBLAS/dlblas/kernels/prefill_attention.py:39-181): same mathematics -- per
// (sequence, query head, query tile) stream the causal prefix of K/V, QK^T in fp32, online
// softmax, P rounded to the input dtype before P.V -- re-tiled for CDNA4:
//   * a workgroup of 4 wavefronts owns 128 query rows (32 per wave) and walks 64-key K/V tiles
//     that are double-buffered in LDS (copied global -> LDS directly, one barrier per tile);
//   * S^T = K.Q^T and O^T = V^T.P^T on 32x32x16 MFMA.  Working on the transposes puts a query
//     in a lane *column*: the row max/sum are register reductions plus one exchange between
//     the two lane halves, the rescale is a per-lane scalar, and the softmax output registers
//     are already the B operand of the second product (P never crosses lanes): the V^T
//     operand is simply fetched in the key order those registers have;
//   * K and V both sit row-major in LDS.  K fragments are 128-bit reads; V^T fragments come
//     from ds_read_b64_tr_b16, which hands lane l of a 16-lane group column l of a 4-row x
//     16-column block (rows supplied by lanes 4j .. 4j+3), i.e. the transpose happens in the
//     LDS read and V never passes through registers on its way in;
//   * the exponent runs in base 2 with the softmax scale folded into one FMA;
//   * fully masked tiles are skipped per wave and only diagonal tiles pay for the mask; the
//     heaviest query tiles are launched first.
#include <cmath>
#include <type_traits>

#include "common.h"

namespace dlb {
namespace {

struct PrefillParams {
  const void* q;
  const void* k;
  const void* v;
  void* o;
  IdxArray start_loc;
  IdxArray seq_len;
  int64_t q_st, q_sh, k_st, k_sh, v_st, v_sh, o_st, o_sh;  // token / head strides (elements)
  int Hq, Hkv, group;
  int xcd_heads;  // heads (head groups) per XCD, != 0: remap blockIdx.x so a KV group's share an XCD
  // PACK kernels: a workgroup's rows are those of 1 << pack_shift query heads of a KV group, the rows of
  // each being (kBlockM >> pack_shift) queries
  int pack_shift;
  // nsplit > 1: the key tiles of a row tile may be shared out among up to nsplit workgroups, see
  // tiles_per_part, which leave unnormalised rows in ws_o [nsplit][tokens][Hq][ws_d] and (maximum,
  // denominator) in ws_ml [nsplit][tokens][Hq][2]
  int nsplit, ws_d;
  int B;  // sequences
  int64_t tokens;
  float* ws_o;
  float* ws_ml;
  float scale_log2e;
  // paged K/V (PAGED kernels): k/v point at caches [pages, page, Hkv, D]; *_st is the slot
  // stride, *_sp the page stride; sequence s reads pages block_table[s][.] and its queries sit
  // at context positions kv_len[s] - seq_len[s] + i
  IdxArray kv_len;
  IdxArray block_table;
  int64_t bt_stride, k_sp, v_sp;
  int page, page_shift;
  int dk, dv;  // real key / value head sizes (<= the padded size D the kernel is built for)
  // generic masking (both layouts): sliding window (> 0) and logit soft-cap (> 0)
  int window;
  float softcap, sm_scale;
  unsigned int share_rcp;  // SHARE kernels: a block's number in their order times this is its quotient by the heads
};

template <int DT>
struct Mma32;
template <>
struct Mma32<DLB_DTYPE_BF16> {
  static __device__ __forceinline__ f32x16 run(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ unsigned int pack2(float a, float b) {
    typedef __attribute__((ext_vector_type(2))) float f2;
    typedef __attribute__((ext_vector_type(2))) __bf16 b2;
    f2 f = {a, b};
    return __builtin_bit_cast(unsigned int, __builtin_convertvector(f, b2));
  }
};
template <>
struct Mma32<DLB_DTYPE_F16> {
  static __device__ __forceinline__ f32x16 run(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ unsigned int pack2(float a, float b) {
    typedef __attribute__((ext_vector_type(2))) float f2;
    typedef __attribute__((ext_vector_type(2))) _Float16 h2;
    f2 f = {a, b};
    return __builtin_bit_cast(unsigned int, __builtin_convertvector(f, h2));
  }
};

constexpr int kThreads = 256;
constexpr int kTileN = 64;    // keys per LDS tile
constexpr int kPartTiles = 8;  // ... per part of a split row tile, at least

// key tiles [first, end) that hold a key visible to one of the `rows` queries from q0 on
struct TileRun {
  int first, end;
};
__device__ __forceinline__ TileRun visible_tiles(int kv_total, int hist, int q0, int rows, int window) {
  return TileRun{window > 0 ? max(hist + q0 - window, 0) / kTileN : 0,
                 (min(kv_total, hist + q0 + rows) + kTileN - 1) / kTileN};
}
// Key tiles of a part.  The launch is cut for the longest context that the block table has room for, and
// engines keep tables of a fixed width; how many parts there are follows from the context itself.
// Parts past the last tile have no work, and where there is one part it writes the output itself.
// 32 heads (8 kv) of 128, a table of 512 pages of 64: 32 queries over 100 keys 36.1 -> 11.4 us, over 1000
// 42 -> 19, over 4000 58.8 -> 20.4; 4 x 100 over 600 27.2 -> 21.7 (in a table without room: 6.7, 15.9, 20.3, 14.6).
__device__ __forceinline__ int tiles_per_part(const TileRun& run, int nsplit) {
  const int tiles = run.end - run.first, parts = min(max(tiles / kPartTiles, 1), nsplit);
  return (tiles + parts - 1) / parts;
}

// ... and the most parts that a row tile of a sequence with kv_total keys has
__device__ __forceinline__ int most_parts(int kv_total, const PrefillParams& p) {
  int tiles = (kv_total + kTileN - 1) / kTileN;
  if (p.window > 0 && p.window < kv_total) tiles = min(tiles, (p.window + (128 >> p.pack_shift)) / kTileN + 2);
  return min(max(tiles / kPartTiles, 1), p.nsplit);
}

template <int D>
struct Smem {
  static constexpr int kRowBytes = D * 2;           // K: [64][D], 16-byte chunks XOR-swizzled
  static constexpr int kBytes = kTileN * kRowBytes;
  static constexpr int vBytes = kBytes;              // V: [64][D], 16-byte chunks XOR-swizzled
  static constexpr int stage = kBytes + vBytes;
};

// D is the padded head size the kernel is built for (64, 96, 128 or 256).  RAGGED: the real key size dk
// and / or value size dv is smaller (any multiple of 8): the query dims past dk are loaded as
// zeros, so the key bytes staged for those dims do not count -- their copies are redirected to
// the row's first 16 bytes to stay inside the tensor -- and value dims past dv (redirected
// likewise) only produce output dims that are never stored.  The reference handles odd head
// sizes by splitting them into power-of-two blocks with masked loads
// (python/dlBLAS/dlblas/kernels/paged_attention.py:531-539).
// PAGED: 0 = packed K/V; 1 = paged, every K/V row looks up its own page (any page size); 2 = paged
// with pages that are whole multiples of the 64-key tile: a tile lies in one page, so its page
// number is one wave-uniform look-up and the copies are addressed as in the packed layout (a
// scalar base per tile plus constant lane offsets).
// RW: row waves, KG = 4 / RW key groups of a workgroup's four waves.  RW = 4: 128 query rows.  RW = 2: 64
// rows, and two pairs of waves that work on every second key tile each, with LDS buffers of their
// own; their partial results meet in LDS at the end.  A wave keeps its SIMD busy by itself, so a
// launch with fewer 128-row workgroups than CUs is as fast as one workgroup's chain of tiles: this
// shape gives it twice the workgroups and half the chain (one sequence of 512 tokens, 32 heads of
// 128: 13.6 -> 11.2 us, of 1125 tokens, 8 heads: 21.7 -> 16.0; eight waves on 128 rows: 13.6 and 19.5).
// PACK: short query runs over a history (every run fits a fraction of the rows): the heads of a KV
// group share a workgroup, so the rows are filled and K/V is staged once for all of them; and the
// key tiles may be split over workgroups.
template <int DT, int D, int PAGED, bool RAGGED, int RW, bool PACK, bool SHARE = false>
__global__ __launch_bounds__(kThreads, D > 128 ? 1 : RW == 2 ? 1 : 2) void prefill_attn_kernel(const PrefillParams p) {
  constexpr int KG = 4 / RW;
  constexpr int kBlockM = 32 * RW;  // query rows per workgroup
  constexpr int KS = D / 16;  // MFMA k-steps over the head dim for S^T
  constexpr int MT = D / 32;  // 32-row tiles of O^T
  constexpr int DG = D / 8;
  using SM = Smem<D>;

  __shared__ __attribute__((aligned(16))) unsigned char smem_all[KG * 2 * SM::stage];

  // The grid runs over (head, query tile, sequence), tile index reversed: what an XCD holds at
  // any time is the query tiles of ONE sequence's heads of ONE KV group (see the head remap
  // below), i.e. workgroups that stream the same K/V rows, which its L2 then serves after the
  // first read; within a sequence the heaviest (last) tiles start first.
  // Paged (chunked) prefill: a sequence's cost is set by its history, which differs widely
  // between the sequences of a batch while the grid holds only a few workgroups per slot, so
  // the sequences are walked longest context first (blockIdx.z = rank, not index): the long
  // ones start in the first round and the short ones fill in behind them.  (The packed layout
  // has many workgroups per slot and gains nothing from the ranking: measured 1.5 % slower.)
  // Where key tiles are split, blockIdx.z counts the parts of one sequence after the other, in the same
  // order; indexes past the last part have no work (the grid has room for nsplit parts of each).
  const int nb = PACK ? p.B : gridDim.z;
  const bool parts_too = PACK && p.nsplit > 1;
  int seq = blockIdx.z, split = 0;
  if (PACK && (nb == 1 || nb > kThreads)) {
    split = nb == 1 ? seq : seq / nb;
    seq -= split * nb;
    if (nb == 1) seq = 0;
  }
  if (PAGED && nb > 1 && nb <= kThreads) {
    __shared__ int32_t rank_key[kThreads];
    __shared__ int32_t rank_parts[PACK ? kThreads : 1];
    __shared__ int32_t rank_seq, rank_split;
    const int t = threadIdx.x;
    const int key = t < nb ? p.kv_len[t] : 0;
    int parts = 1;
    if (parts_too) {
      parts = most_parts(key, p);
      rank_parts[t] = parts;
      if (t == 0) rank_seq = -1;
    }
    rank_key[t] = key;
    __syncthreads();
    if (t < nb) {
      int rank = 0;  // parts_too: in parts
      for (int j = 0; j < nb; ++j) {
        const int kj = rank_key[j];
        rank += (kj > key || (kj == key && j < t)) ? (parts_too ? rank_parts[j] : 1) : 0;
      }
      const int mine = (int)blockIdx.z - rank;
      if (mine >= 0 && mine < parts) {  // exactly one writer, or none
        rank_seq = t;
        rank_split = mine;
      }
    }
    __syncthreads();
    seq = __builtin_amdgcn_readfirstlane(rank_seq);
    if (parts_too) {
      if (seq < 0) return;
      split = __builtin_amdgcn_readfirstlane(rank_split);
    }
  }
  // (vector loads of wave-uniform values: saying that they are keeps loops and conditions scalar)
  const int L = __builtin_amdgcn_readfirstlane(p.seq_len[seq]);
  const int pack = PACK ? p.pack_shift : 0;
  const int qtile = gridDim.y - 1 - blockIdx.y;  // heaviest first
  // SHARE: a wave's rows are 32 queries of one head, and a workgroup takes the next four of the order
  // (query block, head) of a KV group: with the heads of a KV group in that order its waves see the same keys, where those
  // of 128 queries of one head reach the diagonal one after the other, and only a sequence's last workgroup
  // has waves without rows.
  static_assert(!SHARE || (RW == 4 && !PACK), "");
  int q0 = qtile * (kBlockM >> pack), span = kBlockM >> pack;  // queries of the workgroup: first, how many
  int wave_q0 = 0, wave_head = 0;                              // of the wave: offset of its first query, head
  int block_head = 0;                                          // head of the workgroup's first wave
  if (SHARE) {
    const int unit0 = qtile * RW;
    const int first = (int)__umulhi((unsigned)unit0, p.share_rcp);
    q0 = 32 * first;
    block_head = unit0 - first * p.group;
  }
  if (q0 >= L) return;
  if (SHARE) {
    auto block_of = [&](int w, int& dq, int& hd) {
      dq = 0;
      hd = block_head + w;
#pragma unroll
      for (int i = 1; i < RW; ++i)
        if (hd >= p.group) {
          hd -= p.group;
          dq += 32;
        }
    };
    int last_head;
    block_of(RW - 1, span, last_head);
    span += 32;
    block_of(threadIdx.x >> 6, wave_q0, wave_head);
  }
  const int64_t tok0 = __builtin_amdgcn_readfirstlane(p.start_loc[seq]);
  // context seen by this sequence: kv_total keys, the queries are its last L positions
  const int kv_total = PAGED ? __builtin_amdgcn_readfirstlane(p.kv_len[seq]) : L;
  const int hist = kv_total - L;
  if (PAGED && hist < 0) return;  // inconsistent lengths: nothing sensible to compute
  // sliding window (only the paged entry point exposes it; the packed kernel compiles it out)
  const int window = PAGED ? p.window : -1;
  TileRun run = visible_tiles(kv_total, hist, q0, span, window);
  bool parted = false;  // other workgroups have a part of these rows' keys
  if (PACK && p.nsplit > 1) {
    const int per = tiles_per_part(run, p.nsplit);
    parted = run.end - run.first > per;
    run.first += split * per;
    if (run.first >= run.end) return;
    run.end = min(run.end, run.first + per);
  }
  int head = blockIdx.x;  // PACK: first of the workgroup's heads
  if (p.xcd_heads) head = (blockIdx.x & 7) * p.xcd_heads + (blockIdx.x >> 3);
  if (PACK) head <<= pack;
  else if (SHARE) head *= p.group;
  const int kvh = head / p.group;

  const int tid = threadIdx.x;
  const int grp = KG > 1 ? __builtin_amdgcn_readfirstlane((tid >> 6) / RW) : 0;
  const int wave = (tid >> 6) % RW;  // row wave
  const int lane = tid & 63;
  unsigned char* const smem = smem_all + grp * (2 * SM::stage);
  const int col = lane & 31;  // query column / operand row
  const int hh = lane >> 5;   // lane half

  const unsigned short* qb = (const unsigned short*)p.q;
  const unsigned short* kb = (const unsigned short*)p.k + (int64_t)kvh * p.k_sh;
  const unsigned short* vb = (const unsigned short*)p.v + (int64_t)kvh * p.v_sh;

  // ---- Q^T as B operand: lane (n = query, k = dims 16*ks + 8*hh .. +8), kept in registers
  const int brow = 32 * wave + col;  // row of the workgroup
  const int qrow = q0 + (SHARE ? wave_q0 + col : PACK ? brow & (span - 1) : brow);
  if (SHARE) head += __builtin_amdgcn_readfirstlane(wave_head);
  if (PACK) head += brow / span;  // (by lane from here on)
  u32x4 qf[KS];
  {
    const unsigned short* qp =
        qb + (tok0 + min(qrow, L - 1)) * p.q_st + (int64_t)head * p.q_sh + 8 * hh;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      qf[ks] = u32x4{0u, 0u, 0u, 0u};
      if (!RAGGED || 16 * ks + 8 * hh < p.dk) qf[ks] = *(const u32x4*)(qp + 16 * ks);
    }
  }

  const int jfirst = run.first, ntiles = run.end;
  // (a soft-cap takes the masked path for every tile; only the paged entry point exposes it)
  const float softcap = PAGED ? p.softcap : -1.0f;
  // tiles below this index lie entirely under the diagonal for every wave of the workgroup
  // (all 64 keys <= position of row q0): no mask, no clamping of key rows
  const int nfull = softcap > 0.0f ? 0 : min((hist + q0 + 1) / kTileN, ntiles);
  // first tile whose keys every query of the workgroup sees (sliding window)
  const int jopen = window > 0 ? max(hist + q0 + span - 1 - window + kTileN - 1, 0) / kTileN : 0;
  const int qpos = hist + qrow;                          // context position of this lane's query
  // context positions of the wave's first and last query
  if (!SHARE) wave_q0 = PACK ? (32 * wave) & (span - 1) : 32 * wave;
  const int wave_first_pos = hist + q0 + wave_q0;
  const int wave_last_pos = wave_first_pos + (PACK ? min(32, span) : 32) - 1;

  // ---- global -> LDS staging of one K/V tile.  Per-thread base pointers are formed once; a
  // tile adds a workgroup-uniform offset.  CLAMP (tiles that may run past the sequence)
  // redirects rows >= kv_total to the last row so nothing outside the sequence is read.
  // Both operands go global -> LDS directly (global_load_lds_dwordx4: lane l's 16 bytes land
  // at base + 16*l, so one wave instruction fills 1 KB = 1024 / (2*D) rows).  Rows are stored
  // unpadded; bank conflicts are avoided by permuting which 16-byte chunk of its row a lane
  // fetches: position c of row r holds chunk c ^ swz(r), so a reader that wants chunk c of
  // row r reads position c ^ swz(r).  K: swz(r) = r mod DG (128-bit fragment reads, one row
  // per lane).  V: swz(r) spreads the 4 (or 8) rows that one transposing read touches over
  // all banks.
  constexpr int KINS = kTileN * DG / (64 * RW);  // instructions per wave, tile and operand
  // copy i of a wave brings the tile's 16-byte pieces 64 * (RW i + wave) + lane, counted row by row
  auto copy_row = [&](int i) -> int { return ((RW * i + wave) * 64 + lane) / DG; };
  auto copy_pos = [&](int i) -> int { return ((RW * i + wave) * 64 + lane) % DG; };
  const unsigned char* kbytes = (const unsigned char*)kb;
  const unsigned char* vbytes = (const unsigned char*)vb;
  const int64_t k_row_bytes = p.k_st * 2, v_row_bytes = p.v_st * 2;
  const IdxArray bt = {PAGED ? p.block_table.p + (((int64_t)seq * p.bt_stride) << p.block_table.sh) : nullptr,
                       p.block_table.sh};
  // K chunk swizzle of row r.  (Rows of 96 elements start 48 banks apart: four rows fill all 64
  // banks, the swizzle separates the four groups of four that a fragment read touches.)
  auto k_swz = [](int r) -> int { return D == 96 ? (r >> 2) & 3 : r & (DG - 1); };
  // V chunk swizzle of row r (depends on r mod 8 only)
  auto v_swz = [](int r) -> int {
    if (D == 96) return 0;
    return D == 128 ? (((r & 3) << 2) | (((r >> 2) & 1) << 1))
                    : ((((r >> 1) & 1) << 2) | (((r >> 2) & 1) << 1));
  };
  // byte offset inside its source row of the 16-byte chunk that copy i of this lane brings (the
  // swizzle undone; chunks past the real head size fetch the row's first chunk)
  auto k_chunk = [&](int i) -> unsigned int {
    const int c = copy_pos(i) ^ k_swz(copy_row(i));
    return (unsigned int)((RAGGED && 8 * c >= p.dk) ? 0 : c) << 4;
  };
  auto v_chunk = [&](int i) -> unsigned int {
    const int c = copy_pos(i) ^ v_swz(copy_row(i));
    return (unsigned int)((RAGGED && 8 * c >= p.dv) ? 0 : c) << 4;
  };
  // paged layout: the page ids of the rows this lane copies are fetched one tile ahead of the
  // copy that needs them, so the block-table latency never sits in front of a tile's copies
  int pg_next[KINS];
  int pg_tile = 0;  // PAGED == 2: the page of the next tile to stage (wave-uniform)
  auto fetch_pages = [&](int t0) {
    if (PAGED == 2) {
      const int key = min(t0, kv_total - 1);
      pg_tile = bt[p.page_shift >= 0 ? (key >> p.page_shift) : (key / p.page)];
      return;
    }
#pragma unroll
    for (int i = 0; i < KINS; ++i) {
      const int key = min(t0 + copy_row(i), kv_total - 1);
      pg_next[i] = bt[p.page_shift >= 0 ? (key >> p.page_shift) : (key / p.page)];
    }
  };
  const unsigned int smem_base = lds_addr(smem_all) + grp * (2 * SM::stage) + wave * 1024;  // + q * 1024 with q = RW*i + wave
  // source addresses and LDS targets of the copies of the tile being staged: prepare_tile
  // computes them, issue_copy(n) sends copy n of 2 * KINS (K and V slices alternate)
  // Packed layout: a copy's address is a tile base in scalar registers plus a 32-bit lane
  // offset that does not change from tile to tile (row inside the tile x row pitch + chunk),
  // so an unclamped tile costs no vector arithmetic.  Paged layout: every row has its own
  // page, so full 64-bit lane addresses are formed.
  const unsigned char* ksrc[KINS];
  const unsigned char* vsrc[KINS];
  unsigned int koff[KINS], voff[KINS], koff0[KINS], voff0[KINS];
  const unsigned char* kbase = nullptr;
  const unsigned char* vbase = nullptr;
#pragma unroll
  for (int i = 0; i < KINS; ++i) {
    koff0[i] = (unsigned int)(copy_row(i) * k_row_bytes) + k_chunk(i);
    voff0[i] = (unsigned int)(copy_row(i) * v_row_bytes) + v_chunk(i);
  }
  unsigned int stage_dst = 0;
  auto prepare_tile = [&](auto clamp_tag, int t0, int buf) {
    constexpr bool CLAMP = decltype(clamp_tag)::value;
    stage_dst = smem_base + buf * SM::stage;
    if (!PAGED) {
      kbase = uniform_ptr(kbytes + (tok0 + t0) * k_row_bytes);
      vbase = uniform_ptr(vbytes + (tok0 + t0) * v_row_bytes);
    }
    if (PAGED == 2) {
      // t0 is a multiple of the tile and the page a multiple of the tile: slot of the tile's
      // first key inside its page (a tile whose first key lies past the context is never staged)
      const int pi = p.page_shift >= 0 ? (t0 >> p.page_shift) : (t0 / p.page);
      const int64_t pg = __builtin_amdgcn_readfirstlane(pg_tile);
      const int64_t slot0 = t0 - pi * p.page;
      kbase = uniform_ptr(kbytes + (pg * p.k_sp + slot0 * p.k_st) * 2);
      vbase = uniform_ptr(vbytes + (pg * p.v_sp + slot0 * p.v_st) * 2);
    }
#pragma unroll
    for (int i = 0; i < KINS; ++i) {
      const int r = copy_row(i);  // key row inside the tile
      if (PAGED == 1) {
        int key = t0 + r;
        if (CLAMP) key = min(key, kv_total - 1);
        const int pi = p.page_shift >= 0 ? (key >> p.page_shift) : (key / p.page);
        const int64_t slot = key - pi * p.page;
        ksrc[i] = kbytes + ((int64_t)pg_next[i] * p.k_sp + slot * p.k_st) * 2 + k_chunk(i);
        vsrc[i] = vbytes + ((int64_t)pg_next[i] * p.v_sp + slot * p.v_st) * 2 + v_chunk(i);
      } else if (CLAMP) {
        const int rc = min(r, kv_total - 1 - t0);  // >= 0: a staged tile starts inside the context
        koff[i] = (unsigned int)(rc * k_row_bytes) + k_chunk(i);
        voff[i] = (unsigned int)(rc * v_row_bytes) + v_chunk(i);
      } else {
        koff[i] = koff0[i];
        voff[i] = voff0[i];
      }
    }
    if (PAGED) fetch_pages(t0 + KG * kTileN);  // consumed by the next prepare_tile
  };
  auto issue_copy = [&](int n) {
    const int i = n >> 1;  // 1 KB slice RW*i + wave of the tile
    const unsigned int dst = stage_dst + (n & 1) * SM::kBytes + i * (RW * 1024);
    if (PAGED == 1) dma16_global_to_lds((n & 1) ? vsrc[i] : ksrc[i], dst);
    else if (n & 1) dma16_global_to_lds(vbase, voff[i], dst);
    else dma16_global_to_lds(kbase, koff[i], dst);
  };
  auto load_tile = [&](auto clamp_tag, int t0, int buf) {
    prepare_tile(clamp_tag, t0, buf);
#pragma unroll
    for (int n = 0; n < 2 * KINS; ++n) issue_copy(n);
  };

  f32x16 o[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[mt][i] = 0.0f;
  // m_run is the exponent reference in the log2 domain.  It follows the running maximum
  // lazily: the accumulators are rescaled only when a row maximum exceeds it by more than
  // kRescaleGap, so between rescales probabilities stay below 2^kRescaleGap -- exact in the
  // end (the same factor cancels in O / l), and it removes the per-tile rescale of O.
  constexpr float kRescaleGap = 8.0f;
  float m_run = -__builtin_inff();
  float l_run = 0.0f;  // this lane half's share of the denominator
  const float cs = p.scale_log2e;

  // byte offsets of this lane's transposing V reads inside a tile, one per 32-dim block
  int v_off[MT];
  {
    const int s16 = lane & 15, dhalf = (lane >> 4) & 1;
    const int r = 4 * hh + (s16 >> 2);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      v_off[mt] = r * SM::kRowBytes +
                  (((4 * mt + 2 * dhalf + ((s16 >> 1) & 1)) ^ v_swz(r)) << 4) + 8 * (s16 & 1);
  }

  // one K/V tile against this wave's 32 queries; MASK: apply the causal mask
  // COPY: the copies of the tile prepared by prepare_tile go out between the S^T MFMAs, one or two
  // per k-step, instead of as one burst that would hold up this wave's instruction stream
  auto process_tile = [&](auto mask_tag, auto copy_tag, int j, int buf) __attribute__((always_inline)) {
    constexpr bool MASK = decltype(mask_tag)::value;
    constexpr bool COPY = decltype(copy_tag)::value;
    constexpr int kCopies = 2 * KINS / KS;  // per k-step
    static_assert(kCopies * KS == 2 * KINS, "whole copies per k-step");
    const int t0 = j * kTileN;
    if (MASK && t0 > wave_last_pos) return;  // wave-uniform: tile entirely above the diagonal
    if (MASK && window > 0 && t0 + kTileN - 1 < wave_first_pos - window) return;  // below the window
    const unsigned char* ks = smem + buf * SM::stage;
    const unsigned char* vs = ks + SM::kBytes;

    // ---- S^T = K . Q^T : two 32-key tiles x 32 queries (raw scores)
    // k-step outer, key tile inner: two independent accumulator chains, and the K fragments
    // are fetched from LDS two k-steps ahead of the MFMAs that consume them
    f32x16 s[2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[nt][i] = 0.0f;
    // MFMA-dense phase: let this wave's issue win over the other wave of the SIMD, whose
    // softmax arithmetic then fills the gaps while the matrix pipe is busy
    __builtin_amdgcn_s_setprio(1);
    {
      const unsigned char* krow0 = ks + col * SM::kRowBytes;
      const unsigned char* krow1 = ks + (32 + col) * SM::kRowBytes;
      const int ksw = k_swz(col);  // (row 32 + col has the same)
      auto ldk = [&](int kstep, u32x4 (&a)[2]) {
        const int off = ((2 * kstep + hh) ^ ksw) << 4;
        a[0] = *(const u32x4*)(krow0 + off);
        a[1] = *(const u32x4*)(krow1 + off);
      };
      constexpr int kAhead = 2;
      u32x4 ka[kAhead + 1][2];
#pragma unroll
      for (int q = 0; q < kAhead; ++q) ldk(q, ka[q]);
#pragma unroll
      for (int kstep = 0; kstep < KS; ++kstep) {
        if (kstep + kAhead < KS) ldk(kstep + kAhead, ka[(kstep + kAhead) % (kAhead + 1)]);
        if (COPY) {
#pragma unroll
          for (int n = 0; n < kCopies; ++n) issue_copy(kCopies * kstep + n);
        }
        __builtin_amdgcn_sched_barrier(0);  // keep the fetch ahead of the MFMAs (it would be sunk)
        s[0] = Mma32<DT>::run(ka[kstep % (kAhead + 1)][0], qf[kstep], s[0]);
        s[1] = Mma32<DT>::run(ka[kstep % (kAhead + 1)][1], qf[kstep], s[1]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }

    __builtin_amdgcn_s_setprio(0);
    // ---- causal mask and tile maximum of the raw scores (scale > 0 commutes with max)
    // (opaque: a condition on a value the compiler knows to be constant in the loop makes it split the
    // loop by it, and the copies' accumulators do not share registers)
    float cap = softcap;
    if (MASK && PAGED) asm volatile("" : "+s"(cap));
    if (MASK && cap > 0.0f) {  // cap * tanh(x * scale / cap), kept in raw-score units
      const float to_arg = p.sm_scale / cap, to_score = cap / p.sm_scale;
      float top = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) top = fmaxf(top, fmaxf(fabsf(s[0][i]), fabsf(s[1][i])));
      // Mostly none of the wave's scores comes near the cap, and the polynomial is all there is: 8 x 512
      // tokens over 4096, 645 -> 497 us; where some do in every tile the look costs nothing (646).
      if (__any(top * to_arg >= kSoftcapSmall)) {
        // (a factor of its own: with the same one in both branches the compiler moves the polynomial in front
        // of them, 32 more registers live, and calls of 64 dims without a cap lost a third of their waves:
        // 64 heads, 8 x 66 - 134 tokens over 48, 14.9 us instead of 13.7)
        float arg = to_arg;
        asm volatile("" : "+v"(arg));
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[nt][i] = softcap_tanh(s[nt][i] * arg) * to_score;
      } else {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[nt][i] = softcap_tanh_small(s[nt][i] * to_arg) * to_score;
      }
    }
    const int oldest = MASK && window > 0 ? qpos - window : 0;  // first key this lane's query sees
    float mpart[2] = {-__builtin_inff(), -__builtin_inff()};  // two independent chains
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        if (MASK) {
          const int key = t0 + 32 * nt + 8 * (i >> 2) + 4 * hh + (i & 3);
          s[nt][i] = key <= qpos && key >= oldest ? s[nt][i] : -__builtin_inff();
        }
        mpart[nt] = fmaxf(mpart[nt], s[nt][i]);
      }
    }
    // (the scale is applied here, to fp32 scores, as the reference does: folded into Q -- which
    // would save the multiply-add below -- it is rounded to the element type, an error that
    // grows with the score and reaches several percent of the probabilities at |score| ~ 100)
    const float mloc = max_xor32(fmaxf(mpart[0], mpart[1])) * cs;
    if (__any(mloc > m_run + kRescaleGap)) {
      const float m_new = fmaxf(m_run, mloc);  // finite from tile 0 on (key 0 is visible)
      // (a fully masked row under a sliding window keeps m_new = -inf: leave it untouched)
      const float alpha = (MASK && PAGED && m_new == -__builtin_inff()) ? 1.0f : __builtin_amdgcn_exp2f(m_run - m_new);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[mt][i] *= alpha;
    }
    // a row whose keys so far were all masked (sliding window) still has m_run = -inf
    const float m_ref = (MASK && PAGED && m_run == -__builtin_inff()) ? 0.0f : m_run;
    float psum = 0.0f;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(s[nt][i], cs, -m_ref));
        s[nt][i] = e;
        psum += e;
      }
    }
    l_run += psum;

    // ---- O^T += V^T . P^T ; step (nt, st) consumes registers 8*st .. 8*st+7 of s[nt], which
    // belong to keys 32*nt + 16*st + 8*a + 4*hh + r (slot e = 4*a + r).  The A operand wants,
    // for dim d = 32*mt + col, the same 8 keys: two transposing reads (a = 0, 1), in each of
    // which lane s of 16-lane group g supplies row 4*hh + (s >> 2) (+ the step's key base),
    // dims 32*mt + 16*(g & 1) + 4*(s & 3) .. +3.
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        u32x4 pf;
        pf[0] = Mma32<DT>::pack2(s[nt][8 * st + 0], s[nt][8 * st + 1]);
        pf[1] = Mma32<DT>::pack2(s[nt][8 * st + 2], s[nt][8 * st + 3]);
        pf[2] = Mma32<DT>::pack2(s[nt][8 * st + 4], s[nt][8 * st + 5]);
        pf[3] = Mma32<DT>::pack2(s[nt][8 * st + 6], s[nt][8 * st + 7]);
        const unsigned char* vstep = vs + (32 * nt + 16 * st) * SM::kRowBytes;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const u32x2 lo = lds_read_tr16(vstep + v_off[mt]);
          const u32x2 hi = lds_read_tr16(vstep + v_off[mt] + 8 * SM::kRowBytes);
          o[mt] = Mma32<DT>::run(u32x4{lo[0], lo[1], hi[0], hi[1]}, pf, o[mt]);
        }
      }
    }
  };

  using NoClamp = std::integral_constant<bool, false>;
  using Clamp = std::integral_constant<bool, true>;
  // vmcnt(0): the direct-to-LDS loads of this wave have landed before the barrier publishes
  // the buffer (encoding: vmcnt = 0, expcnt / lgkmcnt left at their maxima)
  auto wait_dma = [&]() { __builtin_amdgcn_s_waitcnt(0x0F70); };
  using Yes = std::integral_constant<bool, true>;
  using No = std::integral_constant<bool, false>;
  // Group grp takes tiles jfirst + grp, + KG, ...; both groups make the same number of steps, one barrier
  // each.  A wave whose rows all lie past the sequence only copies.
  const bool wave_rows = q0 + __builtin_amdgcn_readfirstlane(wave_q0) < L;
  int jb = jfirst;  // the step's first tile
  // (the step's LDS buffer, worked out where it is used: carried along as a variable it costs the paged
  // kernels 50 registers)
  auto buf = [&]() -> int { return ((jb - jfirst) / KG) & 1; };
  auto stage_tile = [&](int j, int to) __attribute__((always_inline)) {
    if (j >= ntiles) return;
    if (j < nfull) load_tile(NoClamp{}, j * kTileN, to); else load_tile(Clamp{}, j * kTileN, to);
  };
  if (PAGED) fetch_pages((jb + grp) * kTileN);
  stage_tile(jb + grp, 0);
  wait_dma();
  __syncthreads();

  auto end_step = [&]() __attribute__((always_inline)) {
    wait_dma();
    __syncthreads();
    jb += KG;
  };
  // a step whose tiles may be masked, or whose successors may run past the sequence: at the window's edge,
  // the last unmasked tiles, the diagonal
  auto edge_step = [&]() __attribute__((always_inline)) {
    const int j = jb + grp;
    stage_tile(j + KG, buf() ^ 1);
    // a diagonal tile still lies entirely under the diagonal for the waves further down (and a tile at
    // the window's edge entirely inside it for some)
    const bool wave_full = softcap <= 0.0f && (j + 1) * kTileN - 1 <= wave_first_pos &&
                           (window <= 0 || j * kTileN >= wave_last_pos - window);
    if (j < ntiles) {
      if (wave_full) process_tile(No{}, No{}, j, buf());
      else process_tile(Yes{}, No{}, j, buf());
    }
    end_step();
  };
  if (!wave_rows) {
    while (jb < ntiles) {
      stage_tile(jb + grp + KG, buf() ^ 1);
      end_step();
    }
  } else {
    if (PAGED)
      while (jb < min(jopen, ntiles)) edge_step();
    // tiles under the diagonal (and inside every query's window) whose successor is also under it:
    // nothing to mask or clamp
    while (jb + 2 * KG - 1 < nfull) {
      prepare_tile(NoClamp{}, (jb + grp + KG) * kTileN, buf() ^ 1);
      process_tile(No{}, Yes{}, jb + grp, buf());
      end_step();
    }
    while (jb < ntiles) edge_step();
  }

  if constexpr (KG > 1) {
    // the second group's partial results, by lane: its rows are the first group's
    float* part = (float*)smem_all + wave * ((16 * MT + 2) * 64);
    if (grp == 1) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *(f32x4*)(part + ((4 * mt + q) * 64 + lane) * 4) =
              f32x4{o[mt][4 * q], o[mt][4 * q + 1], o[mt][4 * q + 2], o[mt][4 * q + 3]};
      part[16 * MT * 64 + lane] = m_run;
      part[16 * MT * 64 + 64 + lane] = l_run;
    }
    __syncthreads();
    if (grp == 1) return;
    const float m1 = part[16 * MT * 64 + lane], l1 = part[16 * MT * 64 + 64 + lane];
    const float m = fmaxf(m_run, m1);
    // (a group without a visible key: weight 0)
    const float a0 = m_run == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(m_run - m);
    const float a1 = m1 == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(m1 - m);
    l_run = l_run * a0 + l1 * a1;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 v = *(const f32x4*)(part + ((4 * mt + q) * 64 + lane) * 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) o[mt][4 * q + i] = o[mt][4 * q + i] * a0 + v[i] * a1;
      }
  }

  // ---- epilogue: normalise and store O (lane holds 4 consecutive dims per register quad)
  l_run += __shfl_xor(l_run, 32);
  if (PACK && parted) {
    if (qrow < L) {
      const int64_t row = ((int64_t)split * p.tokens + tok0 + qrow) * p.Hq + head;
      float* wo = p.ws_o + row * p.ws_d;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int qd = 0; qd < 4; ++qd)
          if (!RAGGED || 32 * mt + 8 * qd + 4 * hh < p.dv)
            *(f32x4*)(wo + 32 * mt + 8 * qd + 4 * hh) =
                f32x4{o[mt][4 * qd], o[mt][4 * qd + 1], o[mt][4 * qd + 2], o[mt][4 * qd + 3]};
      if (hh == 0) {
        p.ws_ml[2 * row] = m_run;
        p.ws_ml[2 * row + 1] = l_run;
      }
    }
    return;
  }
  if (qrow < L) {
    const float inv = l_run > 0.0f ? 1.0f / l_run : 0.0f;
    unsigned short* op = (unsigned short*)p.o + (tok0 + qrow) * p.o_st + (int64_t)head * p.o_sh;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        u32x2 w;
        w[0] = Mma32<DT>::pack2(o[mt][4 * qd + 0] * inv, o[mt][4 * qd + 1] * inv);
        w[1] = Mma32<DT>::pack2(o[mt][4 * qd + 2] * inv, o[mt][4 * qd + 3] * inv);
        if (!RAGGED || 32 * mt + 8 * qd + 4 * hh < p.dv) *(u32x2*)(op + 32 * mt + 8 * qd + 4 * hh) = w;
      }
    }
  }
}

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
// filled in (or zeroed) by the caller.
int launch_prefill(PrefillParams& p, bool paged, int B, int Hq, int Hkv, int Dk, int Dv, int max_len,
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
  // Heads of a KV group share workgroups in launches of more than two rounds (two workgroups on a CU, four with
  // up to 64 dims), where the KV heads fall on the XCDs by themselves and the row tiles fit the grid.  32 heads
  // (8 kv) of 128: 8 x 512 - 4096 tokens 284 -> 275 us, 8 x 100 - 1000 44 -> 41.3; 28 (4): 42 -> 39.8, 8 x 300 -
  // 1000 over 2000 110 -> 99.  In one round the workgroups that finish early help their neighbours and it loses:
  // 8 heads (1 kv), 3 x 1000 - 4000 55.5 -> 56.9; 32 (8) of 64 dims, 4 x 60 - 300 6.9 -> 7.5.  Over histories
  // of unequal lengths 2.5 rounds are a matter of luck (8 x 300 - 600 over up to 4096, ten batches: 0.98 - 1.07).
  const int row_waves = small ? 2 : 4;
  const int64_t all_wgs = ceil_div(max_len, 128) * B * Hq, slots = (int64_t)current_device_cu_count() * (D <= 64 ? 4 : 2);
  int64_t qtiles = ceil_div(ceil_div(max_len, 32) * p.group, row_waves);
  // (A kernel of its own: where heads do not share, its longer start costs 1 %, 16 heads, 16 kv, of 64: 176.2 / 178.7.)
  const bool share = !plan.use && !small && all_wgs > (paged ? 3 : 2) * slots && (8 % Hkv == 0 || Hkv % 8 == 0) &&
                     qtiles <= 65535 && p.group > 1 && p.group <= 4096;
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
#define DLB_LAUNCH_PREFILL_RW(DT_, D_, PG_, RW_, PK_, SH_)                                                    \
  do {                                                                                                        \
    if (ragged)                                                                                               \
      launch((prefill_attn_kernel<DT_, D_, PG_, true, RW_, PK_, SH_>), grid, dim3(kThreads), s, p);           \
    else                                                                                                      \
      launch((prefill_attn_kernel<DT_, D_, PG_, false, RW_, PK_, SH_>), grid, dim3(kThreads), s, p);          \
  } while (0)
#define DLB_LAUNCH_PREFILL(DT_, D_, PG_)                                                 \
  do {                                                                                   \
    if (PG_ != 0 && plan.use) DLB_LAUNCH_PREFILL_RW(DT_, D_, PG_, 4, (PG_ != 0), false); \
    else if (small) DLB_LAUNCH_PREFILL_RW(DT_, D_, PG_, 2, false, false);                \
    else if (share) DLB_LAUNCH_PREFILL_RW(DT_, D_, PG_, 4, false, true);                 \
    else DLB_LAUNCH_PREFILL_RW(DT_, D_, PG_, 4, false, false);                           \
  } while (0)
#define DLB_DISPATCH_PREFILL_DT(DT_, PG_)                                                                       \
  do {                                                                                                          \
    if (D == 256 && share)                                                                                      \
      launch((prefill_attn_kernel<DT_, 256, PG_, true, 4, false, true>), grid, dim3(kThreads), s, p);           \
    else if (D == 256)                                                                                          \
      launch((prefill_attn_kernel<DT_, 256, PG_, true, 4, false, false>), grid, dim3(kThreads), s, p);          \
    else if (D == 128) DLB_LAUNCH_PREFILL(DT_, 128, PG_);                                                       \
    else if (D == 96) DLB_LAUNCH_PREFILL(DT_, 96, PG_);                                                         \
    else DLB_LAUNCH_PREFILL(DT_, 64, PG_);                                                                      \
  } while (0)
#define DLB_DISPATCH_PREFILL(PG_)                                               \
  if (dtype == DLB_DTYPE_BF16) DLB_DISPATCH_PREFILL_DT(DLB_DTYPE_BF16, PG_);    \
  else DLB_DISPATCH_PREFILL_DT(DLB_DTYPE_F16, PG_)
  // pages that hold whole 64-key tiles take the kernel with one page look-up per tile (the lane
  // offsets inside a page are 32-bit)
  const bool tile_pages = paged && p.page % kTileN == 0 &&
                          (int64_t)p.page * p.k_st * 2 <= 0x7fffffff && (int64_t)p.page * p.v_st * 2 <= 0x7fffffff;
  if (tile_pages) {
    DLB_DISPATCH_PREFILL(2);
  } else if (paged) {
    DLB_DISPATCH_PREFILL(1);
  } else {
    DLB_DISPATCH_PREFILL(0);
  }
#undef DLB_DISPATCH_PREFILL
#undef DLB_DISPATCH_PREFILL_DT
#undef DLB_LAUNCH_PREFILL
#undef DLB_LAUNCH_PREFILL_RW
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
  return launch_prefill(p, false, B, Hq, Hkv, D, D, max_len, max_len, sm_scale, dtype, nullptr, 0, stream);
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
  return launch_prefill(p, true, B, Hq, Hkv, D, Dv, max_q_len, (int64_t)page * max_blocks, sm_scale, dtype, ws,
                        ws_bytes, stream);
}
