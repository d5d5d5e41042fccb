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
#pragma once
#include <type_traits>

#include "common.h"

namespace dlb {

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
// Which kernel a launch takes: padded head size, layout (PAGED), ragged head sizes, 64-row workgroups, packed heads
// or split keys, heads that share workgroups.
struct PrefillForm {
  int dtype, D, paged;
  bool ragged, small, pack, share;
};
// Soft-capped scores (paged only): the CAP kernels, in a source file of their own, since they take as long to
// compile as the others.
void launch_prefill_capped(const PrefillParams& p, const PrefillForm& form, dim3 grid, hipStream_t s);

namespace {

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
// CAP: the scores are soft-capped.  A kernel of its own, so that the tiles under the diagonal, nearly all, have a copy
// without the mask too; bound by vector instructions, the tanh takes as many as all the rest.  Every tile masked /
// now, us, 8 x 512 tokens over up to 4096, 32 heads (8 kv) of 128: 357 / 268 (no cap 200), of 64 250 / 209; 8 heads
// (1 kv) of 128, 9 x 162 - 650 over up to 5910 272 / 170; 28 (4), 2 x 10 - 30 over up to 5000 46 / 34.
template <int DT, int D, int PAGED, bool RAGGED, int RW, bool PACK, bool SHARE = false, bool CAP = false>
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
  // tiles below this index lie entirely under the diagonal for every wave of the workgroup
  // (all 64 keys <= position of row q0): no mask, no clamping of key rows
  const int nfull = min((hist + q0 + 1) / kTileN, ntiles);
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
  // (CAP: the scores are turned into units of the cap)
  const float cs = CAP ? p.softcap * 1.4426950408889634f : p.scale_log2e;

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
    if constexpr (CAP) {  // tanh(x * scale / cap)
      const float to_arg = p.sm_scale / p.softcap;
      float top = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) top = fmaxf(top, fmaxf(fabsf(s[0][i]), fabsf(s[1][i])));
      // Mostly none of the wave's scores comes near the cap, and the polynomial is all there is: 8 x 512
      // tokens over 4096, every tile masked, 645 -> 497 us; where some do in every tile the look costs nothing (646).
      if (__any(top * to_arg >= kSoftcapSmall)) {
        // (a factor of its own: with the same one in both branches the compiler moves the polynomial in front
        // of them, 32 more registers live)
        float arg = to_arg;
        asm volatile("" : "+v"(arg));
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[nt][i] = softcap_tanh(s[nt][i] * arg);
      } else {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[nt][i] = softcap_tanh_small(s[nt][i] * to_arg);
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
    const bool wave_full = (j + 1) * kTileN - 1 <= wave_first_pos &&
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

// Launches the kernel of `form`.  CAP: paged, without shared heads.
template <int DT, int D, int PAGED, bool RAGGED, bool CAP>
void launch_prefill_as(const PrefillParams& p, const PrefillForm& form, dim3 grid, hipStream_t s) {
  const dim3 block(kThreads);
  if constexpr (D <= 128) {
    if (PAGED && form.pack) {
      launch(prefill_attn_kernel<DT, D, PAGED, RAGGED, 4, (PAGED != 0), false, CAP>, grid, block, s, p);
      return;
    }
    if (form.small) {
      launch(prefill_attn_kernel<DT, D, PAGED, RAGGED, 2, false, false, CAP>, grid, block, s, p);
      return;
    }
  }
  if constexpr (!CAP)
    if (form.share) {
      launch(prefill_attn_kernel<DT, D, PAGED, RAGGED, 4, false, true, false>, grid, block, s, p);
      return;
    }
  launch(prefill_attn_kernel<DT, D, PAGED, RAGGED, 4, false, false, CAP>, grid, block, s, p);
}
template <int DT, int D, bool CAP>
void launch_prefill_size(const PrefillParams& p, const PrefillForm& form, dim3 grid, hipStream_t s) {
  auto by_layout = [&](auto ragged) {
    constexpr bool R = decltype(ragged)::value;
    if (form.paged == 2) launch_prefill_as<DT, D, 2, R, CAP>(p, form, grid, s);
    else if (CAP || form.paged == 1) launch_prefill_as<DT, D, 1, R, CAP>(p, form, grid, s);
    else if constexpr (!CAP) launch_prefill_as<DT, D, 0, R, false>(p, form, grid, s);
  };
  if constexpr (D == 256) by_layout(std::true_type{});
  else if (form.ragged) by_layout(std::true_type{});
  else by_layout(std::false_type{});
}
template <bool CAP>
void launch_prefill_kernel(const PrefillParams& p, const PrefillForm& form, dim3 grid, hipStream_t s) {
  auto by_size = [&](auto dt) {
    constexpr int DT = decltype(dt)::value;
    if (form.D == 256) launch_prefill_size<DT, 256, CAP>(p, form, grid, s);
    else if (form.D == 128) launch_prefill_size<DT, 128, CAP>(p, form, grid, s);
    else if (form.D == 96) launch_prefill_size<DT, 96, CAP>(p, form, grid, s);
    else launch_prefill_size<DT, 64, CAP>(p, form, grid, s);
  };
  if (form.dtype == DLB_DTYPE_BF16) by_size(std::integral_constant<int, DLB_DTYPE_BF16>{});
  else by_size(std::integral_constant<int, DLB_DTYPE_F16>{});
}

}  // namespace
}  // namespace dlb
