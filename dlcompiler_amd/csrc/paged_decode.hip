// Paged decode attention for gfx950: one query token per sequence, KV cache in fixed-size
// pages addressed through a block table, grouped-query heads.
//
// Replaces the decode branch of paged_attention_fwd
// (python/dlBLAS/dlblas/kernels/paged_attention.py:604-671): _fwd_grouped_split_kernel
// (:45-234) and _reduce_split_kernel (:238-285).  Same mathematics -- per (sequence, kv head)
// the query heads of the group are batched against the head's K/V stream, online softmax in
// fp32, P rounded to the cache dtype before P.V, split-KV partials (O, m, l) combined by a
// second kernel -- with a different decomposition:
//   * the KV streams of all sequences are laid end to end (in units of 32 keys) and cut into
//     equal pieces, one per team of wavefronts (one wavefront per kv-head unit), as many
//     teams as fit on the chip at once: every wavefront streams the same number of bytes
//     whatever the mix of context lengths, instead of a fixed four-way split per sequence.
//     A piece that crosses a sequence boundary yields one partial per sequence;
//   * one wavefront per (piece, kv-head unit).  S^T = K.Q^T runs on 16x16x32 MFMA with the K rows loaded
//     straight from HBM into the A-operand layout (d is contiguous in memory and in the
//     operand), so K never touches LDS;
//   * V needs the key index contiguous per lane, so its tile is transposed on the way into
//     LDS (4 keys x 8 dims per lane, v_perm + ds_write_b64) and read back as 128-bit operands;
//     the key order inside each 32-key MFMA step is permuted so that the softmax output
//     registers ARE the B operand of O^T = V^T.P^T: P never moves between lanes.
// The kernel is an HBM stream (4 FLOP/byte at GQA 4:1); everything else is sized to keep
// tens of KB of loads in flight per CU.
// Short contexts are bound by latency instead: there one workgroup of 4 or 8 wavefronts per (sequence,
// kv-head unit) cuts the context among its wavefronts and merges their partials in LDS, in one
// launch (paged_decode_direct_kernel).
#include "common.h"

namespace dlb {
namespace {

struct DecodeParams {
  const void* q;
  const void* k;
  const void* v;
  void* o;
  IdxArray block_table;
  IdxArray kv_len;
  float* ws_o;      // [B, Hq, nsplit_max, D]
  float* ws_ml;     // [B, Hq, nsplit_max, 2]
  int32_t* ws_np;   // [B] partials written for each sequence
  int64_t q_sb, q_sh;
  int64_t k_sp, k_st, k_sh;
  int64_t v_sp, v_st, v_sh;
  int64_t o_sb, o_sh;
  int64_t bt_stride;
  int B, Hq, Hkv, group, hchunks;
  int page, page_shift;  // page_shift < 0: page is not a power of two
  int max_blocks;
  int min_units, nsplit_max;  // smallest piece (32-key units); partial slots per (sequence, head)
  int num_teams;
  int once_units;  // K and V of more units than this go past the caches (CHOICE)
  float scale_log2e;
  float sm_scale;
  int dk, dv;      // real key / value head sizes (<= the padded size the kernel is built for)
  int window;      // > 0: keys older than (ctx - 1 - window) are masked (paged_attention.py:163-167)
  float softcap;   // > 0: logits -> softcap * tanh(logits / softcap) (paged_attention.py:186-189)
};

template <int DT>
struct Mma16;
template <>
struct Mma16<DLB_DTYPE_BF16> {
  static __device__ __forceinline__ f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
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
struct Mma16<DLB_DTYPE_F16> {
  static __device__ __forceinline__ f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ unsigned int pack2(float a, float b) {
    typedef __attribute__((ext_vector_type(2))) float f2;
    typedef __attribute__((ext_vector_type(2))) _Float16 h2;
    f2 f = {a, b};
    return __builtin_bit_cast(unsigned int, __builtin_convertvector(f, h2));
  }
};

constexpr int kTile = 64;          // keys per iteration
constexpr int kVtRowBytes = 144;   // 64 keys * 2 B + 16 B pad

// D is the padded head size the kernel is built for (64 or 128).  RAGGED: the real key size dk
// and / or value size dv is smaller (any multiple of 8): query dims past dk are zero, so whatever
// the key loads of those dims return does not count -- they are redirected to the row's first 16
// bytes to stay inside the cache -- and value dims past dv (redirected likewise) only produce
// output dims that are never stored.  The reference splits odd head sizes the same way into
// power-of-two blocks with masked loads (python/dlBLAS/dlblas/kernels/paged_attention.py:531-539).
// (The masked variant keeps a few more per-lane offsets alive: it is built for one wavefront per
// SIMD instead of two rather than spilling them.)
// ONCE: K and V go past the caches (see may_read_once); without it, V alone.
// HELD: page numbers come from a run of the block table that the lanes hold, else from scalar loads half a tile ahead.
struct PageRun {
  int entry;  // this lane's: page number of the sequence's page `first` + lane
  int first;
};
template <int DT, int D, bool POW2, bool RAGGED, bool ONCE, bool HELD = false>
struct DecodeSegment {
  static constexpr int KS = D / 32;  // MFMA k-steps over the head dim
  // K in whole 128-byte lines.  A load that brings 16 operand rows of one key each touches 16 half lines, so
  // every line twice, and the caches have to keep it in between.  With the halves of a line in two operand rows
  // it touches eight lines, once; each row then meets the query's dims of both halves, and of the two products
  // one counts (twice the MFMAs of S^T, which a stream of K/V has to spare).
  static constexpr bool KL = ONCE && !RAGGED && D % 64 == 0;
  static constexpr int MT = D / 16;  // 16-row tiles of O^T
  static constexpr int DG = D / 8;   // 8-dim groups per key row
  static constexpr int kVtBytes = D * kVtRowBytes;
  f32x4 o[MT];  // O^T: lane (g, c) holds dims 16 mt + 4 g .. + 3 of query head c
  float m_run;  // running maximum of head c (base 2)
  float l_run;  // softmax denominator of head c (complete after run())

  // Keys [k_begin, k_end) of sequence b (context ctx, keys before kv_min masked), for one kv-head
  // unit; k_begin is a multiple of 32.  vt: this wavefront's V^T tile in LDS (kVtBytes).
  __device__ __forceinline__ void run(const DecodeParams& p, unsigned char* vt, int b, int ctx, int kvh, int head,
                                      bool head_ok, int k_begin, int k_end, int kv_min,
                                      const PageRun& pages = PageRun{0, 0}) {
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4;  // lane group 0..3
  const int c = lane & 15;  // column (query head) / row (key) inside a 16-tile
  const unsigned short* qb = (const unsigned short*)p.q;
  // everything that shapes the walk is wave-uniform; saying so keeps the loops and the page
  // arithmetic on the scalar unit
  b = __builtin_amdgcn_readfirstlane(b);
  ctx = __builtin_amdgcn_readfirstlane(ctx);
  kvh = __builtin_amdgcn_readfirstlane(kvh);
  k_begin = __builtin_amdgcn_readfirstlane(k_begin);
  k_end = __builtin_amdgcn_readfirstlane(min(k_end, ctx));
  kv_min = __builtin_amdgcn_readfirstlane(kv_min);
  const int32_t* bt = p.block_table.p + (((int64_t)b * p.bt_stride) << p.block_table.sh);
  const int bt_sh = p.block_table.sh;
  // (what the loops use: arguments that are loaded again, see arguments_again, would be loaded in every step)
  const int page = p.page, page_shift = p.page_shift;
  const int64_t k_sp = p.k_sp, v_sp = p.v_sp;
  const float softcap = p.softcap, sm_scale = p.sm_scale, scale_log2e = p.scale_log2e;

  // Q^T as the B operand: lane (n = query head c, k = dims 32*ks + 8g .. +8)
  u32x4 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    qf[ks] = u32x4{0u, 0u, 0u, 0u};
    if (head_ok && (!RAGGED || 32 * ks + 8 * g < p.dk))
      qf[ks] = *(const u32x4*)(qb + (int64_t)b * p.q_sb + (int64_t)head * p.q_sh + 32 * ks + 8 * g);
  }

#pragma unroll
  for (int mt = 0; mt < MT; ++mt) o[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  m_run = -__builtin_inff();
  l_run = 0.0f;  // per-lane partial of the softmax denominator

  // Addressing: a 16-key sub-tile never straddles a page (page % 16 == 0), so its physical
  // page comes from ONE wave-uniform block-table entry (a scalar load) and every lane adds a
  // 32-bit byte offset to a uniform 64-bit base.
  // (uniform_ptr loses that a pointer is global, and a wait for LDS waits for every flat load in flight, here the half
  // tile just asked for.  Flat / so, 8 kv heads of 128, contexts much shorter than the table: 1 x 4000 keys 26.9 / 23.3
  // us, 8 x 500 - 8000 31.4 / 27.2; filling it, 64 x 512 - 8192 161.4 / 161.7, of 64 97.5 / 96.6)
  typedef const __attribute__((address_space(1))) u32x4* gvec_t;
  const unsigned char* kbytes = (const unsigned char*)p.k + (int64_t)kvh * p.k_sh * 2;
  const unsigned char* vbytes = (const unsigned char*)p.v + (int64_t)kvh * p.v_sh * 2;
  const uint32_t k_tok_bytes = (uint32_t)p.k_st * 2u, v_tok_bytes = (uint32_t)p.v_st * 2u;
  constexpr int VL = 64 / DG < 4 ? 64 / DG : 4;  // 4-key groups of a sub-tile staged per pass
  constexpr int VPASS = 4 / VL;                  // passes per 16-key sub-tile
  const int dg = lane % DG, kgl = lane / DG;     // lanes with kgl >= VL idle
  // byte offsets of this lane's 16-byte pieces inside a key / value row
  uint32_t kdim_off[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) kdim_off[ks] = (!RAGGED || 32 * ks + 8 * g < p.dk) ? 64u * ks + 16u * g : 0u;
  const uint32_t kl_off = (uint32_t)(4 * (c >> 2) + ((c >> 1) & 1)) * k_tok_bytes + 64u * (c & 1) + 16u * g;
  const uint32_t vdim_off = (!RAGGED || 8 * dg < p.dv) ? 16u * dg : 0u;

  // The chunk is walked in half tiles of 32 keys (one k-step of the second product).  The loads
  // of half tile h + 1 are issued before half tile h is computed, so every wave keeps 16 KB of
  // requests in flight while it works; a wave's V^T staging buffer is private and LDS
  // operations of one wave execute in order, so no barrier is needed.
  struct HalfTile {
    u32x4 kf[2][KS];          // K: 2 sub-tiles of 16 keys, already in A-operand layout
    u32x4 vr[2][VPASS][4];    // V: per lane 4 consecutive keys x 8 dims per pass
  };
  // Block-table lookups are wave-uniform and must be SCALAR loads: as vector loads they sit in
  // the same in-order return queue as the K/V stream, and waiting for a page number means
  // waiting for every half tile still in flight.  The compiler will not use the scalar path for
  // memory the kernel might have written, so the load is issued by hand (and waited for on
  // the scalar counter), one half tile ahead of the loads that need the page numbers.
  int pg_ahead[2];  // physical pages of the two 16-key sub-tiles of the next half tile to load
  auto lookup_pages = [&](int h0) {
    const int32_t* entry[2];
    if constexpr (HELD) {
#pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
        const int base_key = min(h0 + 16 * sub, ctx - 1);
        const int pi = POW2 ? (base_key >> page_shift) : (base_key / page);
        pg_ahead[sub] = __builtin_amdgcn_readlane(pages.entry, __builtin_amdgcn_readfirstlane(pi - pages.first));
      }
      return;
    }
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const int base_key = min(h0 + 16 * sub, ctx - 1);  // clamp: never look past the context
      const int pi = POW2 ? (base_key >> page_shift) : (base_key / page);
      entry[sub] = (const int32_t*)uniform_ptr((const unsigned char*)(bt + (pi << bt_sh)));
    }
    int p0, p1;
    asm volatile("s_load_dword %0, %2, 0x0\n\ts_load_dword %1, %3, 0x0\n\ts_waitcnt lgkmcnt(0)"
                 : "=&s"(p0), "=&s"(p1)
                 : "s"(entry[0]), "s"(entry[1]));
    pg_ahead[0] = p0;
    pg_ahead[1] = p1;
  };
  auto load_half = [&](int h0, HalfTile& f) {
    const int pg_now[2] = {pg_ahead[0], pg_ahead[1]};
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const int base_key = min(h0 + 16 * sub, ctx - 1);  // uniform; clamp: never read past ctx
      const int pi =
          __builtin_amdgcn_readfirstlane(POW2 ? (base_key >> page_shift) : (base_key / page));
      const int64_t pg = (int64_t)pg_now[sub];
      const int page_key0 = pi * page;
      {
        const unsigned char* base = kbytes + pg * k_sp * 2;
        if constexpr (KL) {
          // Operand row c = 2 k + half: half line of key 4 (k / 2) + 2 pair + k % 2 of the sub-tile that holds
          // base_key.  (Its keys past the context are slots of the same page, and masked.)
#pragma unroll
          for (int pair = 0; pair < 2; ++pair) {
            const unsigned char* from = uniform_ptr(base + (int64_t)((base_key & ~15) - page_key0 + 2 * pair) * k_tok_bytes);
#pragma unroll
            for (int ln = 0; ln < KS / 2; ++ln)
              f.kf[sub][KS / 2 * pair + ln] = __builtin_nontemporal_load((gvec_t)(from + kl_off + 128 * ln));
          }
        } else {
          // K rows are read as two half-line (64-byte) pieces by consecutive k-steps: keep them
          // cacheable so the second piece hits the line the first one brought in
          const int key = min(h0 + 16 * sub + c, ctx - 1);
          const uint32_t off = (uint32_t)(key - page_key0) * k_tok_bytes;
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) {
            f.kf[sub][ks] = *(gvec_t)(base + off + (RAGGED ? kdim_off[ks] : 16u * g + 64 * ks));
          }
        }
      }
      {
        const unsigned char* base = vbytes + pg * v_sp * 2;
#pragma unroll
        for (int ps = 0; ps < VPASS; ++ps) {
          const int key0 = min(h0 + 16 * sub + 4 * (ps * VL + kgl), ctx - 1);
          const int room = ctx - 1 - key0;
          if (kgl < VL) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const uint32_t off = (uint32_t)(key0 - page_key0 + min(r, room)) * v_tok_bytes + vdim_off;
              f.vr[sub][ps][r] = __builtin_nontemporal_load((const u32x4*)(base + off));
            }
          }
        }
      }
    }
    lookup_pages(h0 + 32);
  };
  // st = parity of the half tile inside its 64-key tile = which 4 units of a V^T row it uses
  auto compute_half = [&](int h0, const HalfTile& f, int st) {
    // ---- S^T = K . Q^T (rows = keys, cols = query heads) ----
    f32x4 s[2];
    auto scores = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
        if constexpr (KL) {
#pragma unroll
          for (int pair = 0; pair < 2; ++pair) {
            f32x4 lower = f32x4{0.f, 0.f, 0.f, 0.f}, upper = lower;  // every row against either half line's dims
#pragma unroll
            for (int ln = 0; ln < KS / 2; ++ln) {
              const u32x4& k = f.kf[sub][KS / 2 * pair + ln];
              lower = Mma16<DT>::run(k, qf[2 * ln], lower);
              upper = Mma16<DT>::run(k, qf[2 * ln + 1], upper);
            }
            s[sub][2 * pair] = lower[0] + upper[1];
            s[sub][2 * pair + 1] = lower[2] + upper[3];
          }
        } else {
          s[sub] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) s[sub] = Mma16<DT>::run(f.kf[sub][ks], qf[ks], s[sub]);
        }
      }
    };

    // ---- V^T into LDS: Vt[d][pos], pos = 32*st + 8*g' + 4*a + r for key 32*st + 16*a + 4*g' + r
    auto stage_v = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
#pragma unroll
        for (int ps = 0; ps < VPASS; ++ps) {
          if (kgl < VL) {
            const int unit = 4 * st + ps * VL + kgl;  // 16-byte unit inside the row
            const int half = sub;                     // 8-byte half inside the unit
#pragma unroll
            for (int w = 0; w < 4; ++w) {
              const u32x4* v4 = f.vr[sub][ps];
              const unsigned int lo01 = __builtin_amdgcn_perm(v4[1][w], v4[0][w], 0x05040100u);
              const unsigned int lo23 = __builtin_amdgcn_perm(v4[3][w], v4[2][w], 0x05040100u);
              const unsigned int hi01 = __builtin_amdgcn_perm(v4[1][w], v4[0][w], 0x07060302u);
              const unsigned int hi23 = __builtin_amdgcn_perm(v4[3][w], v4[2][w], 0x07060302u);
              const int d0 = 8 * dg + 2 * w;
              const int sw = ((d0 >> 4) & 3) << 1;  // same for d0 and d0 + 1
              unsigned char* row = vt + d0 * kVtRowBytes + ((unit ^ sw) << 4) + (half << 3);
              *(u32x2*)(row) = u32x2{lo01, lo23};
              *(u32x2*)(row + kVtRowBytes) = u32x2{hi01, hi23};
            }
          }
        }
      }
    };
    if constexpr (KL) {
      stage_v();  // (first: its registers are needed for the two products)
      __builtin_amdgcn_sched_barrier(0);
      scores();
    } else {
      scores();
      stage_v();
    }

    // ---- online softmax over these 32 keys (log2 domain) ----
    float mloc = -__builtin_inff();
    if (softcap > 0.0f) {  // one uniform branch for the half tile, not one per element
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          s[sub][i] = softcap * softcap_tanh(s[sub][i] * sm_scale / softcap) * 1.4426950408889634f;
    } else {
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[sub][i] *= scale_log2e;
    }
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = h0 + 16 * sub + 4 * g + i;
        const float x = (key < k_end && key >= kv_min) ? s[sub][i] : -__builtin_inff();
        s[sub][i] = x;
        mloc = fmaxf(mloc, x);
      }
    }
    mloc = max_xor32(max_xor16(mloc));
    const float m_new = fmaxf(m_run, mloc);
    // a half tile can be entirely masked (sliding window, chunk tail): keep exponents finite
    const float m_ref = (m_new == -__builtin_inff()) ? 0.0f : m_new;
    if (__any(m_new > m_run)) {  // wave-uniform: skip the rescale when no maximum moved
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_ref);
      l_run *= alpha;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) o[mt] *= alpha;
    }
    m_run = m_new;
    float psum = 0.0f;
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float e = __builtin_amdgcn_exp2f(s[sub][i] - m_ref);
        s[sub][i] = e;
        psum += e;
      }
    }
    l_run += psum;

    // P^T as the B operand: slots 0..3 <- sub-tile 0, slots 4..7 <- sub-tile 1
    u32x4 pf;
    pf[0] = Mma16<DT>::pack2(s[0][0], s[0][1]);
    pf[1] = Mma16<DT>::pack2(s[0][2], s[0][3]);
    pf[2] = Mma16<DT>::pack2(s[1][0], s[1][1]);
    pf[3] = Mma16<DT>::pack2(s[1][2], s[1][3]);

    // ---- O^T += V^T . P^T ----
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int d = 16 * mt + c;
      const int sw = (mt & 3) << 1;
      const u32x4 a = *(const u32x4*)(vt + d * kVtRowBytes + (((4 * st + g) ^ sw) << 4));
      o[mt] = Mma16<DT>::run(a, pf, o[mt]);
    }
  };

  HalfTile ha, hb;
  if (k_begin < k_end) {  // (a segment entirely before the window is empty)
    lookup_pages(k_begin);
    load_half(k_begin, ha);
    int t0 = k_begin;
    // steady state: the tile has both halves and another tile follows.  No run-time condition
    // surrounds a load here: where the two paths of a branch around loads join, the compiler
    // has to wait as if the loads had not been issued, i.e. for the ones just sent.
    for (; t0 + kTile < k_end; t0 += kTile) {
      load_half(t0 + 32, hb);
      __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the arithmetic below
      compute_half(t0, ha, 0);
      __builtin_amdgcn_sched_barrier(0);
      load_half(t0 + kTile, ha);
      __builtin_amdgcn_sched_barrier(0);
      compute_half(t0 + 32, hb, 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    // last tile: one or two halves
    const bool second = t0 + 32 < k_end;
    if (second) load_half(t0 + 32, hb);
    __builtin_amdgcn_sched_barrier(0);
    compute_half(t0, ha, 0);
    __builtin_amdgcn_sched_barrier(0);
    if (second) compute_half(t0 + 32, hb, 1);
  }

  l_run = sum_xor32(sum_xor16(l_run));

  }  // run
};

// first visible key of a context
__device__ __forceinline__ int first_visible(const DecodeParams& p, int ctx) {
  return p.window > 0 ? max(ctx - 1 - p.window, 0) : 0;
}

// The kernel's arguments, to be loaded where they are used.  (For two walks of which one runs: what both need, kept
// from before the branch, is more than the scalar registers, and those that spill go to lanes of vector registers that
// are not there.)
__device__ __forceinline__ const DecodeParams& arguments_again() {
  typedef const __attribute__((address_space(4))) DecodeParams* args_t;
  args_t args = (args_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(args));
  return *(const DecodeParams*)args;
}

// CHOICE: whether K and V go past the caches follows from the keys of the batch (see may_read_once).
// ONE: one sequence, pieces of the smallest size (see one_sequence): where a team's piece starts does not depend on the
// context, so the page numbers, the context and the query are asked for together.  A short run is a chain of loads (8 kv
// heads of 128, 1 x 4000 keys: with one link fewer here and one in the merge 10.75 -> 9.3 us, of which the merge 0.7).
template <int DT, int D, bool POW2, bool RAGGED, bool CHOICE, bool ONE>
__global__ __launch_bounds__(64, RAGGED ? 1 : 2) void paged_decode_split_kernel(const DecodeParams p) {
  // grid: x = (kv head, head chunk) unit, y = team.  The unit is the fastest index, so the
  // wavefronts that start together read the 256-byte head slices of the SAME token rows at the
  // same time: whole 2 KB cache rows are in flight together and DRAM pages are hit while open.
  constexpr int kVtBytes = DecodeSegment<DT, D, POW2, RAGGED, false>::kVtBytes;
  const int unit = blockIdx.x;
  const int team = blockIdx.y;
  const int kvh = unit / p.hchunks;
  const int hchunk = unit - kvh * p.hchunks;
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4, c = lane & 15;

  __shared__ __attribute__((aligned(16))) unsigned char vt[kVtBytes];
  __shared__ int32_t seg_lds[3][64];  // (first unit, units, context) of the 64 sequences being walked

  const int hq_local = hchunk * 16 + c;
  const bool head_ok = hq_local < p.group;
  const int head = kvh * p.group + hq_local;

  if constexpr (ONE) {
    using Segment = DecodeSegment<DT, D, POW2, RAGGED, false, true>;
    const int max_ctx = p.max_blocks * p.page, k_begin = team * p.min_units * 32;
    if (k_begin >= max_ctx) return;
    PageRun pages;
    pages.first = POW2 ? k_begin >> p.page_shift : k_begin / p.page;
    pages.entry = p.block_table[min(pages.first + lane, p.max_blocks - 1)];
    const int ctx = __builtin_amdgcn_readfirstlane(min(p.kv_len[0], max_ctx));
    if (k_begin >= ctx) return;
    if (team == 0 && unit == 0 && lane == 0) p.ws_np[0] = (ctx + 32 * p.min_units - 1) / (32 * p.min_units);
    Segment seg;
    seg.run(p, vt, 0, ctx, kvh, head, head_ok, k_begin, k_begin + 32 * p.min_units, 0, pages);
    if (head_ok) {
      const int64_t slot = (int64_t)head * p.nsplit_max + team;
      float* wo = p.ws_o + slot * D;
#pragma unroll
      for (int mt = 0; mt < Segment::MT; ++mt) *(f32x4*)(wo + 16 * mt + 4 * g) = seg.o[mt];
      if (g == 0) {
        p.ws_ml[slot * 2 + 0] = seg.m_run;
        p.ws_ml[slot * 2 + 1] = seg.l_run;
      }
    }
    return;
  }

  // ---- this team's piece of the concatenated KV streams (32-key units, visible keys only: with a
  // sliding window the teams share what the windows leave, not the whole contexts) ----
  auto context_of = [&](int bb) { return bb < p.B ? max(p.kv_len[bb], 0) : 0; };
  auto units_of = [&](int ctx) { return ((ctx + 31) >> 5) - (first_visible(p, ctx) >> 5); };
  // (the first 64 sequences' values serve the walk as well: of a short run's chain of loads and scans every link
  // counts)
  const int first_ctx = context_of(lane);
  const int first_incl = wave_inclusive_scan(units_of(first_ctx));
  int total = __builtin_amdgcn_readlane(first_incl, 63);
  for (int b0 = 64; b0 < p.B; b0 += 64)
    total += __builtin_amdgcn_readlane(wave_inclusive_scan(units_of(context_of(b0 + lane))), 63);
  const int upt = max((total + p.num_teams - 1) / p.num_teams, p.min_units);  // units per team
  const int lo = team * upt;
  if (lo >= total) return;
  const int hi = min(lo + upt, total);

  // ---- walk the sequences this piece overlaps ----
  auto walk = [&](const DecodeParams& p, auto once) __attribute__((always_inline)) {
  using Segment = DecodeSegment<DT, D, POW2, RAGGED, decltype(once)::value>;
  int carry = 0;  // units of all sequences before b0
  for (int b0 = 0; b0 < p.B; b0 += 64) {
    const int ctx_mine = b0 == 0 ? first_ctx : context_of(b0 + lane);
    const int t = units_of(ctx_mine);
    const int incl = b0 == 0 ? first_incl : wave_inclusive_scan(t);
    const int excl = carry + incl - t;
    uint64_t hit = __ballot(t > 0 && excl < hi && excl + t > lo);
    // park the per-sequence values in LDS: nothing per-lane stays live across a segment
    seg_lds[0][lane] = excl;
    seg_lds[1][lane] = t;
    seg_lds[2][lane] = ctx_mine;
    carry += __builtin_amdgcn_readlane(incl, 63);
    while (hit) {  // wave-uniform
      const int l = __builtin_ctzll(hit);
      hit &= hit - 1;
      const int b = b0 + l;
      const int pb = __builtin_amdgcn_readfirstlane(seg_lds[0][l]);
      const int tb = __builtin_amdgcn_readfirstlane(seg_lds[1][l]);
      const int ctx = __builtin_amdgcn_readfirstlane(seg_lds[2][l]);
      const int first_team = pb / upt;
      if (team == first_team && unit == 0 && lane == 0)
        p.ws_np[b] = (pb + tb - 1) / upt - first_team + 1;
      // one segment of sequence b -> partial number team - first_team of b
      const int kv_min = first_visible(p, ctx), k0 = kv_min & ~31;
      Segment seg;
      seg.run(p, vt, b, ctx, kvh, head, head_ok, k0 + (max(lo, pb) - pb) * 32, k0 + (min(hi, pb + tb) - pb) * 32,
              kv_min);
      if (head_ok) {
        const int64_t slot = ((int64_t)b * p.Hq + head) * p.nsplit_max + (team - first_team);
        float* wo = p.ws_o + slot * D;
#pragma unroll
        for (int mt = 0; mt < Segment::MT; ++mt) *(f32x4*)(wo + 16 * mt + 4 * g) = seg.o[mt];
        if (g == 0) {
          p.ws_ml[slot * 2 + 0] = seg.m_run;
          p.ws_ml[slot * 2 + 1] = seg.l_run;
        }
      }
    }
    if (carry >= hi) break;
  }
  };  // walk
  if constexpr (CHOICE) {
    if (total > p.once_units) walk(arguments_again(), std::true_type{});
    else walk(arguments_again(), std::false_type{});
  } else {
    walk(p, std::false_type{});
  }
}

// Combine the partials of one (sequence, head): O = sum_s 2^(m_s - m) O_s / sum_s 2^(m_s - m) l_s
// (paged_attention.py:238-285 with the exponent in base 2).  A row of D floats is read by D / 4 lanes
// and the rows are spread over the workgroup, which asks for 64 of them at once (D = 256: 32); the
// kernel is a chain of memory latencies, so what does not depend on the number of partials (the
// first 64 (m, l) pairs and the first round of rows: inside the scratch whether written or not,
// and masked) is requested together with it.
constexpr int kCombineThreads = 256;
// EARLY: the first 64 rows are all requested with the number of partials instead of after it: for launches of up to a
// workgroup per CU (2 x 1500 - 3000 keys 10.8 -> 10.0 us); larger ones would read rows that no partial was written to.
template <int DT, int D, bool EARLY>
__global__ __launch_bounds__(kCombineThreads) void paged_decode_combine_kernel(const DecodeParams p) {
  constexpr int RL = D / 4;                    // lanes per row
  constexpr int RG = kCombineThreads / RL;     // rows per round
  constexpr int E = EARLY ? (64 + RG - 1) / RG : 1;  // rows per lane requested early
  __shared__ float acc_lds[RG][D];
  __shared__ float w_lds[kCombineThreads / 64][64];
  const int head = blockIdx.x, b = blockIdx.y, tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int d4 = tid % RL, rg = tid / RL;
  const bool row_lane = rg < RG;  // (D = 96: the last lanes have no row)
  const int64_t slot0 = ((int64_t)b * p.Hq + head) * p.nsplit_max;
  const int ctx = p.kv_len[b];
  int ns = p.ws_np[b];  // partials of this sequence (unset if it is empty)
  float m0 = -__builtin_inff(), l0 = 0.0f;
  if (lane < p.nsplit_max) {
    m0 = p.ws_ml[(slot0 + lane) * 2];
    l0 = p.ws_ml[(slot0 + lane) * 2 + 1];
  }
  f32x4 early[E];
#pragma unroll
  for (int u = 0; u < E; ++u)  // (clamped: inside the scratch, masked below)
    early[u] = *(const f32x4*)(p.ws_o + (slot0 + min(rg + u * RG, p.nsplit_max - 1)) * D + 4 * d4);
  if (ctx <= 0) ns = 0;
  if (lane >= ns) {
    m0 = -__builtin_inff();
    l0 = 0.0f;
  }
  float m = m0;
  for (int s0 = 64; s0 < ns; s0 += 64) m = fmaxf(m, s0 + lane < ns ? p.ws_ml[(slot0 + s0 + lane) * 2] : m);
  m = max_xor32(max_xor16(row16_max(m)));
  float den = 0.0f;
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < ns; s0 += 64) {
    float ms = m0, ls = l0;
    if (s0 > 0) {
      ms = s0 + lane < ns ? p.ws_ml[(slot0 + s0 + lane) * 2] : -__builtin_inff();
      ls = s0 + lane < ns ? p.ws_ml[(slot0 + s0 + lane) * 2 + 1] : 0.0f;
    }
    const float w = ms == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(ms - m);
    den += w * ls;
    w_lds[wave][lane] = w;  // (each wave its own copy: no barrier)
    const int n = min(64, ns - s0);
    if (EARLY && s0 == 0) {
#pragma unroll
      for (int u = 0; u < E; ++u) {
        const int r = rg + u * RG;
        const float wr = w_lds[wave][min(r, 63)];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] += r < n ? wr * early[u][i] : 0.0f;
      }
      continue;
    }
    // All 64 rows' loads at once (D <= 128), without a condition: rows past the last are the last one again and
    // count nothing.  Behind a branch each load was waited for before the next (8 kv heads of 128, 1 x 4000 keys,
    // 32 - 63 partials: 11.6 -> 10.6 us; 1 x 32000, 250 partials: 36.0 -> 31.4).  Rows asked for twice cost nothing:
    // with as many loads as D needs, four at 64, and v0 not asked for again 1 x 4000 keys of 64 took 8.6 us, so 8.5.
    constexpr int U = 8;
    if (row_lane) {
      for (int r0 = rg; r0 < n; r0 += U * RG) {
        f32x4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
          v[u] = *(const f32x4*)(p.ws_o + (slot0 + s0 + min(r0 + u * RG, n - 1)) * D + 4 * d4);
        if (s0 == 0 && r0 == rg) v[0] = early[0];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int r = r0 + u * RG;
          const float wr = w_lds[wave][min(r, 63)];
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[i] += r < n ? wr * v[u][i] : 0.0f;
        }
      }
    }
  }
  den = row16_sum(sum_xor16(sum_xor32(den)));
  if (row_lane) *(f32x4*)&acc_lds[rg][4 * d4] = acc;
  __syncthreads();
  if (tid < p.dv) {
    float out = 0.0f;
#pragma unroll
    for (int r = 0; r < RG; ++r) out += acc_lds[r][tid];
    Elem<DT>::store1(p.o, (int64_t)b * p.o_sb + (int64_t)head * p.o_sh + tid, ns > 0 ? out / den : 0.0f);
  }
}

// One workgroup per (kv-head unit, sequence): its W wavefronts take equal runs of the context's
// visible 32-key units and merge their partials in LDS.  No scratch, no second launch.
template <int DT, int D, bool POW2, bool RAGGED, int W>
__global__ __launch_bounds__(64 * W, RAGGED ? 1 : 2) void paged_decode_direct_kernel(const DecodeParams p) {
  using Segment = DecodeSegment<DT, D, POW2, RAGGED, false>;
  constexpr int kPitch = D + 4;  // floats between the O rows of two heads: spreads them over the banks
  static_assert(16 * kPitch * 4 <= Segment::kVtBytes, "a wavefront's O rows fit its V^T tile");
  __shared__ __attribute__((aligned(16))) unsigned char vt[W][Segment::kVtBytes];
  __shared__ float ml_lds[2][W][16];
  const int unit = blockIdx.x, b = blockIdx.y;
  const int kvh = unit / p.hchunks;
  const int hchunk = unit - kvh * p.hchunks;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, c = lane & 15;
  const int hq_local = hchunk * 16 + c;
  const bool head_ok = hq_local < p.group;

  const int ctx = __builtin_amdgcn_readfirstlane(max(p.kv_len[b], 0));
  const int kv_min = first_visible(p, ctx), k0 = kv_min & ~31;
  const int units = (ctx - k0 + 31) >> 5;
  const int u0 = units * wave / W, u1 = units * (wave + 1) / W;
  Segment seg;
  seg.run(p, vt[wave], b, ctx, kvh, kvh * p.group + hq_local, head_ok, k0 + 32 * u0, k0 + 32 * u1, kv_min);
  // O rows into this wavefront's own tile (its LDS operations complete in order)
  float* rows = (float*)vt[wave];
#pragma unroll
  for (int mt = 0; mt < Segment::MT; ++mt) *(f32x4*)(rows + c * kPitch + 16 * mt + 4 * g) = seg.o[mt];
  if (g == 0) {
    ml_lds[0][wave][c] = seg.m_run;
    ml_lds[1][wave][c] = seg.l_run;
  }
  __syncthreads();
  const int heads = min(16, p.group - hchunk * 16);
  for (int i = threadIdx.x; i < heads * (D / 4); i += 64 * W) {
    const int h = i / (D / 4), d4 = i % (D / 4);
    float m = -__builtin_inff();
#pragma unroll
    for (int w = 0; w < W; ++w) m = fmaxf(m, ml_lds[0][w][h]);
    float den = 0.0f;
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float mw = ml_lds[0][w][h];
      const float f = mw == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(mw - m);  // (no keys: weight 0)
      den += f * ml_lds[1][w][h];
      const f32x4 v = *(const f32x4*)((const float*)vt[w] + h * kPitch + 4 * d4);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] += f * v[j];
    }
    const float inv = ctx > 0 ? 1.0f / den : 0.0f;
    const int64_t out = (int64_t)b * p.o_sb + (int64_t)(kvh * p.group + hchunk * 16 + h) * p.o_sh;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (!RAGGED || 4 * d4 + j < p.dv) Elem<DT>::store1(p.o, out + 4 * d4 + j, acc[j] * inv);
  }
}

// Wavefronts per workgroup of the one-launch kernel, 0: the split kernel.
// One workgroup per (sequence, kv-head unit) reads a CU's share of the bandwidth at best, so with few
// workgroups the split is the faster one from about 700 keys of 128 dims on, with its 64-key pieces from about
// 500 keys on (640 of up to 64 dims; direct / split, one sequence of 8 kv heads: 100 keys 4.4 / 7, 320 keys 6.5 /
// 7.1, 448 6.7 / 7.3, 576 8.7 / 7.2, 704 9.0 / 7.2; eight: 448 9.4 / 9.6, 576 10.4 / 9.9; sixteen, for which pieces have
// 128 keys: 576 10.9 / 12.9; 4 kv heads of 64: 576 7.2 / 7.3, 704 7.4 / 7.3).  With most CUs busy it wins up to the lengths where one long context among short
// ones would be the whole time (20 sequences of 16 kv heads, 64 - 1024 keys: 22.7 -> 22.0 us; 250
// of one kv head 23.9 -> 16.3; 128 x 100 keys 20.1 -> 13.4); past 1024 keys mixed lengths cost 3 - 6 %.
// What a sliding window leaves is about the same for every sequence.
// Eight wavefronts pay where the rows are short and a few CUs read many keys (1000 keys of 64 dims,
// one sequence: 9.2 us, with four 10.7).
int direct_waves(int B, int units, int max_ctx, int window, int D, bool short_pieces, int64_t cus) {
  if (D > 128) return 0;
  // (a window of any size up to 2^31 - 1 says "none" as well as -1 does)
  const bool windowed = window > 0 && window < max_ctx - 32;
  const int keys = windowed ? window + 32 : max_ctx;
  const int64_t wgs = (int64_t)B * units;
  const bool few_keys = short_pieces ? keys <= (D <= 64 ? 640 : 512) : (int64_t)keys * D <= 700 * 128;
  const bool busy = keys <= (windowed ? 2048 : 1024) && wgs >= (windowed ? cus / 2 : 3 * cus / 4);
  if (!few_keys && !busy) return 0;
  return D <= 64 && keys > 512 && wgs < cus ? 8 : 4;
}

// Do K and V go past the caches, K in whole lines?  A table without room for more than the 256 MB behind the L2s keeps
// them.  In a larger one it goes by the keys that the contexts have, which the kernel counts anyway: from half of that
// on.  Kept / past, 8 kv heads of 128, each step on other caches, as the layers of a model are: 8 x 1500 keys 22.7 /
// 24.8 us, 8 x 500 - 8000 (111 MB) 27.4 / 27.2, 32 x 500 - 2000 (145 MB) 37.4 / 34.9, 16 x 500 - 8000 48.2 / 45.9,
// 64 x 512 - 8192 169.0 / 160.7.  On the same keys over and over, which the caches then partly hold, 111 MB 25.1 / 26.5,
// 145 MB 33.2 / 33.3, 215 MB 44.3 / 45.4, and 256 x 100 - 300 52.3 / 57.5 (on others 63.2 / 58.5).
constexpr int64_t kCacheBytes = (int64_t)256 << 20;
bool may_read_once(int B, int Hkv, int dims, int max_ctx, int window) {
  const int64_t keys = window > 0 && window < max_ctx ? window : max_ctx;
  return (int64_t)B * keys * Hkv * dims * 2 > kCacheBytes;
}
int once_units(int Hkv, int dims) { return (int)(kCacheBytes / 2 / ((int64_t)32 * Hkv * dims * 2)); }

// Smallest piece a team may get, in 32-key units: 512 keys, less for small problems so that
// the chip still sees a few thousand wavefronts.  64 keys, two steps of a wavefront, where that leaves each CU
// at most four of them and a head at most 64 partials, or 65 where pieces cross sequences (128 / 64 keys, measured with
// another merge: 8 kv heads of 128, 1 x 2000 11.1 / 9.4 us, 8 x 2000 18.2 / 19.1, 1 x 8000 14.5 / 17.1; of 64, 1 x 4000
// 11.3 / 9.7).
// 64-key pieces need twice the scratch; a call that brings less, say what a larger batch or a wider table with its
// longer pieces needs, gets 128-key ones.
int pick_min_units(int B, int Hkv, int hchunks, int max_ctx, bool short_pieces, int64_t cus) {
  const int64_t units = (int64_t)B * Hkv * hchunks;
  auto pieces = [&](int keys) { return ((int64_t)max_ctx + keys - 1) / keys; };
  int kps = 512;
  while (kps > 128 && units * pieces(kps) < 4096) kps >>= 1;
  if (short_pieces && kps == 128 && pieces(64) <= 64 && units * pieces(64) <= 4 * cus) kps = 64;
  return kps / 32;
}

// partial slots per (sequence, head): a sequence of T units cut into pieces of >= min_units
// overlaps at most T / min_units + 2 of them
int partial_slots(int max_ctx, int min_units) {
  const int t = (max_ctx + 31) / 32;
  return t / min_units + 2;
}

// One sequence whose teams all have pieces of min_units units, whatever its context is, and at most 64 pages per piece
bool one_sequence(int B, int max_ctx, int min_units, int num_teams, int window) {
  return B == 1 && window <= 0 && (max_ctx + 31) / 32 <= (int64_t)num_teams * min_units && min_units <= 16;
}

size_t scratch_bytes(int B, int Hq, int D, int max_ctx, int min_units) {
  return (size_t)B * Hq * partial_slots(max_ctx, min_units) * (D + 2) * sizeof(float) + (size_t)B * sizeof(int32_t);
}

// teams that are resident together: wavefronts per CU (2 per SIMD, 1 in the masked variant) /
// wavefronts per team
int pick_num_teams(int units_per_team, bool ragged, int cus) {
  return max(1, cus * (ragged ? 4 : 8) / units_per_team);
}

// head size the kernel instance is built for; past 128 one instance, for 256, takes every size on
// its masked path
int padded_head_size(int D, int Dv) {
  const int d = D > Dv ? D : Dv;
  return d <= 64 ? 64 : d <= 96 ? 96 : d <= 128 ? 128 : 256;
}

}  // namespace
}  // namespace dlb

extern "C" size_t dlb_paged_decode_ws_bytes(int B, int Hq, int Hkv, int D, int page,
                                            int max_blocks) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || D <= 0 || D > 256 || page <= 0 || max_blocks <= 0) return 0;
  D = dlb::padded_head_size(D, D);
  const int group = Hq / Hkv;
  const int hchunks = (group + 15) / 16;
  const int64_t max_ctx = (int64_t)page * max_blocks;
  if (max_ctx > 0x7fffffff) return 0;
  return dlb::scratch_bytes(B, Hq, D, (int)max_ctx, dlb::pick_min_units(B, Hkv, hchunks, (int)max_ctx, true,
                                                                         dlb::current_device_cu_count()));
}

extern "C" int dlb_paged_decode_attn(const void* q, const void* k_cache, const void* v_cache,
                                     void* o, const void* block_table, const void* kv_len,
                                     int index64_mask, int B, int Hq, int Hkv, int D, int Dv, int page,
                                     int max_blocks, int64_t q_stride_b, int64_t q_stride_h, int64_t k_stride_page,
                                     int64_t k_stride_tok, int64_t k_stride_head,
                                     int64_t v_stride_page, int64_t v_stride_tok,
                                     int64_t v_stride_head, int64_t o_stride_b, int64_t o_stride_h,
                                     int64_t bt_stride, float sm_scale, int window_size,
                                     float logit_softcapping, int dtype, void* ws,
                                     size_t ws_bytes, void* stream) {
  using namespace dlb;
  if (B < 0 || Hq < 1 || Hkv < 1 || D < 1 || Dv < 1 || page < 1 || max_blocks < 1) return DLB_ERR_BAD_ARG;
  if (Hq % Hkv != 0) return DLB_ERR_BAD_ARG;
  if (B == 0) return DLB_OK;
  if (!q || !k_cache || !v_cache || !o || !block_table || !kv_len) return DLB_ERR_BAD_ARG;
  if (D % 8 != 0 || Dv % 8 != 0 || D > 256 || Dv > 256) return DLB_ERR_UNSUPPORTED;
  const int Dp = padded_head_size(D, Dv);
  const bool ragged = D != Dp || Dv != Dp || Dp == 256;
  if (page % 16 != 0) return DLB_ERR_UNSUPPORTED;
  if (dtype != DLB_DTYPE_BF16 && dtype != DLB_DTYPE_F16) return DLB_ERR_UNSUPPORTED;
  if ((int64_t)page * max_blocks > 0x7fffffff) return DLB_ERR_UNSUPPORTED;
  // per-lane byte offsets inside a page are 32-bit
  if ((int64_t)page * k_stride_tok * 2 > 0x7fffffff || (int64_t)page * v_stride_tok * 2 > 0x7fffffff)
    return DLB_ERR_UNSUPPORTED;
  // 128-bit operand loads
  if (!aligned16(q) || !aligned16(k_cache) || !aligned16(v_cache)) return DLB_ERR_UNSUPPORTED;
  const int64_t strides[] = {q_stride_b,   q_stride_h,    k_stride_page, k_stride_tok,
                             k_stride_head, v_stride_page, v_stride_tok,  v_stride_head};
  for (int64_t sd : strides)
    if (sd % 8 != 0) return DLB_ERR_UNSUPPORTED;
  const int max_ctx = page * max_blocks, cus = current_device_cu_count();
  DecodeParams p;
  p.group = Hq / Hkv;
  p.hchunks = (p.group + 15) / 16;
  p.min_units = pick_min_units(B, Hkv, p.hchunks, max_ctx, true, cus);
  if (ws_bytes < scratch_bytes(B, Hq, Dp, max_ctx, p.min_units))
    p.min_units = pick_min_units(B, Hkv, p.hchunks, max_ctx, false, cus);
  if (!ws || ws_bytes < scratch_bytes(B, Hq, Dp, max_ctx, p.min_units)) return DLB_ERR_WORKSPACE;
  p.nsplit_max = partial_slots(max_ctx, p.min_units);
  p.q = q;
  p.k = k_cache;
  p.v = v_cache;
  p.o = o;
  if (index64_mask & ~3) return DLB_ERR_BAD_ARG;
  p.block_table = idx_array(block_table, index64_mask, 0);
  p.kv_len = idx_array(kv_len, index64_mask, 1);
  p.q_sb = q_stride_b;
  p.q_sh = q_stride_h;
  p.k_sp = k_stride_page;
  p.k_st = k_stride_tok;
  p.k_sh = k_stride_head;
  p.v_sp = v_stride_page;
  p.v_st = v_stride_tok;
  p.v_sh = v_stride_head;
  p.o_sb = o_stride_b;
  p.o_sh = o_stride_h;
  p.bt_stride = bt_stride;
  p.B = B;
  p.Hq = Hq;
  p.Hkv = Hkv;
  p.page = page;
  p.page_shift = -1;
  for (int sh = 0; sh < 31; ++sh)
    if ((1 << sh) == page) p.page_shift = sh;
  p.max_blocks = max_blocks;
  p.scale_log2e = sm_scale * 1.4426950408889634f;
  p.sm_scale = sm_scale;
  p.window = window_size;
  p.softcap = logit_softcapping;
  p.dk = D;
  p.dv = Dv;
  p.ws_o = (float*)ws;
  p.ws_ml = p.ws_o + (size_t)B * Hq * p.nsplit_max * Dp;
  p.ws_np = (int32_t*)(p.ws_ml + (size_t)B * Hq * p.nsplit_max * 2);

  hipStream_t s = (hipStream_t)stream;
  const int units = Hkv * p.hchunks;
  p.num_teams = pick_num_teams(units, ragged, cus);
  if (units > 65535 || p.num_teams > 65535 || B > 65535) return DLB_ERR_UNSUPPORTED;
  const dim3 grid1((uint32_t)units, (uint32_t)p.num_teams);
  const dim3 grid2((uint32_t)Hq, (uint32_t)B), grid_direct((uint32_t)units, (uint32_t)B);
  const int direct = direct_waves(B, units, max_ctx, window_size, Dp, p.min_units == 2, cus);
  p.once_units = once_units(Hkv, D + Dv);
  const bool one = one_sequence(B, max_ctx, p.min_units, p.num_teams, window_size);
  const bool early = (int64_t)B * Hq <= cus;
  const bool choice = may_read_once(B, Hkv, D + Dv, max_ctx, window_size);
#define DLB_LAUNCH_SPLIT(DT_, D_, P2_, RG_)                                                                       \
  do {                                                                                                            \
    if (direct == 4)                                                                                              \
      launch((paged_decode_direct_kernel<DT_, D_, P2_, RG_, 4>), grid_direct, dim3(256), s, p);    \
    else if (D_ == 64 && direct == 8)                                                                             \
      launch((paged_decode_direct_kernel<DT_, 64, P2_, RG_, 8>), grid_direct, dim3(512), s, p);    \
    else if (D_ % 64 == 0 && !RG_ && choice)                                                                      \
      launch((paged_decode_split_kernel<DT_, D_, P2_, RG_, D_ % 64 == 0 && !RG_, false>), grid1, dim3(64), s, p); \
    else if (one)                                                                                                 \
      launch((paged_decode_split_kernel<DT_, D_, P2_, RG_, false, true>), grid1, dim3(64), s, p);  \
    else                                                                                                          \
      launch((paged_decode_split_kernel<DT_, D_, P2_, RG_, false, false>), grid1, dim3(64), s, p); \
  } while (0)
#define DLB_LAUNCH_DECODE(DT_, D_)                                                                           \
  do {                                                                                                       \
    if (p.page_shift >= 0) {                                                                                 \
      if (ragged) DLB_LAUNCH_SPLIT(DT_, D_, true, true);                                                     \
      else DLB_LAUNCH_SPLIT(DT_, D_, true, false);                                                           \
    } else {                                                                                                 \
      if (ragged) DLB_LAUNCH_SPLIT(DT_, D_, false, true);                                                    \
      else DLB_LAUNCH_SPLIT(DT_, D_, false, false);                                                          \
    }                                                                                                        \
    if (!direct && early)                                                                                    \
      launch((paged_decode_combine_kernel<DT_, D_, true>), grid2, dim3(kCombineThreads), s, p); \
    else if (!direct)                                                                                        \
      launch((paged_decode_combine_kernel<DT_, D_, false>), grid2, dim3(kCombineThreads), s, p); \
  } while (0)
#define DLB_LAUNCH_DECODE_256(DT_)                                                                           \
  do {                                                                                                       \
    if (p.page_shift >= 0)                                                                                   \
      launch((paged_decode_split_kernel<DT_, 256, true, true, false, false>), grid1, dim3(64), s, p);        \
    else                                                                                                     \
      launch((paged_decode_split_kernel<DT_, 256, false, true, false, false>), grid1, dim3(64), s, p);       \
    launch((paged_decode_combine_kernel<DT_, 256, false>), grid2, dim3(kCombineThreads), s, p);       \
  } while (0)
#define DLB_DISPATCH_DECODE(DT_)                        \
  do {                                                  \
    if (Dp == 256) DLB_LAUNCH_DECODE_256(DT_);          \
    else if (Dp == 128) DLB_LAUNCH_DECODE(DT_, 128);    \
    else if (Dp == 96) DLB_LAUNCH_DECODE(DT_, 96);      \
    else DLB_LAUNCH_DECODE(DT_, 64);                    \
  } while (0)
  if (dtype == DLB_DTYPE_BF16) DLB_DISPATCH_DECODE(DLB_DTYPE_BF16);
  else DLB_DISPATCH_DECODE(DLB_DTYPE_F16);
#undef DLB_DISPATCH_DECODE
#undef DLB_LAUNCH_DECODE_256
#undef DLB_LAUNCH_DECODE
#undef DLB_LAUNCH_SPLIT
  return launch_status();
}
