// Shared device/host helpers for the gfx950 kernels of libdlblas_hip.so.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "../../include/dlblas_hip.h"

namespace dlb {

constexpr int kWave = 64;  // CDNA wavefront width

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
typedef __attribute__((ext_vector_type(8))) int i32x8;

// ---- bf16 / f16 <-> f32 scalar conversions on raw 16-bit patterns -----------------------
__device__ __forceinline__ float bf16_bits_to_f32(unsigned int b) {
  return __uint_as_float(b << 16);
}
// round-to-nearest-even, NaN kept quiet
__device__ __forceinline__ unsigned int f32_to_bf16_bits(float f) {
  unsigned int u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;
  u += 0x7fffu + ((u >> 16) & 1u);
  return u >> 16;
}
__device__ __forceinline__ float f16_bits_to_f32(unsigned int b) {
  _Float16 h = __builtin_bit_cast(_Float16, (unsigned short)b);
  return (float)h;
}
__device__ __forceinline__ unsigned int f32_to_f16_bits(float f) {
  _Float16 h = (_Float16)f;  // v_cvt_f16_f32: RNE
  return (unsigned int)__builtin_bit_cast(unsigned short, h);
}

template <int DT>
struct Elem;
template <>
struct Elem<DLB_DTYPE_BF16> {
  static __device__ __forceinline__ float lo(unsigned int w) { return __uint_as_float(w << 16); }
  static __device__ __forceinline__ float hi(unsigned int w) {
    return __uint_as_float(w & 0xffff0000u);
  }
  // two floats -> two bf16 in one word: v_cvt_pk_bf16_f32 (round to nearest even, NaN quiet)
  static __device__ __forceinline__ unsigned int pack(float a, float b) {
    typedef __attribute__((ext_vector_type(2))) float f2;
    typedef __attribute__((ext_vector_type(2))) __bf16 b2;
    const f2 f = {a, b};
    return __builtin_bit_cast(unsigned int, __builtin_convertvector(f, b2));
  }
  static __device__ __forceinline__ float load1(const void* p, int64_t i) {
    return bf16_bits_to_f32(((const unsigned short*)p)[i]);
  }
  static __device__ __forceinline__ void store1(void* p, int64_t i, float v) {
    ((unsigned short*)p)[i] = (unsigned short)f32_to_bf16_bits(v);
  }
};
template <>
struct Elem<DLB_DTYPE_F16> {
  static __device__ __forceinline__ float lo(unsigned int w) { return f16_bits_to_f32(w & 0xffffu); }
  static __device__ __forceinline__ float hi(unsigned int w) { return f16_bits_to_f32(w >> 16); }
  static __device__ __forceinline__ unsigned int pack(float a, float b) {
    typedef __attribute__((ext_vector_type(2))) float f2;
    typedef __attribute__((ext_vector_type(2))) _Float16 h2;
    const f2 f = {a, b};
    return __builtin_bit_cast(unsigned int, __builtin_convertvector(f, h2));
  }
  static __device__ __forceinline__ float load1(const void* p, int64_t i) {
    return f16_bits_to_f32(((const unsigned short*)p)[i]);
  }
  static __device__ __forceinline__ void store1(void* p, int64_t i, float v) {
    ((unsigned short*)p)[i] = (unsigned short)f32_to_f16_bits(v);
  }
};

// ---- DPP cross-lane moves within a row of 16 lanes ---------------------------------------
// dpp_ctrl encodings (GCN3+/CDNA): quad_perm = 0x00..0xff, row_mirror = 0x140,
// row_half_mirror = 0x141.
constexpr int kDppQuadXor1 = 0xB1;  // quad_perm [1,0,3,2]
constexpr int kDppQuadXor2 = 0x4E;  // quad_perm [2,3,0,1]
constexpr int kDppRowHalfMirror = 0x141;
constexpr int kDppRowMirror = 0x140;

template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ unsigned int dpp_u32(unsigned int v) {
  return (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}

// all-reduce over each aligned group of 16 lanes (a DPP row); every lane gets the result.
// After the two quad steps all lanes of a quad agree, so the mirror steps (i <-> 7-i,
// i <-> 15-i) complete a butterfly for any commutative, associative, idempotent-or-not op:
// each step combines two disjoint halves whose members already hold their half's result.
__device__ __forceinline__ float row16_max(float v) {
  v = fmaxf(v, dpp_f32<kDppQuadXor1>(v));
  v = fmaxf(v, dpp_f32<kDppQuadXor2>(v));
  v = fmaxf(v, dpp_f32<kDppRowHalfMirror>(v));
  v = fmaxf(v, dpp_f32<kDppRowMirror>(v));
  return v;
}
__device__ __forceinline__ float row16_sum(float v) {
  v += dpp_f32<kDppQuadXor1>(v);
  v += dpp_f32<kDppQuadXor2>(v);
  v += dpp_f32<kDppRowHalfMirror>(v);
  v += dpp_f32<kDppRowMirror>(v);
  return v;
}

// inclusive prefix sum over the 64 lanes of a wave with DPP moves only (shifts inside each row
// of 16 lanes, then the row totals broadcast to the rows after them): no LDS round trips and no
// per-lane address registers, which a shuffle-based scan keeps live across the whole kernel
__device__ __forceinline__ int wave_inclusive_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 -> rows 1, 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 -> rows 2, 3
  return v;
}

// a pointer the caller knows to be wave-uniform, moved into scalar registers
__device__ __forceinline__ const unsigned char* uniform_ptr(const unsigned char* p) {
  const uint64_t v = (uint64_t)(uintptr_t)p;
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
  return (const unsigned char*)(uintptr_t)(((uint64_t)hi << 32) | lo);
}
// descriptor of `bytes` bytes at p (wave-uniform): raw buffer, no swizzle, loads past the end give 0
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(uniform_ptr((const unsigned char*)p)), 0,
                                           (int)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000);
}

// wave-uniform LDS byte address of a pointer into __shared__ memory, in a scalar register
__device__ __forceinline__ unsigned int lds_addr(const void* p) {
  typedef const __attribute__((address_space(3))) void* lds_ptr_t;
  return (unsigned int)__builtin_amdgcn_readfirstlane((int)(uintptr_t)(lds_ptr_t)p);
}
// Direct global -> LDS copy of 16 bytes per lane: lane l's bytes land at lds_base + 16 * l
// (lds_base: wave-uniform LDS byte address).  Issued through inline assembly rather than
// __builtin_amdgcn_global_load_lds because the compiler's wait-count pass models the builtin as
// a FLAT access that may complete out of order with LDS reads: while one is in flight every
// LDS wait it inserts becomes lgkmcnt(0), which serialises a pipelined ds_read -> MFMA stream.
// The copy is counted by vmcnt like any other vector load (loads return in order); the compiler
// does not see it, so the caller waits for it explicitly (s_waitcnt vmcnt) before the barrier
// that publishes the data.  Waits the compiler inserts for its own loads stay correct: an
// unseen load that is older completes first, one that is younger only makes the wait longer.
// The helpers write m0 and say so in their clobber lists, so the compiler never keeps a live
// value of its own (an LDS-direct or indexed-register base) in m0 across one of them.
__device__ __forceinline__ void dma16_global_to_lds(const void* gsrc, unsigned int lds_base) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               :
               : "v"(gsrc), "s"(__builtin_amdgcn_readfirstlane((int)lds_base))
               : "memory", "m0");
}

// same copy, addressed as a wave-uniform 64-bit base (scalar registers) plus a 32-bit lane offset
__device__ __forceinline__ void dma16_global_to_lds(const void* sbase, unsigned int voff,
                                                    unsigned int lds_base) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(voff), "s"(sbase), "s"(__builtin_amdgcn_readfirstlane((int)lds_base))
               : "memory", "m0");
}

// the 4-byte form: lane l's dword lands at lds_base + 4 * l
__device__ __forceinline__ void dma4_global_to_lds(const void* gsrc, unsigned int lds_base) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off"
               :
               : "v"(gsrc), "s"(__builtin_amdgcn_readfirstlane((int)lds_base))
               : "memory", "m0");
}

// the 4-byte form restricted to the lanes of `lane_mask` (a compile-time constant); the other
// lanes neither read nor write
template <unsigned long long lane_mask>
__device__ __forceinline__ void dma4_global_to_lds_masked(const void* gsrc, unsigned int lds_base) {
  unsigned long long saved;
  asm volatile("s_mov_b64 %0, exec\n\ts_mov_b64 exec, %3\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\t"
               "global_load_lds_dword %1, off\n\ts_mov_b64 exec, %0"
               : "=&s"(saved)
               : "v"(gsrc), "s"(__builtin_amdgcn_readfirstlane((int)lds_base)), "s"(lane_mask)
               : "memory", "m0");
}

// ds_read_b64_tr_b16: every lane passes the address of four consecutive 16-bit elements; in
// each group of 16 lanes the 16 x 4 elements form a 4-row x 16-column block (row j = lanes
// 4j .. 4j+3 of the group, four columns each) and lane l of the group receives column l,
// rows 0..3, lowest row in the low half of the first register.
__device__ __forceinline__ u32x2 lds_read_tr16(const void* p) {
  typedef __attribute__((ext_vector_type(4))) short s16x4;
  typedef __attribute__((address_space(3))) s16x4* lds_s16x4_ptr;
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)p));
}

// the masked 4-byte form addressed as a wave-uniform 64-bit base plus a 32-bit lane offset
template <unsigned long long lane_mask>
__device__ __forceinline__ void dma4_global_to_lds_masked(const void* sbase, unsigned int voff,
                                                          unsigned int lds_base) {
  unsigned long long saved;
  asm volatile("s_mov_b64 %0, exec\n\ts_mov_b64 exec, %4\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\t"
               "global_load_lds_dword %1, %2\n\ts_mov_b64 exec, %0"
               : "=&s"(saved)
               : "v"(voff), "s"(sbase), "s"(__builtin_amdgcn_readfirstlane((int)lds_base)),
                 "s"(lane_mask)
               : "memory", "m0");
}

// Around non-temporal stores on one side of a condition whose other side makes the same stores through the caches:
// the compiler would make them one, without the hint.
__device__ __forceinline__ void keep_apart() { asm volatile("" ::: "memory"); }

// a value and its partner 16 / 32 lanes away combined (v_permlane16_swap, v_permlane32_swap: register-file
// exchanges, no trip through LDS as with ds_bpermute)
typedef __attribute__((ext_vector_type(2))) unsigned int permlane_pair;
__device__ __forceinline__ permlane_pair lanes_xor16(float v) {
  return __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
}
__device__ __forceinline__ permlane_pair lanes_xor32(float v) {
  return __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
}
__device__ __forceinline__ float max_of(permlane_pair r) { return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])); }
__device__ __forceinline__ float sum_of(permlane_pair r) { return __uint_as_float(r[0]) + __uint_as_float(r[1]); }
__device__ __forceinline__ float max_xor16(float v) { return max_of(lanes_xor16(v)); }
__device__ __forceinline__ float max_xor32(float v) { return max_of(lanes_xor32(v)); }
__device__ __forceinline__ float sum_xor16(float v) { return sum_of(lanes_xor16(v)); }
__device__ __forceinline__ float sum_xor32(float v) { return sum_of(lanes_xor32(v)); }

// tanh for the logit soft-cap: no less accurate than tanhf, in half its instructions and without a branch.
// Below 0.85 an odd polynomial (least squares on Chebyshev nodes, reweighted towards the smallest
// largest relative error, 8e-9); from there on the term in 1 - 2 / (e^2|x| + 1), whose exponential and
// reciprocal are each up to an ulp off, is at most a third of the result.  Against 64 bits over all
// floats in [0.2, 1) and every seventh in [2^-10, 16), either sign: largest relative error 1.1e-7,
// 1.30 ulp, root mean square 0.30 ulp; tanhf 1.5e-7, 1.41 and 0.32; a seam at 0.25 6.3e-7, 10.2 and 1.2.
// (tanhf is two branches, and a wave whose scores lie on both sides walks both: 8 x 512 tokens over 4096, every
// tile capped, 581 us where all scores are small and 804 us where they are not; this one 645 us throughout.)
constexpr float kSoftcapSmall = 0.85f;
__device__ __forceinline__ float softcap_tanh_small(float x) {
  const float z = x * x;
  float c = 0.0014401802327483892f;
  c = fmaf(z, c, -0.007142828777432442f);
  c = fmaf(z, c, 0.02112109400331974f);
  c = fmaf(z, c, -0.05379646271467209f);
  c = fmaf(z, c, 0.13331478834152222f);
  c = fmaf(z, c, -0.3333326578140259f);
  return fmaf(x * z, c, x);
}
__device__ __forceinline__ float softcap_tanh(float x) {
  const float a = fabsf(x), poly = softcap_tanh_small(x);
  // e2 = 2 e^-2|x|: 1 - e2 / (1 + e2 / 2)
  const float e2 = __builtin_amdgcn_exp2f(fmaf(a, -2.8853900817779268f, 1.0f));
  const float big = fmaf(-e2, __builtin_amdgcn_rcpf(fmaf(0.5f, e2, 1.0f)), 1.0f);
  return a < kSoftcapSmall ? poly : copysignf(big, x);
}
__host__ __device__ __forceinline__ int64_t ceil_div(int64_t a, int64_t b) {
  return (a + b - 1) / b;
}

// Index arrays (sequence lengths, start offsets, block tables) arrive as int32 or as int64, as the
// caller's framework holds them; element i is read as the 32-bit word i << sh (sh = 1: the low
// half of a little-endian int64 -- the values are token counts and page numbers below 2^31).
struct IdxArray {
  const int32_t* p;
  int sh;
  __device__ __forceinline__ int operator[](int64_t i) const { return p[i << sh]; }
};
inline IdxArray idx_array(const void* p, int index64_mask, int bit) {
  return IdxArray{(const int32_t*)p, (index64_mask >> bit) & 1};
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// compute units of the device that is current on this thread (256 if it cannot be read), kept
// per device: a process may drive GPUs of different sizes.  The table is filled lazily; two
// threads racing on one entry write the same value.
inline int current_device_cu_count() {
  constexpr int kMaxDevices = 64;
  static std::atomic<int> table[kMaxDevices];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 256;
  int n = table[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    table[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Launches `kernel`.  A launch is most of what a small call costs: 2.3 us here, 2.5 through <<<>>>, which pushes the
// configuration onto a stack of the runtime's and has the kernel's stub pop it again.
template <typename T>
struct AsIs {
  typedef T type;
};
template <typename... A>
inline void launch(void (*kernel)(A...), dim3 grid, dim3 block, hipStream_t s, typename AsIs<A>::type... args) {
  void* ptrs[] = {(void*)&args...};
  (void)hipLaunchKernel((const void*)kernel, grid, block, ptrs, 0, s);
}
// status of the launch just issued on this thread
inline int launch_status() { return hipGetLastError() == hipSuccess ? DLB_OK : DLB_ERR_LAUNCH; }

}  // namespace dlb
