// Pieces shared by the rank-r passes (lora_skinny.hip, lora_da_direct.hip, lora_stream.hip): routing of a 128-row block, MFMA wrapper,
// keep-mask arithmetic, sums of fp32 partials, and the direct-to-LDS loads with their counted waits (internal).
#pragma once
#include "lf_common.h"
#include "philox.h"

namespace {

constexpr int ROWS = 128;  // rows per workgroup = one routing block

template <typename T> struct Mfma16;
template <> struct Mfma16<__bf16> {
  static __device__ __forceinline__ lf_f32x4 run(lf_u32x4 a, lf_u32x4 b, lf_f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(lf_bf16x8, a), __builtin_bit_cast(lf_bf16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint16_t cvt(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
};
template <> struct Mfma16<_Float16> {
  static __device__ __forceinline__ lf_f32x4 run(lf_u32x4 a, lf_u32x4 b, lf_f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(lf_f16x8, a), __builtin_bit_cast(lf_f16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint16_t cvt(float f) { return __builtin_bit_cast(uint16_t, (_Float16)f); }
};

struct BlockInfo {
  int rank, valid, seg;
  float scale, p;
};

// Routing of the 128-row block `blk` (wave-uniform).
__device__ __forceinline__ BlockInfo block_info(const LfSegTable& seg, int blk, int M) {
  BlockInfo b;
  if (seg.table == nullptr) {
    b.rank = seg.rank[0];
    b.valid = min(ROWS, M - blk * ROWS);
    b.seg = 0;
    b.scale = seg.scale;
    b.p = seg.p;
  } else {
    b.rank = seg.table[3 * blk + 0];
    b.valid = seg.table[3 * blk + 1];
    const int fb = seg.table[3 * blk + 2];
    int s = 0;
    for (int i = 1; i < seg.n_seg; i++) s = (seg.first_block[i] == fb) ? i : s;
    b.seg = s;
    b.scale = seg.block_scale ? seg.block_scale[blk] : 1.f;
    b.p = seg.block_p ? seg.block_p[blk] : 0.f;
  }
  return b;
}

// keep ? x : 0 on 8 packed 16-bit elements given their 8 mask bytes.
__device__ __forceinline__ lf_u32x4 apply_mask8(lf_u32x4 x, lf_u32x2 m) {
  lf_u32x4 r;
#pragma unroll
  for (int d = 0; d < 4; d++) {
    const uint32_t mw = d < 2 ? m[0] : m[1];
    const uint32_t two = (mw >> (16 * (d & 1))) & 0xffffu;           // bytes (2d, 2d+1)
    const uint32_t sel = ((two & 0xffu) ? 0x0000ffffu : 0u) | ((two & 0xff00u) ? 0xffff0000u : 0u);
    r[d] = x[d] & sel;
  }
  return r;
}

// The direct-to-LDS loads of a keep-mask fetch 4 bytes of bits or 16 bytes of bytes at a time: a mask that does not lie on such an address is
// read by each lane for itself.
inline bool mask_off_grid(const uint8_t* mask, int mask_bits) { return mask != nullptr && ((uintptr_t)mask & (mask_bits ? 3 : 15)) != 0; }
__device__ __forceinline__ lf_u32x2 keep_bytes8(const uint8_t* p) {
  lf_u32x2 m;
  __builtin_memcpy(&m, p, 8);
  return m;
}

// Bit-packed keep-masks: element k of a row = bit k & 7 of byte k >> 3 of the row (K / 8 bytes per row).
// The eight keep bytes (0/1 each, `lo` = the first four) as eight bits, and back: one multiply gathers / spreads four
// single bits (no two partial products meet in one bit position, so nothing carries).
__device__ __forceinline__ uint32_t pack_keep8(uint32_t lo, uint32_t hi) {
  return ((lo * 0x01020408u) >> 24) | (((hi * 0x01020408u) >> 24) << 4);
}
__device__ __forceinline__ lf_u32x2 expand_keep8(uint32_t b) {
  return lf_u32x2{((b & 0xfu) * 0x00204081u) & 0x01010101u, (((b >> 4) & 0xfu) * 0x00204081u) & 0x01010101u};
}

// keep bits of 8 elements as four dword selectors
__device__ __forceinline__ lf_u32x4 select8(uint32_t bits) {
  lf_u32x4 m;
#pragma unroll
  for (int d = 0; d < 4; d++) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_sbfe((int)bits, 2 * d, 1), hi = (uint32_t)__builtin_amdgcn_sbfe((int)bits, 2 * d + 1, 1);
    m[d] = (lo & 0xffffu) | (hi & 0xffff0000u);
  }
  return m;
}

// The eight draws of a counter against the threshold (>= 1): selectors, and the keep bits.  Two draws per packed 16-bit
// operation: draw -sat (thr - 1) is non-zero exactly where draw >= thr.
__device__ __forceinline__ lf_u32x4 draw8(uint64_t ctr, uint32_t thr, uint32_t seed_lo, uint32_t seed_hi, uint32_t& bits) {
  typedef uint16_t us2 __attribute__((ext_vector_type(2)));
  uint32_t w[4];
  lf_philox4x32_10((uint32_t)ctr, (uint32_t)(ctr >> 32), 0u, 0u, seed_lo, seed_hi, w);
  const uint16_t t1 = (uint16_t)(thr - 1);
  const us2 thr2 = {t1, t1}, one = {1, 1}, zero = {0, 0};
  lf_u32x4 m;
  uint32_t v = 0;
#pragma unroll
  for (int d = 0; d < 4; d++) {
    const us2 k = __builtin_elementwise_min(__builtin_elementwise_sub_sat(__builtin_bit_cast(us2, w[d]), thr2), one);
    m[d] = __builtin_bit_cast(uint32_t, (us2)(zero - k));
    v |= __builtin_bit_cast(uint32_t, k) << (2 * d);
  }
  bits = (v | (v >> 15)) & 0xffu;   // even draws at bits 0, 2, 4, 6, odd draws at 16, 18, ...
  return m;
}

// Sum of `n` fp32x4 partials `stride` floats apart, in index order (deterministic).
__device__ __forceinline__ lf_f32x4 sum_parts(const float* __restrict__ p, int64_t stride, int n) {
  // Up to sixteen partials are requested before the first is added: these second stages are short launches whose
  // time is the chain of memory round trips of one thread, and with four loads in flight a sum of sixteen was four
  // round trips long (5 us for a few hundred KB).  The order of the additions is the index order either way.
  lf_f32x4 v = {0.f, 0.f, 0.f, 0.f};
  int i = 0;
  for (; i + 16 <= n; i += 16) {
    lf_f32x4 t[16];
#pragma unroll
    for (int k = 0; k < 16; k++) t[k] = *(const lf_f32x4*)(p + (int64_t)(i + k) * stride);
#pragma unroll
    for (int k = 0; k < 16; k++) v += t[k];
  }
  if (i < n) {
    lf_f32x4 t[16];
#pragma unroll
    for (int k = 0; k < 16; k++) t[k] = (i + k < n) ? *(const lf_f32x4*)(p + (int64_t)(i + k) * stride) : lf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 16; k++) v += t[k];   // (adding the zeros beyond n changes nothing: x + 0 = x, and -0 cannot arise from a sum that started at +0)
  }
  return v;
}
template <typename T>
__device__ __forceinline__ lf_u32x2 pack4(lf_f32x4 v) {
  return lf_u32x2{(uint32_t)Mfma16<T>::cvt(v[0]) | ((uint32_t)Mfma16<T>::cvt(v[1]) << 16),
                  (uint32_t)Mfma16<T>::cvt(v[2]) | ((uint32_t)Mfma16<T>::cvt(v[3]) << 16)};
}

// A product that is rounded to fp32 before anything else happens to it.  The compiler folds fp32 multiply and conversion to fp16 into one
// instruction (v_fma_mixlo_f16), which rounds once where the two round twice: kernels that have to agree bit for bit would not.
__device__ __forceinline__ float fp32_product(float a, float b) {
  float v = a * b;
  asm("" : "+v"(v));
  return v;
}

__device__ __forceinline__ uint32_t to_sgpr(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

__device__ __forceinline__ lf_u32x4 window_rsrc(const void* base, int64_t bytes) {
  const uint64_t a = (uint64_t)(uintptr_t)base;
  const int64_t n = bytes > 0xffffffffll ? 0xffffffffll : bytes;   // (never negative: a window starts inside its matrix)
  return lf_u32x4{to_sgpr((uint32_t)a), to_sgpr((uint32_t)(a >> 32)) & 0xffffu, to_sgpr((uint32_t)n), 0x00020000u};
}
// one wave instruction: lane l fetches 16 bytes at window offset `voff` into LDS byte lds_addr + 16 l
__device__ __forceinline__ void dma16(const lf_u32x4& rsrc, uint32_t voff, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds_addr), "v"(voff), "s"(rsrc) : "memory");
}
// one wave instruction: lane l fetches 4 bytes at window offset `voff` into LDS byte lds_addr + 4 l
__device__ __forceinline__ void dma4(const lf_u32x4& rsrc, uint32_t voff, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds" ::"s"(lds_addr), "v"(voff), "s"(rsrc) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// at most `groups` groups of G operations each may still be outstanding (above four: four; a ring with more stages on order would not use them)
constexpr int WAIT_MOST = 4;
template <int G>
__device__ __forceinline__ void wait_groups(int groups) {
  switch (groups) {
    case 0: wait_vm<0>(); break;
    case 1: wait_vm<G>(); break;
    case 2: wait_vm<2 * G>(); break;
    case 3: wait_vm<3 * G>(); break;
    default: wait_vm<WAIT_MOST * G>(); break;
  }
}
__device__ __forceinline__ void ring_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

int rt_of(int R) { return R <= 16 ? 1 : R <= 32 ? 2 : R <= 64 ? 4 : 8; }

int n_row_blocks(int M, const LfSegTable& seg) { return seg.table ? seg.n_blocks : (M + ROWS - 1) / ROWS; }

int lds_slots(int smem_bytes) {
  const int per_cu = (160 * 1024) / smem_bytes;
  return 256 * (per_cu > 0 ? per_cu : 1);
}

}  // namespace
