// MFMA GEMM for outputs of about one round of the chip, with the LoRA term added behind the K loop, for gfx950 (MI355X).
//
//   C[M,N] = A[M,K] * op(B) + mult * (L[M,R] * Rop) (+ bias)        (operands as in gemm_lora.hip)
//
// Stands in, for short and medium batches, for fused_lora_xw_sb / fused_multi_lora_xw_sb
// (lorafusion/ops/triton_ops/fused_lora_xw_sb.py:74-206, fused_multi_lora_xw_sb.py:66-218) and fused_lora_dyw_dsa /
// fused_multi_lora_dyw_dsa (fused_lora_dyw_dsa.py:69-181, fused_multi_lora_dyw_dsa.py:60-185).
//
// What bounds it: the path into a compute unit's LDS.  A unit takes in 100 - 130 GB/s of direct loads, whatever the number of stages in
// flight beyond two (four here; five and six measured level) -- a loads-only loop over the tiles of 300 x 4096 x 4096 takes 17 us, the
// kernel 19 on warm weights -- and the MFMAs of a 160x128 tile take about as long as its loads.  (Where a large weight comes from HBM, the reads from there:
// loads alone over the tiles of 333 x 14336 x 4096 take 45 us cold and 29 warm, the kernel 46 - 50.)  Hence:
//  * whole 128-byte lines per load (K steps of 64), one every few MFMAs over the whole step: gemm_lora.hip's four-wave tiles load
//    half lines in pairs, all of them in every second step of 32, more than the texture addresser takes there;
//  * the LoRA term behind the K loop: its rows of L and keep bits come into registers while the first tiles land, its skinny operand
//    into a dead LDS stage during the last three steps.  Seeding the accumulators with it cost 8 - 12 us of a 55 us launch
//    (1280 x 4096 x 4096, ranks to 64): routing table, operands and mask are three round trips in a row before the first step.
// Against the same tiles of gemm_lora.hip (cold weights, rank-16 term, keep bits in the NN product; us, NT / NN): 300 x 4096 x 4096 on 128x64
// 25.3 / 26.8 -> 22.7 / 21.1; 1280 x 4096 x 4096 on 160x128 50.2 / 50.2 (192x128) -> 43.7 / 41.4; 1024 x 4096 x 4096 on 128x128 39.5 / 42.2 -> 36.1 / 35.6;
// 333 x 14336 x 4096 on 192x128 55.0 / 54.3 -> 51.8 / 49.4 (the weight from HBM; 46 where the 256 MB cache holds it).
//
// One workgroup per tile of 32 TI x 32 TJ, four waves of 16 TI x 16 TJ (16x16x32 MFMA blocks, accumulators in the accumulation
// registers, the loop's memory instructions in assembly: see gemm_big.hip for the reasons).
//
// Tiles of up to 128x128 leave room in the register file for four waves more (LOADERS), which do nothing but load.  A wave that does both stops multiplying
// while the texture addresser, which four waves' loads keep 60 - 80 % busy, takes its next load; the loading waves stop in its place, and they order a
// stage's loads as soon as it is free.  Cold weights, rank-16 term, us, NT / NN: 300 x 4096 x 4096 on 128x64 22.1 / 22.9 -> 21.2 / 21.3; 1024 x 4096 x 4096
// on 128x128 34.9 / 38.1 -> 33.2 / 36.0; 600 x 4096 x 4096 28.8 / 30.8 -> 27.7 / 28.1.  (160x128 and 192x128 would spill at 256 registers a wave.  Measured
// level: fragments waited for by count and a barrier behind the first MFMAs of a half, other priorities; slower: the two halves of a step on
// two sets of four waves.)
// The 96x64 and 64x64 tiles move fewer operand bytes per compute unit where a few hundred rows do not fill a round with larger ones: 300 x 4096 x 4096
// on 96x64 (256 tiles) 19.7 / 19.6, 500 x 2048 x 4096 20.6 / 21.0 (128x64) -> 17.7 / 17.6.
#include "lf_common.h"
#include <type_traits>
#include <utility>

namespace {

constexpr int BK = 64;

template <typename T> struct MidOp;
template <> struct MidOp<__bf16> {
  // accumulators stay in the accumulation registers (see gemm_big.hip); hazards against compiler-generated code: mfma_fence()
  static __device__ __forceinline__ void mfma(lf_f32x4& c, lf_u32x4 a, lf_u32x4 b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  }
  static __device__ __forceinline__ void mfma_first(lf_f32x4& c, lf_u32x4 a, lf_u32x4 b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b));
  }
  // the term: d = a b and d += a b in ordinary vector registers
  static __device__ __forceinline__ void mfma_v0(lf_f32x4& d, lf_u32x4 a, lf_u32x4 b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "v"(b));
  }
  static __device__ __forceinline__ void mfma_v(lf_f32x4& d, lf_u32x4 a, lf_u32x4 b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "v"(b));
  }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    bf2 v = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(uint32_t, v);
  }
  static __device__ __forceinline__ float to_float(uint16_t bits) { return __builtin_bit_cast(float, (uint32_t)bits << 16); }
};
template <> struct MidOp<_Float16> {
  static __device__ __forceinline__ void mfma(lf_f32x4& c, lf_u32x4 a, lf_u32x4 b) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  }
  static __device__ __forceinline__ void mfma_first(lf_f32x4& c, lf_u32x4 a, lf_u32x4 b) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b));
  }
  // the term: d = a b and d += a b in ordinary vector registers
  static __device__ __forceinline__ void mfma_v0(lf_f32x4& d, lf_u32x4 a, lf_u32x4 b) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "v"(b));
  }
  static __device__ __forceinline__ void mfma_v(lf_f32x4& d, lf_u32x4 a, lf_u32x4 b) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "v"(b));
  }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    h2 v = {(_Float16)lo, (_Float16)hi};
    return __builtin_bit_cast(uint32_t, v);
  }
  static __device__ __forceinline__ float to_float(uint16_t bits) { return (float)__builtin_bit_cast(_Float16, bits); }
};

__device__ __forceinline__ void mfma_fence() { asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory"); }

template <int N, typename F>
__device__ __forceinline__ void sfor(F&& f) {
  [&]<int... I>(std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }(std::make_integer_sequence<int, N>{});
}

template <int TI, int TJ> struct MidLds {
  static constexpr int STAGE = (TI + TJ) * 4096;   // bytes: (32 TI + 32 TJ) rows of 128
  static constexpr int NST = 4;
  static constexpr int BYTES = NST * STAGE;
  static constexpr bool LOADERS = TI * TJ <= 16;   // four waves more, which only load
  static constexpr int THREADS = LOADERS ? 512 : 256;
  static_assert(BYTES <= 160 * 1024, "stages fit the LDS of a CU");
};

template <typename T, bool NN, int TI, int TJ>
__global__ void __launch_bounds__((MidLds<TI, TJ>::THREADS), 1)
gemm_mid_kernel(const LfGemmParams p, const LfSegTable seg) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass only needs the launch stub (buffer-resource types are device-only)
  using std::integral_constant;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  constexpr int BM = TI * 32, BN = TJ * 32, WROWS = TI * 16, WCOLS = TJ * 16;
  constexpr int STAGE = MidLds<TI, TJ>::STAGE, NST = MidLds<TI, TJ>::NST, STAGE_A = TI * 4096;
  constexpr bool LOADERS = MidLds<TI, TJ>::LOADERS;
  constexpr int NL = TI + TJ;          // tile loads per (loading) wave and step
  constexpr int NLH = (NL + 1) / 2;    // of which in the first sub-step
  constexpr int NM = TI * TJ;          // MFMAs per wave and sub-step
  constexpr int LDP = NM / NLH;        // a tile load every LDP MFMAs
  static_assert(LDP >= 2 && NL <= NM, "a sub-step has a gap for every fragment read and two for every tile load");
  const int tid = threadIdx.x & 255, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // (among those that multiply, or among those that load)
  const int wm = wave >> 1, wn = wave & 1;

  // ---- tile: XCD-aware order, grouped along M (a split contraction: slice by slice)
  const int total = p.grid_m * p.grid_n;
  int pid = lf_xcd_order((int)(blockIdx.y * gridDim.x + blockIdx.x), total * (int)gridDim.y);
  const int slice = p.ksplit > 1 ? pid / total : 0;
  pid -= slice * total;
  const int width = p.group_m * p.grid_n;
  const int group = pid / width;
  const int first_m = group * p.group_m;
  const int gsz = min(p.grid_m - first_m, p.group_m);
  const int pid_m = first_m + (pid % width) % gsz;
  const int pid_n = (pid % width) / gsz;
  const int m0 = pid_m * BM, n0 = pid_n * BN;
  // K steps of this workgroup: [kbeg, kbeg + nk); tile columns start their walk one step apart (memory channels)
  const int kbeg = slice * (p.ks_steps >> 1);
  const int nk = p.ksplit > 1 ? min(p.ks_steps >> 1, p.K / BK - kbeg) : p.K / BK;
  const int kstart = (pid_n & 15) % nk;

  // ---- tile loads: direct to LDS, 1024 bytes per wave instruction; load idx fills [idx * 4096 + wave * 1024, + 1024) of a
  // stage.  K-contiguous operands: 8 rows of 128 bytes, granule g of row r at slot g ^ ((r >> 1) & 7).  Rows beyond the
  // matrix are clamped to its last (their products are not stored).  NN operand B [K,N]: rows of BN elements; the k-rows
  // that 32 lanes of a transposing read touch together (r and r+8 for four consecutive r) lie in different wave
  // instructions and differ in the key that permutes a row's 32-byte units: they cover all 64 banks.
  uint32_t voff[NL];
  {
    const int lrow = tid >> 3, srcg = (tid & 7) ^ ((lrow >> 1) & 7);
#pragma unroll
    for (int i = 0; i < TI; i++) voff[i] = (uint32_t)((min(m0 + i * 32 + lrow, p.M - 1) - m0) * (int)p.lda * 2 + srcg * 16);
#pragma unroll
    for (int i = 0; i < TJ; i++) {
      if constexpr (!NN) {
        voff[TI + i] = (uint32_t)((i * 32 + lrow) * (int)p.ldb * 2 + srcg * 16);
      } else if constexpr (TJ == 4) {
        // row r = 32 ks + 16 b4 + 8 b3 + 4 hh + j4: instruction j4 + 4 b3 + 8 ks, row 2 b4 + hh of it, key j4 + 4 b3
        const int row = 32 * (i >> 1) + 16 * (lane >> 5) + 8 * (i & 1) + 4 * ((lane >> 4) & 1) + wave;
        voff[TI + i] = (uint32_t)(row * (int)p.ldb * 2 + ((lane & 15) ^ ((wave + 4 * (i & 1)) << 1)) * 16);
      } else {
        static_assert(TJ == 4 || TJ == 2, "tile columns");
        // instruction j4 + 4 ks, row b3 + 2 hh + 4 b4 of it, key j4
        const int idx = lane >> 3, row = 32 * i + 16 * (idx >> 2) + 8 * (idx & 1) + 4 * ((idx >> 1) & 1) + wave;
        voff[TI + i] = (uint32_t)(row * (int)p.ldb * 2 + ((lane & 7) ^ (wave << 1)) * 16);
      }
    }
  }
  lf_u32x4 ra, rb;
  {
    const char* a_base = (const char*)p.A + (int64_t)m0 * p.lda * 2;
    const char* b_base = NN ? (const char*)p.B + (int64_t)n0 * 2 : (const char*)p.B + (int64_t)n0 * p.ldb * 2;
    ra = lf_u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uintptr_t)a_base),
                  (uint32_t)__builtin_amdgcn_readfirstlane((int)((uintptr_t)a_base >> 32)) & 0xffffu, 0x7fffffffu, 0x00020000u};
    rb = lf_u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uintptr_t)b_base),
                  (uint32_t)__builtin_amdgcn_readfirstlane((int)((uintptr_t)b_base >> 32)) & 0xffffu, 0x7fffffffu, 0x00020000u};
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  const uint32_t m0w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds0 + wave * 1024));
  // scalars of the K loop through an empty asm: the compiler waits for the kernel arguments behind them here, not in the loop
  int nk_s = nk, kb_mul = NN ? BK * (int)p.ldb * 2 : BK * 2, kbeg_s = kbeg, kstart_s = kstart;
  asm volatile("" : "+s"(nk_s), "+s"(kb_mul), "+s"(kbeg_s), "+s"(kstart_s));
  auto kbase = [&](int k, int& ka, int& kb) __attribute__((always_inline)) {
    int kp = kstart_s + k;
    kp = kp >= nk_s ? kp - nk_s : kp;
    kp += kbeg_s;
    ka = kp * (BK * 2);
    kb = kp * kb_mul;
  };
  auto set_m0 = [&](uint32_t base, auto OFF) __attribute__((always_inline)) {
    asm volatile("s_add_u32 m0, %0, %1" ::"s"(base), "n"(OFF.value) : "memory", "scc", "m0");
  };
  auto issue_load = [&](lf_u32x4 rsrc, uint32_t vo, int so) __attribute__((always_inline)) {
    asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(vo), "s"(rsrc), "s"(so) : "memory");
  };
  auto load_stage = [&](int k, auto ST) __attribute__((always_inline)) {
    int ka, kb;
    kbase(k, ka, kb);
    sfor<NL>([&](auto I) {
      constexpr int idx = I.value;
      set_m0(m0w, integral_constant<int, ST.value * STAGE + idx * 4096>{});
      asm volatile("s_nop 0" ::: "memory");
      issue_load(idx < TI ? ra : rb, voff[idx], idx < TI ? ka : kb);
    });
  };
  auto lgkm0 = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
  auto barrier = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    lgkm0();
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // (nk >= NST: the launcher's condition)
  if constexpr (LOADERS) {
    if (__builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8) != 0) {
      // The loading waves keep NST - 1 steps on order.  Barrier of step s: step s+1 has landed and every multiplying wave has read all of
      // step s, whose stage takes step s+NST.  They end behind the last step's barrier with nothing in flight; later barriers are the other waves' own.
      sfor<NST>([&](auto I) { load_stage(I.value, I); });
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 1) * NL) : "memory");
      barrier();
      uint32_t st = 0;
      for (int s = 0; s + NST < nk; s++) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 2) * NL) : "memory");
        barrier();
        int ka, kb;
        kbase(s + NST, ka, kb);
        const uint32_t mb = m0w + st;
        sfor<NL>([&](auto I) {
          set_m0(mb, integral_constant<int, I.value * 4096>{});
          asm volatile("s_nop 0" ::: "memory");
          issue_load(I.value < TI ? ra : rb, voff[I.value], I.value < TI ? ka : kb);
        });
        st = st + STAGE == NST * STAGE ? 0 : st + STAGE;
      }
      sfor<NST - 1>([&](auto I) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 2 - I.value) * NL) : "memory");
        barrier();
      });
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      barrier();
      return;
    }
  } else {
    sfor<NST - 1>([&](auto I) { load_stage(I.value, I); });
  }
  __builtin_amdgcn_sched_barrier(0);

  // ---- LoRA term: adapters of the wave's rows.  A wave's rows meet at most two routing blocks (their size is a multiple
  // of 128, a wave has at most 96 rows): block rows from `isplit` on belong to the second, which is multiplied on its own.  The
  // products of an adapter are not formed for the other's rows at all: a zero operand would still carry its infinities
  // and NaNs over.
  const int wrow0 = m0 + wm * WROWS, wcol0 = n0 + wn * WCOLS;
  const int l16 = lane & 15, kg = lane >> 4;
  struct Term { const T* rp; int rank; float mult; bool mask; };
  const bool term = p.L != nullptr && kbeg == 0 && wrow0 < p.M;   // (split contraction: the first slice carries the term)
  Term t0{}, t1{};
  int isplit = TI, nterm = term ? 1 : 0;
  const T* __restrict__ L = (const T*)p.L;
  const int nch = (p.R + 31) >> 5;   // chunks of 32 rank columns
  lf_u32x4 lf0[TI], lf1[TI];         // chunks 0 and 1 of L, fetched now
  uint32_t mw[TI][TJ / 2];           // the lane's keep bits: block (i, j): bits (j & 1) * 16 + kg * 4 .. + 3 of mw[i][j >> 1]
  auto load_l = [&](int t, lf_u32x4 (&lf)[TI]) __attribute__((always_inline)) {
    const int r0 = min(t * 32 + kg * 8, p.R - 8);
#pragma unroll
    for (int i = 0; i < TI; i++) lf[i] = *(const lf_u32x4*)(L + (int64_t)min(wrow0 + i * 16 + l16, p.M - 1) * p.R + r0);
  };
  bool use_mask = false;
  if (term) {
    // (constant address space: scalar loads.  Vector loads would wait for all the tile loads in flight, table and scale one after
    // the other.)
    typedef const __attribute__((address_space(4))) int32_t* tab_t;
    typedef const __attribute__((address_space(4))) float* val_t;
    auto term_of_block = [&](int blk) __attribute__((always_inline)) {
      const tab_t tab = (tab_t)(uintptr_t)seg.table;
      const val_t val = (val_t)(uintptr_t)(p.mult_mode == 0 ? seg.block_scale : seg.block_p);
      const int rank = tab[3 * blk], fb = tab[3 * blk + 2];
      const float v = val[blk];
      int s = 0;
      for (int i = 1; i < seg.n_seg; i++) s = (seg.first_block[i] == fb) ? i : s;
      Term t{(const T*)seg.ptr[s], rank, v, false};
      if (p.mult_mode == 1) {
        t.mask = p.mask != nullptr && v > 0.f;
        t.mult = t.mask ? 1.f / (1.f - v) : 1.f;
      }
      return t;
    };
    // mult_mode 1 without a keep-mask means no dropout, whatever p says: the term is not rescaled
    const bool drop = p.mask != nullptr && p.mult_mode == 1 && seg.p > 0.f;
    t0 = Term{(const T*)seg.ptr[0], seg.rank[0], p.mult_mode == 0 ? seg.scale : (drop ? 1.f / (1.f - seg.p) : 1.f), drop};
    load_l(0, lf0);
    if (nch > 1) load_l(1, lf1);
    if (seg.table != nullptr) {
      const int row = p.row0 + wrow0, blk = min(row / seg.block_size_m, seg.n_blocks - 1);
      t0 = term_of_block(blk);
      const int left = (blk + 1) * seg.block_size_m - row;
      if (left < WROWS && blk + 1 < seg.n_blocks) {
        t1 = term_of_block(blk + 1);
        if (t1.rp != t0.rp || t1.rank != t0.rank || t1.mult != t0.mult || t1.mask != t0.mask) isplit = left / 16, nterm = 2;   // (else two blocks of one adapter)
      }
    }
    use_mask = t0.mask || (nterm == 2 && t1.mask);
    if (use_mask) {
#pragma unroll
      for (int i = 0; i < TI; i++)
#pragma unroll
        for (int d = 0; d < TJ / 2; d++)
          mw[i][d] = *(const uint32_t*)(p.mask + (int64_t)min(wrow0 + i * 16 + l16, p.M - 1) * p.ldmask + (wcol0 >> 3) + d * 4);
    }
  }
  // The skinny operand (B_i rows of the wave's columns, A_i columns) goes to the wave's own part of a dead stage as direct
  // loads, 32 rank columns (one MFMA step) at a time; rank columns beyond the adapter's rank lie beyond the buffer's
  // end and read as zeros.  Slot c of a wave: chunk c & 3 of part c >> 2.
  constexpr int CH = TJ * 1024;        // bytes of a chunk
  uint32_t dead = 0;                   // the stage of step nk - NST: read by nobody in the last NST - 1 steps
  auto area_of = [&](int c) {
    const uint32_t st = dead + (uint32_t)(c >> 1) * STAGE;
    return (st >= NST * STAGE ? st - NST * STAGE : st) + (uint32_t)(wave * 2 + (c & 1)) * CH;
  };
  static_assert(8 * CH <= STAGE, "two chunks per wave and stage");
  auto load_rop = [&](const Term& t, int ch, int c) __attribute__((always_inline)) {
    typedef __attribute__((address_space(3))) void* lds_ptr_t;
    char* dst = smem + area_of(c);
    const int elems = NN ? t.rank * p.N : p.N * t.rank;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)t.rp, 0, elems * 2, 0x00020000);
#pragma unroll
    for (int q = 0; q < TJ; q++) {
      uint32_t vo;
      if constexpr (!NN) {
        // 16 rows of 64 bytes; granule g of row r at slot g ^ ((r >> 1) & 3)
        const int r = q * 16 + (lane >> 2), g = (lane & 3) ^ ((r >> 1) & 3), col = ch * 32 + g * 8;
        vo = col < t.rank ? (uint32_t)(((wcol0 + r) * t.rank + col) * 2) : 0x7fffffffu;
      } else if constexpr (TJ == 4) {
        // 8 rank rows of 128 bytes, their 32-byte units permuted (rows read together: r, r+8 for four r)
        const int r = q * 8 + (lane >> 3), key = ((r >> 1) & 1) | (((r >> 3) & 1) << 1);
        vo = ch * 32 + r < t.rank ? (uint32_t)(((ch * 32 + r) * p.N + wcol0 + ((lane & 7) ^ (key << 1)) * 8) * 2) : 0x7fffffffu;
      } else {
        const int r = q * 16 + (lane >> 2);   // 16 rank rows of 64 bytes
        vo = ch * 32 + r < t.rank ? (uint32_t)(((ch * 32 + r) * p.N + wcol0 + (lane & 3) * 8) * 2) : 0x7fffffffu;
      }
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(dst + q * 1024), 16, vo, 0, 0, 0);
    }
  };

  // ---- fragments: two register sets, one per half of a step
  lf_u32x4 fa[2][TI], fb[2][TJ];
  lf_f32x4 acc[TI][TJ];
  uint32_t fa_off[2], fb_off[NN ? TJ : 2];
  {
    const int key = (l16 >> 1) & 7;
#pragma unroll
    for (int ks = 0; ks < 2; ks++) fa_off[ks] = lds0 + (wm * WROWS + l16) * 128 + (((ks * 4 + kg) ^ key) << 4);
    if constexpr (!NN) {
#pragma unroll
      for (int ks = 0; ks < 2; ks++) fb_off[ks] = lds0 + STAGE_A + (wn * WCOLS + l16) * 128 + (((ks * 4 + kg) ^ key) << 4);
    } else {
      // ds_read_b64_tr_b16: within a 16-lane group, lane 4j+c addresses row j, columns 4c..4c+3 and receives column
      // (lane & 15), rows 0..3.  Group kg takes k-rows kg * 8 + j4 (and + 4: 256 bytes on)
      const int j4 = l16 >> 2, c = l16 & 3, b3 = kg & 1, b4 = kg >> 1;
#pragma unroll
      for (int j = 0; j < TJ; j++) {
        if constexpr (TJ == 4)
          fb_off[j] = lds0 + STAGE_A + (j4 + 4 * b3) * 1024 + b4 * 512 + (((wn * 4 + j) ^ (j4 + 4 * b3)) << 5) + c * 8;
        else
          fb_off[j] = lds0 + STAGE_A + j4 * 1024 + b3 * 128 + b4 * 512 + (((wn * 2 + j) ^ j4) << 5) + c * 8;
      }
    }
  }
  // the ORD-th fragment read of half KS of the stage at LDS byte offset st: B 0, A 0, the other B, the other A
  auto read_one = [&](auto SET, auto KS, uint32_t st, auto ORD) __attribute__((always_inline)) {
    constexpr int set = SET.value, ks = KS.value, ord = ORD.value;
    constexpr bool isa = ord == 1 || ord > TJ;
    constexpr int o = isa ? (ord == 1 ? 0 : ord - TJ) : (ord == 0 ? 0 : ord - 1);
    if constexpr (isa) {
      const uint32_t ad = fa_off[ks] + st;
      lf_u32x4 tmp;
      asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(tmp) : "v"(ad), "n"(o * 2048) : "memory");
      fa[set][o] = tmp;
    } else if constexpr (!NN) {
      const uint32_t ad = fb_off[ks] + st;
      lf_u32x4 tmp;
      asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(tmp) : "v"(ad), "n"(o * 2048) : "memory");
      fb[set][o] = tmp;
    } else {
      const uint32_t ad = fb_off[o] + st;
      lf_u32x2 lo, hi;
      asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(lo) : "v"(ad), "n"(ks * TJ * 2048) : "memory");
      asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(hi) : "v"(ad), "n"(ks * TJ * 2048 + 256) : "memory");
      fb[set][o] = lf_u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
  };
  auto mfma_one = [&](int set, int m, auto FIRST) __attribute__((always_inline)) {
    const int i = m / TJ, j = m % TJ;
    if constexpr (FIRST.value) MidOp<T>::mfma_first(acc[i][j], fb[set][j], fa[set][i]);
    else MidOp<T>::mfma(acc[i][j], fb[set][j], fa[set][i]);
  };
  using S0 = integral_constant<int, 0>;
  using S1 = integral_constant<int, 1>;
  using F_ = std::false_type;
  using T_ = std::true_type;
  // ---- K loop.  Step s lives in stage s % NST.  Its two halves (k 0-31, k 32-63) run on fragment set 0 and 1; while one
  // half's MFMAs run, the other set is read, one fragment per MFMA.  Between the halves: wait until this wave's loads of step s+1
  // have landed (those of steps s+2 .. s+NST-2 and half of step s+NST-1's may be outstanding) and its fragment reads are
  // complete, then the barrier: it publishes step s+1 and ends all reads of step s.  The loads of step s+NST-1 go into the stage of
  // step s-1, spread over both halves.
  uint32_t cst = 0;
  auto k_step = [&](int s, auto FIRST, auto LOAD, auto NEXT, auto WAIT) __attribute__((always_inline)) {
    const uint32_t cur = cst, nxt = cur + STAGE >= NST * STAGE ? 0 : cur + STAGE, prv = cur >= STAGE ? cur - STAGE : (NST - 1) * STAGE;
    int ka = 0, kb = 0;
    if constexpr (LOAD.value) kbase(s + NST - 1, ka, kb);
    const uint32_t mb = m0w + prv;
    auto half = [&](auto SET, auto READ, uint32_t rst, auto BASE, auto COUNT, auto ZERO) __attribute__((always_inline)) {
      constexpr int set = SET.value;
      sfor<NM>([&](auto MM) {
        constexpr int m = MM.value;
        if constexpr (READ.value && m < NL) read_one(integral_constant<int, 1 - set>{}, integral_constant<int, 1 - set>{}, rst, MM);
        if constexpr (!LOADERS && LOAD.value && m / LDP < COUNT.value) {
          constexpr int idx = BASE.value + m / LDP;
          if constexpr (m % LDP == 0) set_m0(mb, integral_constant<int, idx * 4096>{});
          if constexpr (m % LDP == 1) issue_load(idx < TI ? ra : rb, voff[idx], idx < TI ? ka : kb);
        }
        mfma_one(set, m, ZERO);
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    half(S0{}, T_{}, cur, integral_constant<int, 0>{}, integral_constant<int, NLH>{}, FIRST);
    if constexpr (!LOADERS && WAIT.value >= 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(WAIT.value) : "memory");
    barrier();
    half(S1{}, NEXT, nxt, integral_constant<int, NLH>{}, integral_constant<int, NL - NLH>{}, F_{});
    __builtin_amdgcn_sched_barrier(0);
    lgkm0();
    __builtin_amdgcn_sched_barrier(0);
    cst = nxt;
  };
  constexpr int INFLIGHT = (NST - 3) * NL + NLH;
  static_assert(NST >= 4 && (NST - 2) * NL + 2 * TJ < 64, "vmcnt is a 6-bit counter");
  if constexpr (!LOADERS) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 2) * NL) : "memory");
  barrier();
  sfor<NL>([&](auto I) { read_one(S0{}, S0{}, 0u, I); });
  lgkm0();
  k_step(0, T_{}, T_{}, T_{}, integral_constant<int, INFLIGHT>{});
  int s = 1;
  for (; s + NST - 1 < nk; s++) k_step(s, F_{}, T_{}, T_{}, integral_constant<int, INFLIGHT>{});
  __builtin_amdgcn_sched_barrier(0);
  // the term's skinny operand (no term: an empty buffer, zeros)
  dead = cst >= STAGE ? cst - STAGE : (NST - 1) * STAGE;
  load_rop(t0, 0, 0);
  load_rop(t0, 1, 1);
  __builtin_amdgcn_sched_barrier(0);
  sfor<NST - 1>([&](auto I) {
    constexpr int left = NST - 3 - I.value;   // whole steps of loads that may be outstanding
    k_step(s + I.value, F_{}, F_{}, std::bool_constant<(I.value < NST - 2)>{}, integral_constant<int, left >= 0 ? left * NL + 2 * TJ : -1>{});
  });
  mfma_fence();
  // The term's operand has landed, in waves without a term too: an empty buffer still writes its zeros to LDS, and the stages take
  // other waves' results from here on (a split contraction's later slices end here: nothing may land behind the workgroup's end).
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  barrier();   // every wave is done with the stages

  // ---- results into ordinary vector registers: acc + mult * (masked) term
  lf_f32x4 P[TI][TJ];
  // chunk c of part `part` (its slot in LDS: 4 part + c); FIRST: the part's first, which writes P
  auto chunk = [&](int part, int c, lf_u32x4 (&lf)[TI], auto FIRST) __attribute__((always_inline)) {
    const int rank = part ? t1.rank : t0.rank;
    lf_u32x4 rf[TJ], lz[TI];
    const bool in_r = c * 32 + kg * 8 < rank;   // lanes beyond the rank feed zeros
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
      for (int d = 0; d < 4; d++) lz[i][d] = in_r ? lf[i][d] : 0u;
    const uint32_t ar = lds0 + area_of(part * 4 + c);
    if constexpr (!NN) {
      const uint32_t ad = ar + l16 * 64 + ((kg ^ ((l16 >> 1) & 3)) << 4);
      sfor<TJ>([&](auto J) {
        lf_u32x4 t;
        const uint32_t ad_ = ad;
        asm volatile("ds_read_b128 %0, %1 offset:%2\n\ts_waitcnt lgkmcnt(0)" : "=v"(t) : "v"(ad_), "n"(J.value * 1024) : "memory");
        rf[J.value] = t;
      });
    } else {
      const int j4 = l16 >> 2, cc = l16 & 3, row = kg * 8 + j4;
      sfor<TJ>([&](auto J) {
        constexpr int pitch = TJ * 32;
        const int key = TJ == 4 ? (((row >> 1) & 1) | (((row >> 3) & 1) << 1)) : 0;
        const uint32_t ad = ar + row * pitch + ((J.value ^ key) << 5) + cc * 8;
        lf_u32x2 lo, hi;
        asm volatile("ds_read_b64_tr_b16 %0, %2\n\tds_read_b64_tr_b16 %1, %2 offset:%3\n\ts_waitcnt lgkmcnt(0)"
                     : "=&v"(lo), "=&v"(hi) : "v"(ad), "n"(4 * pitch) : "memory");
        rf[J.value] = lf_u32x4{lo[0], lo[1], hi[0], hi[1]};
      });
    }
    // the MFMAs are inline assembly, which the compiler's hazard recogniser does not see: wait states between the vector
    // instructions that made their operands and the first of them
#pragma unroll
    for (int i = 0; i < TI; i++) asm volatile("s_nop 1" : "+v"(lz[i]));
#pragma unroll
    for (int j = 0; j < TJ; j++) asm volatile("s_nop 1" : "+v"(rf[j]));
#pragma unroll
    for (int i = 0; i < TI; i++) {
      if (nterm == 2 && (i >= isplit) != (part == 1)) continue;
#pragma unroll
      for (int j = 0; j < TJ; j++) {
        if constexpr (FIRST.value) MidOp<T>::mfma_v0(P[i][j], rf[j], lz[i]);
        else MidOp<T>::mfma_v(P[i][j], rf[j], lz[i]);
      }
    }
  };
  if (nterm > 0) {
    for (int c = 2; c < nch; c++) load_rop(t0, c, c);
    if (nterm == 2)
      for (int c = 0; c < nch; c++) load_rop(t1, c, 4 + c);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    for (int part = 0; part < nterm; part++) {
      chunk(part, 0, lf0, T_{});
      if (nch > 1) chunk(part, 1, lf1, F_{});
      for (int c = 2; c < nch; c++) {
        lf_u32x4 lf[TI];
        load_l(c, lf);
        chunk(part, c, lf, F_{});
      }
    }
    mfma_fence();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < TI; i++) {
      const float mult = i >= isplit ? t1.mult : t0.mult;
      const bool masked = i >= isplit ? t1.mask : t0.mask;
#pragma unroll
      for (int j = 0; j < TJ; j++) {
        asm volatile("" : "+v"(P[i][j]));   // (reads of the products stay behind the fence)
        const int bits = masked ? (int)(mw[i][j >> 1] >> ((j & 1) * 16 + kg * 4)) : 0xf;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float pe = P[i][j][e];
          const uint32_t keep = (uint32_t)__builtin_amdgcn_sbfe(bits, e, 1);   // 0 or all ones
          const float pm = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, pe) & keep);
          P[i][j][e] = __builtin_fmaf(pm, mult, acc[i][j][e]);
        }
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
      for (int j = 0; j < TJ; j++) P[i][j] = acc[i][j];
  }
  if (p.ksplit > 1) {
    // split contraction: the fp32 sums of this slice, 16 bytes per lane (row l16 of a block, columns kg*4 .. +3)
    float* __restrict__ part = p.ks_ws + (int64_t)slice * p.M * p.N;
#pragma unroll
    for (int i = 0; i < TI; i++) {
      const int gm = wrow0 + i * 16 + l16;
#pragma unroll
      for (int j = 0; j < TJ; j++) {
        if (gm < p.M) *(lf_f32x4*)(part + (int64_t)gm * p.N + wcol0 + j * 16 + kg * 4) = P[i][j];
      }
    }
    return;
  }

  // ---- epilogue: bias, convert, through the wave's own LDS so that stores are 16 bytes per lane and cover whole rows of
  // the wave's tile.  Granule g (16 bytes) of row r at slot g ^ ((r / RPB) & KEY): RPB rows span the 64 banks once.
  T* __restrict__ C = (T*)p.C;
  const uint16_t* bias16 = (const uint16_t*)p.bias;
  constexpr int PITCH = WCOLS * 2, LPR = PITCH / 16, RPI = 64 / LPR, RPB = 256 / PITCH, KEY = LPR - 1;
  barrier();   // every wave has read its skinny operands
  char* ep = smem + wave * (WROWS * PITCH);
#pragma unroll
  for (int j = 0; j < TJ; j++) {
    lf_u32x2 bv = {0u, 0u};
    if (bias16 != nullptr) bv = *(const lf_u32x2*)(bias16 + wcol0 + j * 16 + kg * 4);
    const float b0 = MidOp<T>::to_float((uint16_t)(bv[0] & 0xffffu)), b1 = MidOp<T>::to_float((uint16_t)(bv[0] >> 16));
    const float b2 = MidOp<T>::to_float((uint16_t)(bv[1] & 0xffffu)), b3 = MidOp<T>::to_float((uint16_t)(bv[1] >> 16));
#pragma unroll
    for (int i = 0; i < TI; i++) {
      const lf_f32x4 a = P[i][j];
      const lf_u32x2 o = {MidOp<T>::pack2(a[0] + b0, a[1] + b1), MidOp<T>::pack2(a[2] + b2, a[3] + b3)};
      const int r = i * 16 + l16, g = j * 2 + (kg >> 1);
      *(lf_u32x2*)(ep + r * PITCH + ((g ^ ((r / RPB) & KEY)) << 4) + (kg & 1) * 8) = o;
    }
  }
#pragma unroll
  for (int q = 0; q < WROWS / RPI; q++) {
    const int r = q * RPI + lane / LPR, g = lane % LPR;
    const lf_u32x4 v = *(const lf_u32x4*)(ep + r * PITCH + ((g ^ ((r / RPB) & KEY)) << 4));
    if (wrow0 + r < p.M) __builtin_nontemporal_store(v, (lf_u32x4*)(C + (int64_t)(wrow0 + r) * p.ldc + wcol0 + g * 8));
  }
#endif
}

template <typename T, bool NN, int TI, int TJ>
int launch_mid(LfGemmParams p, const LfSegTable& seg, hipStream_t st) {
  p.grid_m = (p.M + TI * 32 - 1) / (TI * 32);
  p.grid_n = p.N / (TJ * 32);
  p.group_m = 8;
  auto kern = gemm_mid_kernel<T, NN, TI, TJ>;
  static LfLdsFlags lds_ok;
  if (!lf_allow_lds(kern, MidLds<TI, TJ>::BYTES, lds_ok)) return LF_ELAUNCH;
  return lf_launch(kern, dim3(p.grid_m * p.grid_n, p.ksplit > 1 ? p.ksplit : 1), dim3(MidLds<TI, TJ>::THREADS), MidLds<TI, TJ>::BYTES, st, p, seg);
}

template <int TI, int TJ>
int launch_mid_any(const LfGemmParams& p, const LfSegTable& seg, bool nn, int dtype, hipStream_t st) {
  if (dtype == LF_BF16) return nn ? launch_mid<__bf16, true, TI, TJ>(p, seg, st) : launch_mid<__bf16, false, TI, TJ>(p, seg, st);
  if (dtype == LF_F16) return nn ? launch_mid<_Float16, true, TI, TJ>(p, seg, st) : launch_mid<_Float16, false, TI, TJ>(p, seg, st);
  return LF_EINVAL;
}

}  // namespace

int lf_launch_gemm_mid(const LfGemmParams& p, const LfSegTable& seg, bool nn, int dtype, int cfg, hipStream_t st) {
  // whole tiles along N; at least as many K steps as stages, in the last slice of a split contraction too
  if (p.K % BK != 0 || p.M < 1 || p.N % (cfg == 12 || cfg >= 14 ? 64 : 128) != 0 || p.R > LF_MAX_RANK) return LF_ESHAPE;
  if (p.ksplit > 1 && p.ks_steps % 2 != 0) return LF_ESHAPE;
  if ((p.ksplit > 1 ? p.K / BK - (p.ksplit - 1) * (p.ks_steps / 2) : p.K / BK) < 4) return LF_ESHAPE;
  if (seg.table != nullptr && seg.block_size_m % 128 != 0) return LF_ESHAPE;
  if (p.mask != nullptr && (!p.mask_bits || p.N % 32 != 0 || p.ldmask % 4 != 0)) return LF_ESHAPE;
  switch (cfg) {
    case 13: return launch_mid_any<6, 4>(p, seg, nn, dtype, st);
    case 10: return launch_mid_any<5, 4>(p, seg, nn, dtype, st);
    case 11: return launch_mid_any<4, 4>(p, seg, nn, dtype, st);
    case 12: return launch_mid_any<4, 2>(p, seg, nn, dtype, st);
    case 14: return launch_mid_any<3, 2>(p, seg, nn, dtype, st);
    case 15: return launch_mid_any<2, 2>(p, seg, nn, dtype, st);
    default: return LF_EINVAL;
  }
}
