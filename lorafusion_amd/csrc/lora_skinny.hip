// Rank-r ("skinny") products of the LoRA branch for gfx950.  All are HBM-bandwidth bound:
// each streams one [M, K] or [M, N] operand once and does a few MFMA 16x16x32 per 16 rows.
//
//   xa      : S  = drop(X) A^T                       (replaces seeded_dropout + cuBLAS X~ A^T,
//             lorafusion/ops/lora_v1.py:111-119, and fused_dropout_matmul.py:152-277)
//   dys_dyb : dS = scale dY B ; dB = scale dY^T S    (fused_lora_dys_dyb.py:71-179,
//             fused_multi_lora_dys_dyb.py:61-185; fp32 atomics there, two-stage sums here)
//   da      : dA = dS^T X~                           (the cuBLAS call at lora_v1.py:153,
//             multi_lora.py:576-581; X~ is rebuilt from X and the keep-mask, never stored)
//
// Every kernel works on 128-row token blocks (= the routing block of the multi-LoRA batch
// info) and writes fp32 partial sums; the small reduce kernels add the partials in a fixed
// order, apply scale / 1/(1-p), zero padded rows and rank columns, and cast.  Results are
// therefore run-to-run deterministic.
//
// Streaming: the big operand moves as 128-row x 64-column tiles.  Global loads are coalesced
// (8 consecutive lanes read one 128-byte row segment) and the tile sits in LDS with the same XOR
// swizzle as the GEMM (granule g of row r at slot g ^ ((r>>1)&7)), from where both MFMA access
// patterns are bank-conflict free: row fragments (ds_read_b128) and transposed fragments
// (ds_read_b64_tr_b16).  Loading MFMA fragments straight from global memory would put every
// lane on a different row (one cache line per lane) and runs at a quarter of the coalesced rate.
// Two transports: through registers (xa: load, keep-mask applied on the way, LDS store), or as buffer
// loads that write LDS themselves, several tiles ahead through a ring of stages (dys_dyb / da; rank_ring.h).
//
// MFMA 16x16x32 operand layout (64 lanes): lane l holds row/col (l & 15) and the 8
// contraction elements of chunk (l >> 4).  Where the contraction index is the slow memory
// dimension, tiles are staged in LDS and read with ds_read_b64_tr_b16 (16 lanes read a
// 4-row x 16-column patch; lane 4j+c addresses row j, columns 4c..4c+3; each lane receives
// its column's 4 rows).
#include "lf_common.h"
#include "act_math.h"
#include "rank_ring.h"
#include <algorithm>
#include <cmath>
#include <numeric>
#include <type_traits>

namespace {

// ------------------------------------------------------------------------------------ xa
// Ranks to 64, where the sliced pass of lora_stream.hip is not the faster one or has no memory for its sums (lf_xa_takes_stream), and without a mask
// its ring kernel is not (lf_xa_rings).
// One workgroup of 8 waves per 16 rows (64 at ranks 48-64); no partial sums leave the workgroup.  The K range is dealt
// to the waves in 64-column steps (step s goes to wave s % 8), each wave streams its steps of the
// 16 rows with coalesced 16-byte loads (8 lanes cover one 128-byte line), the next step's loads in flight while one is used
// (ranks to 32), applies the keep-mask in registers and turns the row-major
// granules into MFMA row fragments through a 2 KB LDS patch of its own (same-wave LDS traffic is
// ordered: no barrier).  The adapter matrix A (L2 resident) takes the same route: fragment-shaped
// loads would put the four lanes of every quad on four different rows, a quarter of the
// coalesced rate in the texture addresser.  The eight partial [16, R] accumulators are added in a fixed order through LDS,
// scaled by 1/(1-p), zeroed in padded rows and beyond the adapter's rank, and stored as S.
// Rows per workgroup: every workgroup reads the whole adapter matrix (from L2), which at rank 64 is four times the
// bytes of 16 rows of X: ranks 48-64 take 64 rows (four row blocks share one set of A fragments; with the activation prologue the
// up-half registers of four do not fit next to the rest: two).  At rank 16 two row blocks per
// workgroup measured slower (0.27 -> 0.34 ms at the 8B layer: the registers of the second block cost loads in flight).
constexpr int XA_WAVES = 8;
constexpr int xa_nb(int rt, bool act) { return rt == 4 ? (act ? 2 : 4) : 1; }
constexpr int xa_rows(int rt, bool act) { return 16 * xa_nb(rt, act); }

// GEN: the keep-mask is not read but drawn here (Philox, the definition of the standalone mask
// kernel) from (seed, element index) and written to `mask_out` for the backward pass: the integer
// work hides behind the X stream, and one launch and one 1-byte-per-element read disappear.
// ACT: the rows of X do not exist yet: X = round16(round16(silu(G)) * U) is computed here from the gate and up halves of a
// SwiGLU MLP (`X` = G, `U`, rows `ldx` elements apart: the two halves of one merged projection output, or two
// tensors), written once to `act_out` [rows, K] (every element of X is loaded by exactly one lane of the grid) for the
// base GEMM and the backward, and fed to the rank-r product from registers: the activation pass and this pass's own
// read of X disappear.
template <typename T, int RT, bool GEN, bool ACT>
__global__ void __launch_bounds__(XA_WAVES * 64)
lora_xa_kernel(const T* __restrict__ X, const T* __restrict__ U, int64_t ldx, T* __restrict__ act_out,
               const uint8_t* __restrict__ mask, uint8_t* __restrict__ mask_out, int mask_bits,
               uint32_t seed_lo, uint32_t seed_hi, T* __restrict__ S, int M, int K, int R, const LfSegTable seg) {
  constexpr int NB = xa_nb(RT, ACT), XA_ROWS = xa_rows(RT, ACT);
  // the partial accumulators of the final sum reuse the patches (a barrier separates the two uses): at
  // rank 64 the separate 16 KB pushed the workgroup over 40 KB, and a CU then holds two workgroups, not four
  constexpr int PATCH_BYTES = XA_WAVES * 2048 * (NB + RT), RED_BYTES = XA_WAVES * XA_ROWS * RT * 16 * 4;
  __shared__ __attribute__((aligned(16))) char patch_all[PATCH_BYTES > RED_BYTES ? PATCH_BYTES : RED_BYTES];
  float (*red)[XA_ROWS][RT * 16] = (float (*)[XA_ROWS][RT * 16])patch_all;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, qq = lane >> 4;
  const int row0 = blockIdx.x * XA_ROWS;
  const int blk = row0 / ROWS;
  const BlockInfo bi = block_info(seg, blk, M);
  const T* __restrict__ A = (const T*)seg.ptr[bi.seg];
  const bool use_mask = GEN ? true : (mask != nullptr && bi.p > 0.f);
  const uint32_t thr = lf_keep_threshold(bi.p);
  const int Mrows = seg.table ? seg.n_blocks * ROWS : M;
  const int nsteps = K / 64;
  char* patch = patch_all + wave * 2048 * (NB + RT);  // one X patch per 16-row block, then one patch per 16 rank rows of A

  // loader mapping: lane -> (row lane>>3 (+8), granule lane&7); fragment mapping: (row li, granule 4h+qq)
  const int lrow = lane >> 3, lg = lane & 7;
  const T* xrow[2 * NB];
  const uint8_t* mrow[2 * NB];
  int64_t erow[2 * NB];    // GEN, ACT: element index of this lane's first column in each of its rows (two per 16-row block)
  bool row_real[2 * NB];   // GEN, ACT: the row exists (is not a clamped duplicate): its mask bytes / activations are written
#pragma unroll
  for (int i = 0; i < 2 * NB; i++) {
    const int r = min(row0 + i * 8 + lrow, Mrows - 1);
    xrow[i] = X + (int64_t)r * ldx + lg * 8;
    mrow[i] = mask_bits ? mask + (((int64_t)r * K + lg * 8) >> 3) : mask + (int64_t)r * K + lg * 8;
    erow[i] = (int64_t)r * K + lg * 8;
    row_real[i] = row0 + i * 8 + lrow < Mrows;
  }
  // ACT: the up half lies at one distance from the gate half for every row (a scalar, not a second set of row pointers)
  const int64_t u_off = ACT ? (int64_t)((uintptr_t)U - (uintptr_t)X) : 0;
  const int wr_off[2] = {lrow * 128 + ((lg ^ ((lrow >> 1) & 7)) << 4), (8 + lrow) * 128 + ((lg ^ (((8 + lrow) >> 1) & 7)) << 4)};
  const int rd_row = li * 128, rd_key = (li >> 1) & 7;

  lf_f32x4 acc[NB][RT];
#pragma unroll
  for (int nb = 0; nb < NB; nb++)
#pragma unroll
    for (int c = 0; c < RT; c++) acc[nb][c] = lf_f32x4{0.f, 0.f, 0.f, 0.f};

  // Two register sets of one step each at ranks up to 32, one set above: the loads of one set are requested before
  // the other set is used, so a wave's memory time and its integer / LDS / MFMA time overlap.  All waves of a launch
  // start together and would otherwise sit in the same phase -- everyone waiting for memory, then everyone
  // computing.  Measured at 16512 x 4096, rank 16, mask drawn in the kernel: one set of four steps 44.5 us, two sets
  // of two steps 45.4 (126 registers: half the waves per SIMD), two sets of one step 42.2.
  constexpr int NSET = RT <= 2 ? 2 : 1, UB = 1;
  lf_u32x4 xv[NSET][UB][2 * NB], av[NSET][UB][RT][2];
  lf_u32x4 uv[NSET][UB][ACT ? 2 * NB : 1];
  lf_u32x2 mv[NSET][UB][2 * NB];
  auto load_batch = [&](auto B, int s0) {
    constexpr int b = B.value;
#pragma unroll
    for (int u = 0; u < UB; u++) {
      const int s = s0 + u * XA_WAVES;
      if (s < nsteps) {
#pragma unroll
        for (int i = 0; i < 2 * NB; i++) {
          if constexpr (ACT) {
            // gate and up are read once, here: loads that do not allocate in the caches
            xv[b][u][i] = __builtin_nontemporal_load((const lf_u32x4*)(xrow[i] + s * 64));
            uv[b][u][i] = __builtin_nontemporal_load((const lf_u32x4*)((const char*)(xrow[i] + s * 64) + u_off));
          } else {
            xv[b][u][i] = *((const lf_u32x4*)(xrow[i] + s * 64));
          }
          if constexpr (!GEN) {
            // (bit format: the byte is only requested here and spread into eight bytes where it is used, so that no
            // wait for it separates the loads of a batch)
            if (use_mask) {
              if (mask_bits) mv[b][u][i][0] = mrow[i][s * 8];
              else mv[b][u][i] = *((const lf_u32x2*)(mrow[i] + s * 64));
            }
          }
        }
#pragma unroll
        for (int i = 0; i < 2; i++) {
#pragma unroll
          for (int c = 0; c < RT; c++) {
            const int ar = c * 16 + i * 8 + lrow;
            av[b][u][c][i] = lf_u32x4{0, 0, 0, 0};
            if (ar < bi.rank) av[b][u][c][i] = *(const lf_u32x4*)(A + (int64_t)ar * K + s * 64 + lg * 8);
          }
        }
      }
    }
  };
  auto use_batch = [&](auto B, int s0) {
    constexpr int b = B.value;
#pragma unroll
    for (int u = 0; u < UB; u++) {
      const int s = s0 + u * XA_WAVES;
      if (s < nsteps) {
#pragma unroll
        for (int i = 0; i < 2 * NB; i++) {
          if constexpr (ACT) {
            xv[b][u][i] = silu_mul8<T>(xv[b][u][i], uv[b][u][i]);
            if (row_real[i]) __builtin_nontemporal_store(xv[b][u][i], (lf_u32x4*)(act_out + erow[i] + s * 64));
          }
          lf_u32x4 kept = xv[b][u][i];
          if constexpr (GEN) {
            uint32_t bits = 0xffu;
            if (thr > 0) kept &= draw8((uint64_t)(erow[i] + s * 64) >> 3, thr, seed_lo, seed_hi, bits);   // (p = 0: everything is kept)
            if (mask_bits) {
              // this lane's eight bits are byte lg of the row's eight bytes of the step: the four lanes of a quad join
              // theirs (two cross-lane moves) and one of them stores the dword
              uint32_t w = bits << (8 * (lg & 3));
              w |= (uint32_t)__builtin_amdgcn_mov_dpp((int)w, 0xB1, 0xf, 0xf, true);   // lanes 1 0 3 2
              w |= (uint32_t)__builtin_amdgcn_mov_dpp((int)w, 0x4E, 0xf, 0xf, true);   // lanes 2 3 0 1
              if (row_real[i] && (lg & 3) == 0) *(uint32_t*)(mask_out + ((erow[i] + s * 64) >> 3)) = w;
            } else {
              if (row_real[i]) *(lf_u32x2*)(mask_out + erow[i] + s * 64) = expand_keep8(bits);
            }
          } else {
            if (use_mask) kept = mask_bits ? kept & select8(mv[b][u][i][0]) : apply_mask8(kept, mv[b][u][i]);
          }
          *(lf_u32x4*)(patch + (i >> 1) * 2048 + wr_off[i & 1]) = kept;
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
          for (int c = 0; c < RT; c++) *(lf_u32x4*)(patch + (NB + c) * 2048 + wr_off[i]) = av[b][u][c][i];
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const int fo = rd_row + (((h * 4 + qq) ^ rd_key) << 4);
          lf_u32x4 af[RT];
#pragma unroll
          for (int c = 0; c < RT; c++) af[c] = *(const lf_u32x4*)(patch + (NB + c) * 2048 + fo);
#pragma unroll
          for (int nb = 0; nb < NB; nb++) {
            const lf_u32x4 xf = *(const lf_u32x4*)(patch + nb * 2048 + fo);
#pragma unroll
            for (int c = 0; c < RT; c++) acc[nb][c] = Mfma16<T>::run(xf, af[c], acc[nb][c]);
          }
        }
      }
    }
  };
  using Set0 = std::integral_constant<int, 0>;
  using Set1 = std::integral_constant<int, NSET - 1>;
  constexpr int STRIDE = XA_WAVES * UB;   // steps between a wave's consecutive batches
  if constexpr (NSET == 1) {
    for (int s0 = wave; s0 < nsteps; s0 += STRIDE) {
      load_batch(Set0{}, s0);
      use_batch(Set0{}, s0);
    }
  } else {
    load_batch(Set0{}, wave);
    for (int s0 = wave; s0 < nsteps; s0 += 2 * STRIDE) {
      load_batch(Set1{}, s0 + STRIDE);      // (steps beyond the row's end are skipped inside)
      use_batch(Set0{}, s0);
      load_batch(Set0{}, s0 + 2 * STRIDE);
      use_batch(Set1{}, s0 + STRIDE);
    }
  }
  __syncthreads();  // every wave is done with its patches
  // C layout: lane holds column (lane & 15), rows 4*(lane >> 4) + e
#pragma unroll
  for (int nb = 0; nb < NB; nb++)
#pragma unroll
    for (int c = 0; c < RT; c++)
#pragma unroll
      for (int e = 0; e < 4; e++) red[wave][nb * 16 + qq * 4 + e][c * 16 + li] = acc[nb][c][e];
  __syncthreads();
  const float mult = (use_mask && bi.p > 0.f) ? 1.f / (1.f - bi.p) : 1.f;  // no mask given: no dropout, whatever p says
  for (int o = tid; o < XA_ROWS * RT * 16; o += XA_WAVES * 64) {
    const int r = o / (RT * 16), c = o % (RT * 16);
    const int row = row0 + r;
    if (row < Mrows && c < R) {
      float v = 0.f;
      if (row - blk * ROWS < bi.valid && c < bi.rank) {
#pragma unroll
        for (int w = 0; w < XA_WAVES; w++) v += red[w][r][c];
        v *= mult;
      }
      ((uint16_t*)S)[(int64_t)row * R + c] = Mfma16<T>::cvt(v);
    }
  }
}

// S[row][col] = cast( mult * sum_p part[p][row][col] ), zero for padded rows / rank columns.
template <typename T>
__device__ __forceinline__ void reduce_rows_body(int bx, const float* __restrict__ part, T* __restrict__ out, int nparts, int M, int R,
                   int mode /*0: times 1/(1-p); 1: times scale*/, const LfSegTable seg) {
  // four consecutive columns per thread (R and every rank are multiples of 8): 16-byte loads
  const int Mrows = seg.table ? seg.n_blocks * ROWS : M;
  const int64_t idx = ((int64_t)bx * 256 + threadIdx.x) * 4;
  if (idx >= (int64_t)Mrows * R) return;
  const int row = (int)(idx / R), col = (int)(idx % R);
  const int blk = row / ROWS;
  const BlockInfo bi = block_info(seg, blk, M);
  lf_f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if (row - blk * ROWS < bi.valid && col < bi.rank) {
    v = sum_parts(part + idx, (int64_t)Mrows * R, nparts);
    v *= (mode == 0) ? (bi.p > 0.f ? 1.f / (1.f - bi.p) : 1.f) : bi.scale;
  }
  *(lf_u32x2*)((uint16_t*)out + idx) = pack4<T>(v);
}

// out_s = cast( mult * sum over parts of part[...] ) for segment s = blockIdx.y.
//   transposed == 0 (dB): parts are the segment's chunks, part[(s*max_chunks + ch)][n][R] -> out [rows, rank]
//   transposed == 1 (dA): parts are the segment's chunks, part[(s*max_chunks + ch)][R][rows] -> out [rank, rows]
//   mult_mode 0: segment scale ; 1: 1/(1-p) of the segment ; 2: none (no keep-mask was given: no dropout).
template <typename T>
__device__ __forceinline__ void reduce_segments_body(int bx, int s, const float* __restrict__ part, int rows, int R, int transposed, int mult_mode, int M,
                       int group, int max_chunks, const LfSegTable seg) {
  const int rank = seg.rank[s];
  const int64_t idx = ((int64_t)bx * 256 + threadIdx.x) * 4;  // four consecutive outputs of [rows, rank] or [rank, rows]
  if (idx >= (int64_t)rows * rank) return;
  int b0, b1;
  segment_blocks(seg, s, M, b0, b1);
  float mult;
  if (mult_mode == 2) {
    mult = 1.f;
  } else if (seg.table == nullptr) {
    mult = mult_mode == 0 ? seg.scale : (seg.p > 0.f ? 1.f / (1.f - seg.p) : 1.f);
  } else {
    mult = mult_mode == 0 ? (seg.block_scale ? seg.block_scale[b0] : 1.f)
                          : ((seg.block_p && seg.block_p[b0] > 0.f) ? 1.f / (1.f - seg.block_p[b0]) : 1.f);
  }
  lf_f32x4 v;
  const int nch = (b1 - b0 + group - 1) / group;
  if (!transposed) {
    const int n = (int)(idx / rank), r = (int)(idx % rank);
    v = sum_parts(part + (int64_t)s * max_chunks * rows * R + (int64_t)n * R + r, (int64_t)rows * R, nch);
  } else {
    const int r = (int)(idx / rows), k = (int)(idx % rows);
    v = sum_parts(part + (int64_t)s * max_chunks * R * rows + (int64_t)r * rows + k, (int64_t)R * rows, nch);
  }
  *(lf_u32x2*)((uint16_t*)seg.out[s] + idx) = pack4<T>(v * mult);
}

template <typename T>
__global__ void __launch_bounds__(256)
reduce_segments_kernel(const float* __restrict__ part, int rows, int R, int transposed, int mult_mode, int M,
                       int group, int max_chunks, const LfSegTable seg) {
  reduce_segments_body<T>((int)blockIdx.x, (int)blockIdx.y, part, rows, R, transposed, mult_mode, M, group, max_chunks, seg);
}

// Second stage of dys_dyb in one launch: blocks [0, nb_rows) reduce the dS partials, the rest the
// dB partials (nb_seg blocks per segment).
template <typename T>
__global__ void __launch_bounds__(256)
reduce_ds_db_kernel(const float* __restrict__ ds_part, T* __restrict__ dS, int nparts, int M, int R, int nb_rows,
                    const float* __restrict__ db_part, int N, int nb_seg, int group, int max_chunks, const LfSegTable seg) {
  const int b = blockIdx.x;
  if (b < nb_rows) {
    reduce_rows_body<T>(b, ds_part, dS, nparts, M, R, 1, seg);
  } else {
    const int c = b - nb_rows;
    reduce_segments_body<T>(c % nb_seg, c / nb_seg, db_part, N, R, 0, 0, M, group, max_chunks, seg);
  }
}

// ---- dys_dyb.  grid (n_seg * max_chunks, n_slices).  Workgroup (s, ch, ns): the tiles of N slice ns (balanced, 2 .. TPW
// tiles) and chunk ch of segment s (chunks are balanced too); pairs (block, tile) in block-major order.  A load group
// is the dY tile and its B tile [64, rank]; the S block of a row block comes with the block's first tile, into one of
// two buffers.  Per pair:
//   dS partial [128, R] += dY_tile * B_tile      (registers over the slice; stored when the block ends)
//   dB partial [64, R]  += dY_tile^T * S_block    (registers over ALL blocks of the chunk; stored at the end)
// The stores of a block's dS partial are vector memory operations like the loads: the group counts that follow them
// wait for more than they must (the ring runs empty once per block), never for less.
template <typename T, int RT, int TPW, int NS>
__global__ void __launch_bounds__(256, RT >= 4 ? 1 : 2)
lora_dys_dyb_ring_kernel(const T* __restrict__ dY, const T* __restrict__ S, float* __restrict__ ds_part, float* __restrict__ db_part,
                         int M, int N, int R, int n_slices, int group, int max_chunks, const LfSegTable seg) {
  constexpr int NIB = RT >= 2 ? RT / 2 : 1;         // B tile: 64 rows of RT*32 bytes (a 4 KB region at rank 16: all threads fetch)
  constexpr int BT = NIB * 4096;
  constexpr int STAGE = TILE_BYTES + BT;
  constexpr int SIDE = ROWS * RT * 32;
  constexpr int G = 4 + NIB;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  char* ring = lds;
  char* side = lds + NS * STAGE;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  const int s = blockIdx.x / max_chunks, ch = blockIdx.x % max_chunks, sl = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wave = to_sgpr(tid >> 6);
  const int li = lane & 15, qq = lane >> 4, j4 = li >> 2, c4 = li & 3;
  int b0, b1, bb0, bb1;
  segment_blocks(seg, s, M, b0, b1);
  chunk_blocks(b0, b1, group, ch, bb0, bb1);
  if (bb0 >= bb1) return;  // this segment has fewer chunks (uniform for the whole workgroup)
  const int rank = seg.rank[s];
  const T* __restrict__ Bl = (const T*)seg.ptr[s];
  const int64_t Mrows = seg.table ? (int64_t)seg.n_blocks * ROWS : M;
  const int T64 = N / 64;
  const int t0 = sl * (T64 / n_slices) + min(sl, T64 % n_slices);
  const int nt = T64 / n_slices + (sl < T64 % n_slices ? 1 : 0);
  const int ns = min(NS, nt + 1);   // stages in use

  uint32_t yv[4], bv[NIB], sv[RT];
  tile_voffs(yv, N, tid);
  side_voffs<RT, NIB>(bv, rank, rank, tid);
  side_voffs<RT, RT>(sv, R, R, tid);

  // Load group of the next pair into stage `ist`; behind the last pair the last tile is ordered again.  The windows
  // move with the pair (byte pointers and bytes left up to the end of the matrix): a few scalar additions per group.
  int ib = bb0, ij = 0, ist = 0;
  const char* yb = (const char*)(dY + (int64_t)bb0 * ROWS * N + (int64_t)t0 * 64);
  int64_t yleft = (((int64_t)Mrows - (int64_t)bb0 * ROWS) * N - (int64_t)t0 * 64) * 2;
  const char* bp = (const char*)(Bl + (int64_t)t0 * 64 * rank);
  int64_t bleft = ((int64_t)N - (int64_t)t0 * 64) * rank * 2;
  const char* sb = (const char*)(S + (int64_t)bb0 * ROWS * R);
  int64_t sleft = ((int64_t)Mrows - (int64_t)bb0 * ROWS) * R * 2;
  const int64_t slast = (int64_t)to_sgpr(seg.table ? seg.table[3 * (b1 - 1) + 1] : ROWS) * R * 2;   // (as in the da kernel)
  const int64_t ynext = (int64_t)ROWS * N * 2 - (int64_t)nt * 128;   // from behind a block's last tile to the next block's first
  const int64_t bstep = (int64_t)64 * rank * 2;
  auto issue = [&]() {
    tile_dma(window_rsrc(yb, yleft), yv, lds0 + ist * STAGE, wave);
    side_dma<NIB>(window_rsrc(bp, bleft), bv, lds0 + ist * STAGE + TILE_BYTES, wave);
    if (ij == 0 && ib < bb1) side_dma<RT>(window_rsrc(sb, ib == b1 - 1 ? min(sleft, slast) : sleft), sv, lds0 + NS * STAGE + ((ib - bb0) & 1) * SIDE, wave);
    ist = ist + 1 == ns ? 0 : ist + 1;
    if (ib < bb1) {
      if (++ij < nt) {
        yb += 128, yleft -= 128;
        bp += bstep, bleft -= bstep;
      } else if (ib + 1 < bb1) {
        ij = 0, ib++;
        yb += 128 + ynext, yleft -= 128 + ynext;
        bp -= (nt - 1) * bstep, bleft += (nt - 1) * bstep;
        sb += ROWS * R * 2, sleft -= ROWS * R * 2;
      } else {
        ib = bb1;   // the cursor stays on the last tile
      }
    }
  };
#pragma unroll 1
  for (int i = 0; i < ns - 1; i++) issue();

  lf_f32x4 acc_db[TPW][RT];
#pragma unroll
  for (int t = 0; t < TPW; t++)
#pragma unroll
    for (int c = 0; c < RT; c++) acc_db[t][c] = lf_f32x4{0.f, 0.f, 0.f, 0.f};

  int cst = 0;
  for (int b = bb0; b < bb1; b++) {
    const char* scur = side + ((b - bb0) & 1) * SIDE;
    lf_f32x4 acc_ds[2][RT];
    lf_u32x4 sf[4][RT];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
      for (int c = 0; c < RT; c++) acc_ds[a][c] = lf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < TPW; t++) {
      if (t < nt) {
        wait_groups<G>(ns - 2);
        ring_barrier();
        issue();
        const char* ycur = ring + cst * STAGE;
        const char* bcur = ycur + TILE_BYTES;
        // All fragments of the tile first, then the MFMAs (one wave per SIMD at rank 64: nothing else hides the LDS
        // latency).  dS += dY_tile * B_tile: a = dY row fragment, b = B^T through the transpose read; dB tile:
        // D[n][r] += sum_m dY[m][n] S[m][r], wave w owns columns 16w..16w+15 of the tile
        lf_u32x4 yf[2][2], bf[2][RT], yt[4];
        if (t == 0) {   // the S fragments serve every tile of the block
#pragma unroll
          for (int kk = 0; kk < 4; kk++)
#pragma unroll
            for (int c = 0; c < RT; c++) sf[kk][c] = side_tr8<RT>(scur, kk * 32 + qq * 8 + j4, c, c4);
        }
#pragma unroll
        for (int step = 0; step < 2; step++) {
#pragma unroll
          for (int rt = 0; rt < 2; rt++) yf[step][rt] = tile_row_frag(ycur, wave * 32 + rt * 16 + li, step * 4 + qq);
#pragma unroll
          for (int c = 0; c < RT; c++) bf[step][c] = side_tr8<RT>(bcur, step * 32 + qq * 8 + j4, c, c4);
        }
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
          const int mrow = kk * 32 + qq * 8 + j4;
          yt[kk] = tile_tr_frag(ycur, mrow, wave * 16 + 4 * c4);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int step = 0; step < 2; step++)
#pragma unroll
          for (int c = 0; c < RT; c++)
#pragma unroll
            for (int rt = 0; rt < 2; rt++) acc_ds[rt][c] = Mfma16<T>::run(yf[step][rt], bf[step][c], acc_ds[rt][c]);
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
#pragma unroll
          for (int c = 0; c < RT; c++) acc_db[t][c] = Mfma16<T>::run(yt[kk], sf[kk][c], acc_db[t][c]);
        __builtin_amdgcn_sched_barrier(0);
        cst = cst + 1 == ns ? 0 : cst + 1;
      }
    }
    float* dso = ds_part + (int64_t)sl * Mrows * R;
#pragma unroll
    for (int rt = 0; rt < 2; rt++)
#pragma unroll
      for (int c = 0; c < RT; c++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int64_t row = (int64_t)b * ROWS + wave * 32 + rt * 16 + qq * 4 + e;
          if (row < Mrows && c * 16 < R) dso[row * R + c * 16 + li] = acc_ds[rt][c][e];
        }
  }
  wait_vm<0>();   // the unconsumed loads behind the last pair must not land in another workgroup's LDS
  // C layout: column (r) = lane & 15, rows (n) = 4*(lane >> 4) + e
  float* dbo = db_part + (((int64_t)s * max_chunks + ch) * N + (int64_t)t0 * 64) * R;
#pragma unroll
  for (int t = 0; t < TPW; t++)
    if (t < nt) {
#pragma unroll
      for (int c = 0; c < RT; c++)
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (c * 16 < R) dbo[(int64_t)(t * 64 + wave * 16 + qq * 4 + e) * R + c * 16 + li] = acc_db[t][c][e];
    }
}

}  // namespace

// ---- work split of the ring kernels.  Workgroups (slice x chunk) of w tiles each run on `slots` resident slots; the
// pass lasts about as long as its busiest slot.  Two upper bounds of that (in tiles): whole rounds of the largest
// workgroup, and the list-scheduling bound sum / slots + largest; the smaller one is the estimate (ring_us).
// Of one chunk length, independent of the slices.  busy: workgroups per slice on the busiest of the eight XCDs when the grid is [segments * max_chunks, slices] and an id's XCD is its remainder:
// columns beyond a segment's last chunk end at once, and where the row of the grid is a multiple of 2, 4 or 8 the others can share a few remainders.
struct GroupStats { long chunks, total; int max_chunks, big; double busy; };
static GroupStats group_stats(const int* blocks, int nseg, int g) {
  GroupStats r{0, 0, 1, 0, 0.0};
  for (int s = 0; s < nseg; s++) {
    const int c = (blocks[s] + g - 1) / g;
    if (c <= 0) continue;
    r.chunks += c;
    r.max_chunks = c > r.max_chunks ? c : r.max_chunks;
    const int sz = (blocks[s] + c - 1) / c;
    r.big = sz > r.big ? sz : r.big;
    r.total += blocks[s];
  }
  const int period = std::gcd(nseg * r.max_chunks, 8);
  long at[8] = {};
  for (int s = 0; s < nseg; s++) {
    const int c = (blocks[s] + g - 1) / g;
    for (int q = 0; q < period; q++) at[(s * r.max_chunks + q) % period] += c / period + (q < c % period ? 1 : 0);
  }
  r.busy = *std::max_element(at, at + period) * period / 8.0;
  return r;
}
// Microseconds of a pass and its second stage: tiles and row blocks of the busiest slot, rounds of workgroups, partials in MB (dS: one [rows, R] slab per slice; dB or dA: one slab per
// chunk), the side operand that every workgroup fetches per block in MB, and the share of a slot if all tiles were spread evenly.  Fitted, by rank tiling, to 35 plans each of 2423
// batches (700 - 16400 rows in 1 - 8 segments, 1024 - 14336 columns): on shapes that were not fitted dys_dyb is 5.5 % behind the best plan timed, dA 2.4 % and without a mask 1.8 %;
// the bytes moved, by which plans were chosen before, 8.5, 3.9 and 5.9 %.  (The eight-tile slices of the byte model leave three quarters of the compute units idle at 2048 x 4096.)
// Then each model was put on the scale of a second campaign (a factor and a constant, which leave its choice of plans alone): there these two passes, direct dA and the short
// backward below were timed the same way, twelve launches a graph, 10200 batches (60 - 16400 rows in 1 - 8 segments, N 1024 - 14336, K 1024 - 8192, ranks 8 - 128, with keep bits
// and without).  On a quarter of them that was not fitted dys_dyb is 8 % off at ranks to 32 and 13 % above, dA 5 - 10 %, and the two in a row take their sum.  Measured (model), us, x
// 4096 columns at rank 16: dys_dyb of 1000 rows 10.7 (10.7), 2048 13.6 (13.3), 3000 14.3 (15.5); dA with keep bits 9.3 (9.9), 13.6 (12.5), 14.7 (14.8), without 7.7 (8.0), 9.6 (9.7),
// 10.5 (11.0).
struct RingModel { double fixed, tile, block, round, ds, slab, side, even; };
static double ring_us(const RingModel& m, const GroupStats& r, int T, int nsl, int slots, bool chunk_rows, double ds_mb, double slab_mb, double side_mb) {
  const int t_max = (T + nsl - 1) / nsl;
  // (chunk_rows: the grid of `busy`.  eight adapters of 7, 2, 2, 2, 2, 1, 1 and 2 blocks, 10752 columns, rank 64: 231 workgroups in chunks of two, four columns on each of two XCDs, 71.7 us; 456 in chunks
  // of one 50.7.  With the busiest XCD's rounds the plan is 1.2 % behind the best one timed at ranks 33 - 64 and 0.9 % above, with the chip's 3.1 and 1.9)
  const double chip = (double)((r.chunks * nsl + slots - 1) / slots), rounds = chunk_rows ? std::max(chip, std::ceil(std::ceil(r.busy * nsl) / (slots / 8))) : chip;
  const double even = (double)r.total * T / slots, largest = (double)r.big * t_max;
  const double span = std::max(std::min(rounds * largest, even + largest), even);
  const double blocks = std::max(std::min(rounds * r.big, (double)r.total * nsl / slots + r.big), 1.0);
  return m.fixed + m.tile * span + m.block * blocks + m.round * rounds + m.ds * ds_mb + m.slab * slab_mb + m.side * side_mb + m.even * even;
}
static int model_of(int rt) { return rt >= 8 ? 3 : rt >= 4 ? 2 : rt >= 2 ? 1 : 0; }
static const RingModel kDysModel[4] = {{5.779, 0.184, 0.263, 1.256, 0.090, 0.477, 0.677, 1.194}, {5.803, 0.358, 0.656, 1.130, 0.251, 0.564, 0.362, 0.602},
                                       {3.217, 0.643, 0.223, 4.497, 0.466, 0.504, 0.310, 0.0}, {6.341, 0.956, 0.571, 4.305, 0.188, 0.298, 0.275, 0.080}};
static const RingModel kDaModel[2][4] = {{{4.711, 0.256, 0.058, 0.496, 0.0, 0.892, 0.034, 0.694}, {5.569, 0.227, 0.282, 0.0, 0.0, 0.626, 0.082, 0.607},
                                          {4.813, 0.334, 0.0, 1.095, 0.0, 0.405, 0.055, 0.759}, {3.906, 0.758, 0.003, 3.348, 0.0, 0.454, 0.077, 0.0}},
                                         {{1.255, 0.733, 0.016, 4.521, 0.0, 0.559, 0.407, 0.999}, {5.160, 0.711, 0.105, 0.946, 0.0, 0.731, 0.412, 0.0},
                                          {4.415, 0.829, 0.0, 1.720, 0.0, 0.575, 0.176, 0.0}, {4.659, 1.024, 0.025, 3.297, 0.0, 0.504, 0.118, 0.0}}};   // without and with a keep-mask
static void seg_block_counts(int M, const LfSegTable& seg, int* blocks, int& nseg) {
  nseg = seg.table ? seg.n_seg : 1;
  for (int s = 0; s < nseg; s++) {
    const int b0 = seg.table ? seg.first_block[s] : 0;
    const int b1 = seg.table ? ((s + 1 < nseg) ? seg.first_block[s + 1] : seg.n_blocks) : (M + ROWS - 1) / ROWS;
    blocks[s] = b1 - b0;
  }
}
static const int kGroups[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 64};
constexpr int kNGroups = 11;
// Chunk lengths worth pricing: up to the longest segment (longer ones repeat its figures).
static int all_group_stats(const int* blocks, int nseg, GroupStats (&st)[kNGroups]) {
  int longest = 0;
  for (int s = 0; s < nseg; s++) longest = blocks[s] > longest ? blocks[s] : longest;
  int n = 0;
  for (; n < kNGroups; n++) {
    st[n] = group_stats(blocks, nseg, kGroups[n]);
    if (kGroups[n] >= longest) return n + 1;
  }
  return n;
}

constexpr int dysr_tpw(int rt) { return rt >= 8 ? 4 : rt >= 2 ? 12 : 16; }   // dB accumulators: TPW * RT * 4 registers, next to 8 * RT of dS
constexpr int dysr_ns(int rt) { return rt == 4 ? 5 : 3; }   // (rank 128: three stages of 32 KB and two S blocks of 32 KB are all of the LDS)
static int dysr_smem(int rt) { return dysr_ns(rt) * (TILE_BYTES + (rt >= 2 ? rt / 2 : 1) * 4096) + 2 * ROWS * rt * 32; }
struct DysRingPlan { int n_slices, group, max_chunks; double us; };   // us: by the model above
// The cheapest plan whose partials take at most `limit` bytes (if none does: the cheapest of all).
static DysRingPlan dysr_plan_of(int M, int N, int R, const int* blocks, int nseg, const LfSegTable& seg, size_t limit) {
  const int rt = rt_of(R), T = N / 64;
  const int64_t rows = seg.table ? (int64_t)seg.n_blocks * ROWS : M;
  const int slots = lds_slots(dysr_smem(rt));
  DysRingPlan best{1, 1, 1, 1e300};
  if (T < 2) return best;   // fewer than two column tiles: nothing to split (and no division by a zero slice count)
  GroupStats stats[kNGroups];
  const int ng = all_group_stats(blocks, nseg, stats);
  double best_cost = 1e300;
  bool best_fits = false;
  for (int t = dysr_tpw(rt); t >= 2; t--) {   // tiles of the longest slice -> fewest slices that reach it
    const int nsl = (T + t - 1) / t;
    if (nsl > T / 2 || (T + nsl - 1) / nsl != t) continue;
    for (int k = 0; k < ng; k++) {
      const GroupStats& st = stats[k];
      const double cost = ring_us(kDysModel[model_of(rt)], st, T, nsl, slots, true, 4e-6 * R * nsl * (double)rows, 4e-6 * R * (double)st.chunks * N,
                                  2e-6 * (double)st.chunks * nsl * kGroups[k] * ROWS * R);
      const bool fits = ((size_t)nsl * rows * R + (size_t)nseg * st.max_chunks * N * R) * sizeof(float) <= limit;
      if (fits == best_fits ? cost < best_cost : fits) { best_fits = fits; best_cost = cost; best = DysRingPlan{nsl, kGroups[k], st.max_chunks, cost}; }
    }
  }
  return best;
}

// (what the plans read: sizes, and the blocks of each segment)
struct PlanKey { int64_t v[5 + LF_MAX_SEG / 2]; };
static void plan_key(PlanKey& k, int M, int dim, int R, int what, size_t limit, const LfSegTable& seg, int* blocks, int& nseg) {
  seg_block_counts(M, seg, blocks, nseg);
  k = PlanKey{};
  k.v[0] = M, k.v[1] = dim, k.v[2] = R, k.v[3] = (int64_t)what << 32 | (seg.table != nullptr) << 16 | nseg, k.v[4] = (int64_t)limit;
  for (int s = 0; s < nseg; s++) k.v[5 + s / 2] |= (int64_t)(uint32_t)blocks[s] << 32 * (s & 1);
}
static DysRingPlan dysr_plan(int M, int N, int R, const LfSegTable& seg, size_t limit) {
  static thread_local LfMemo<DysRingPlan, 5 + LF_MAX_SEG / 2> memo;
  int blocks[LF_MAX_SEG], nseg;
  PlanKey k;
  plan_key(k, M, N, R, 0, limit, seg, blocks, nseg);
  return memo.get(k.v, [&] { return dysr_plan_of(M, N, R, blocks, nseg, seg, limit); });
}

// (lora_stream.hip)
int lf_xa_stream_slices(int, int, int, bool, const LfSegTable&);
size_t lf_xa_stream_workspace(int, int, int, bool, const LfSegTable&);
int lf_launch_xa_ring(const void*, void*, int, int, int, const LfSegTable&, int, hipStream_t);
int lf_launch_xa_stream(const void*, const uint8_t*, uint8_t*, int, uint64_t, void*, float*, int, int, int, const LfSegTable&, int, hipStream_t);

// The products that the sliced pass (lora_stream.hip) is the faster one for, given memory for the slices' sums.  Microseconds below: mask drawn /
// keep bits read / no mask, this file's kernel against the sliced pass, launches replayed from a graph.
// - Above 64 rank columns, always: 64 x 1024 at rank 128 22.4 / 18.6 / 15.4 -> 10.2 / 8.7 / 8.0, 14000 x 8192 194 / 145 / 105 -> 92 / 81 / 53.
// - 33 to 64: this kernel reads A once per 64 rows and has a workgroup per 64 rows, each of which walks K alone.  Up to 48 of
//   them always (1000 x 4096 38 / 24 / 17 -> 12 / 10 / 9); beyond, the second stage and the partial sums cost a fixed part
//   and the slices give one that grows with K: the table.  One round of the chip full of workgroups (170 to 256) leaves nothing to
//   gain (16384 x 4096 44 / 30 / 27 against 46 / 31 / 28), a second round does (20000 x 4096 79 / 52 / 42 -> 58 / 43 / 35).  Without
//   a mask there is half as much to share, and K has to be twice as long.  Either side of the lines:
//     64 groups   K 1024  13.5/10.0/ 8.0 -> 11.4/ 9.7/ 8.8   2048  21.9/15.0/11.1 -> 14.4/11.5/10.1
//     110         K 1024  13.7/10.2/ 8.2 -> 14.4/11.3/10.1   1536  18.8/13.3/10.4 -> 17.3/12.9/10.7   3072 31.7/21.0/16.0 -> 23.4/17.5/15.3
//     141         K 1536  19.2/13.6/10.9 -> 18.5/14.5/12.4   2048  24.5/17.2/13.6 -> 22.6/16.5/14.0   4096 40.5/26.7/20.2 -> 34.1/22.8/19.9
//     192         K 4096  41.7/28.3/23.7 -> 38.7/28.9/24.8   8192  75.0/47.8/38.6 -> 65.6/46.2/39.8   14336 149/110/90 -> 111/100/82
//     219         K 8192  75.6/49.2/42.2 -> 77.9/64.4/49.7 (eight slices; two: 80.3/49.3/42.8)
// - To 32: up to 1024 rows from K = 4096 with a mask (300 rows at rank 16: K = 3072 8.8 / 6.1 -> 9.0 / 7.1, 4096 10.9 / 7.3 -> 8.9 / 7.2, 8192 19.1 /
//   11.6 -> 11.7 / 8.7; a second launch costs what a short K saves).  Without one, against lora_xa_ring_kernel (us, rank to 16 / to 32): 333 rows, K = 8192
//   6.8 / 7.4 -> 6.3 / 9.6, 14336 8.7 / 9.4 -> 12.1 / 17.0; 1000 rows, 8192 8.7 / 10.0 -> 8.4 / 10.7.  At 333 x 4096 and rank 32 the ring takes 5.7
//   against 6.4 when X comes from the caches, but inside a forward whose weight has pushed X out of them (117 MB, 14336 columns) the sliced
//   pass's 96 workgroups fetch it sooner than 21 and the whole forward takes 57.8 against 58.2: there it stays sliced.
// The same choice for every mask format, drawn or read: S does not depend on how the mask came.
static bool lf_xa_streams(int M, int K, int R, bool masked, const LfSegTable& seg) {
  const int64_t rows = seg.table ? (int64_t)seg.n_blocks * ROWS : M;
  if (R > 64) return true;
  if (R > 32) {
    const int64_t groups = (rows + 63) / 64;
    if (groups <= 48 || groups > 256) return true;
    const int k_min = groups <= 64 ? 1024 : groups <= 128 ? 1536 : groups <= 170 ? 2048 : groups <= 192 ? 8192 : 1 << 30;
    return K >= (masked || k_min == 1 << 30 ? k_min : 2 * k_min);
  }
  return rows <= 1024 && K >= (masked ? 4096 : R <= 16 ? 8320 : rows <= 512 ? 4096 : 8192);
}
// ... and those it takes.  Without the memory (entry points that have no workspace to give, or too small a one) this file's kernel
// runs to rank 64; above, and where a single slice needs none, the sliced pass all the same.
// A mask read from an address that the direct loads do not take also stays with this file's kernel to rank 64.
bool lf_xa_takes_stream(int M, int K, int R, const uint8_t* mask, int mask_bits, bool drawn, const LfSegTable& seg, const void* ws, size_t ws_bytes) {
  const bool masked = mask != nullptr || drawn;
  if (R <= 64 && mask_off_grid(mask, mask_bits)) return false;
  return lf_xa_streams(M, K, R, masked, seg) && (R > 64 || lf_xa_stream_slices(M, K, R, masked, seg) == 1 ||
                                                 (ws != nullptr && ws_bytes >= lf_xa_stream_workspace(M, K, R, masked, seg)));
}
// The products without a mask that lora_xa_ring_kernel (lora_stream.hip) is the faster one for: ranks to 32 while there are no more than one
// workgroup per compute unit -- its LDS holds one at a time.  This file's kernel against it, us, rank 16: 333 x 2048 3.8 -> 3.6, 1000 x 4096 6.6 -> 5.3,
// 4096 x 4096 9.2 -> 8.3, 4096 x 14336 27.7 -> 24.9; 8192 rows 15.0 -> 14.2 at K = 4096 but 9.4 -> 9.8 at 2048 and 29.7 -> 30.4 at 8192.  X or A off a
// dword stays with this file's kernel.
static bool lf_xa_rings(const void* X, int M, int R, const LfSegTable& seg) {
  if (R > 32 || (seg.table ? (int64_t)seg.n_blocks * ROWS : M) > 256 * 16) return false;
  uintptr_t at = (uintptr_t)X;
  for (int i = 0; i < (seg.table ? seg.n_seg : 1); i++) at |= (uintptr_t)seg.ptr[i];
  return (at & 3) == 0;
}
size_t lf_xa_workspace(int M, int K, int R, const LfSegTable& seg) {
  size_t n = 0;
  for (const bool masked : {false, true})
    if (lf_xa_streams(M, K, R, masked, seg)) n = std::max(n, lf_xa_stream_workspace(M, K, R, masked, seg));
  return n;
}

template <typename T, int RT>
static int xa_launch(const void* X, const void* U, int64_t ldx, void* act_out, const uint8_t* mask, uint8_t* mask_out, int mask_bits,
                     uint64_t seed, void* S, int M, int K, int R, int64_t rows, const LfSegTable& seg, hipStream_t st) {
  const bool gen = mask_out != nullptr, act = U != nullptr;
  const int wg_rows = xa_rows(RT, act);
  const unsigned grid = (unsigned)((rows + wg_rows - 1) / wg_rows);
  const uint32_t lo = gen ? (uint32_t)seed : 0u, hi = gen ? (uint32_t)(seed >> 32) : 0u;
#define LF_XA(GEN, ACT)                                                                                              \
  return lf_launch((lora_xa_kernel<T, RT, GEN, ACT>), dim3(grid), dim3(XA_WAVES * 64), 0, st, (const T*)X,       \
                   (const T*)U, ldx, (T*)act_out, mask, mask_out, mask_bits, lo, hi, (T*)S, M, K, R, seg)
  if (gen && act) LF_XA(true, true);
  if (act) LF_XA(false, true);
  if (gen) LF_XA(true, false);
  LF_XA(false, false);
#undef LF_XA
}

template <typename T>
static int xa_impl(const void* X, const void* U, int64_t ldx, void* act_out, const uint8_t* mask, uint8_t* mask_out, int mask_bits,
                   uint64_t seed, void* S, int M, int K, int R, const LfSegTable& seg, hipStream_t st) {
  const int nblk = n_row_blocks(M, seg);
  const int64_t rows = seg.table ? (int64_t)nblk * ROWS : M;
  switch (rt_of(R)) {
    case 1: return xa_launch<T, 1>(X, U, ldx, act_out, mask, mask_out, mask_bits, seed, S, M, K, R, rows, seg, st);
    case 2: return xa_launch<T, 2>(X, U, ldx, act_out, mask, mask_out, mask_bits, seed, S, M, K, R, rows, seg, st);
    case 4: return xa_launch<T, 4>(X, U, ldx, act_out, mask, mask_out, mask_bits, seed, S, M, K, R, rows, seg, st);
    default: return LF_ESHAPE;   // (lf_xa_takes_stream: above rank 64 the sliced pass, behind an activation pass of its own)
  }
}

// mask_out != nullptr: draw the keep-mask from `seed` (written to mask_out [rows, K]) instead of reading `mask`.
// U != nullptr: X and U are the gate and up halves (rows ldx elements apart) and the pass's input
// round16(round16(silu(X)) * U) is written to act_out [rows, K]; otherwise X [rows, K] is dense.
int lf_launch_xa(const void* X, const void* U, int64_t ldx, void* act_out, const uint8_t* mask, uint8_t* mask_out, int mask_bits,
                 uint64_t seed, void* S, void* ws, size_t ws_bytes, int M, int K, int R, const LfSegTable& seg, int dtype, hipStream_t st) {
  if (!X || !S || M <= 0 || K <= 0) return LF_EINVAL;
  if (K % 128 != 0 || R % 16 != 0 || R <= 0 || R > LF_MAX_RANK) return LF_ESHAPE;
  if (seg.table && seg.block_size_m != ROWS) return LF_ESHAPE;
  if (mask_out != nullptr && ((uintptr_t)mask_out & (mask_bits ? 3 : 7)) != 0) return LF_ESHAPE;
  if (U != nullptr) {
    if (!act_out) return LF_EINVAL;
    if (ldx < K || ldx % 8 != 0 || (((uintptr_t)X | (uintptr_t)U | (uintptr_t)act_out) & 15) != 0) return LF_ESHAPE;
  } else {
    ldx = K;
    const bool masked = mask != nullptr || mask_out != nullptr;
    if ((dtype == LF_BF16 || dtype == LF_F16) && lf_xa_takes_stream(M, K, R, mask, mask_bits, mask_out != nullptr, seg, ws, ws_bytes))
      return lf_launch_xa_stream(X, mask, mask_out, mask_bits, seed, S, ws_bytes >= lf_xa_stream_workspace(M, K, R, masked, seg) ? (float*)ws : nullptr, M,
                                 K, R, seg, dtype, st);
    if ((dtype == LF_BF16 || dtype == LF_F16) && !masked && lf_xa_rings(X, M, R, seg)) return lf_launch_xa_ring(X, S, M, K, R, seg, dtype, st);
  }
  if (dtype == LF_BF16) return xa_impl<__bf16>(X, U, ldx, act_out, mask, mask_out, mask_bits, seed, S, M, K, R, seg, st);
  if (dtype == LF_F16) return xa_impl<_Float16>(X, U, ldx, act_out, mask, mask_out, mask_bits, seed, S, M, K, R, seg, st);
  return LF_EINVAL;
}

size_t lf_dys_dyb_workspace(int M, int N, int R, const LfSegTable& seg, size_t limit) {
  const int nblk = n_row_blocks(M, seg);
  const int64_t rows = seg.table ? (int64_t)nblk * ROWS : M;
  const int nseg = seg.table ? seg.n_seg : 1;
  const DysRingPlan pl = dysr_plan(M, N, R, seg, limit);
  return ((size_t)pl.n_slices * rows * R + (size_t)nseg * pl.max_chunks * N * R) * sizeof(float);
}

template <typename T, int RT>
static int dysr_launch(const void* dY, const void* S, float* ds_part, float* db_part, int M, int N, int R, const DysRingPlan& pl,
                       int nseg, const LfSegTable& seg, hipStream_t st) {
  auto kern = lora_dys_dyb_ring_kernel<T, RT, dysr_tpw(RT), dysr_ns(RT)>;
  const int smem = dysr_smem(RT);
  static LfLdsFlags lds_ok;
  if (!lf_allow_lds(kern, smem, lds_ok)) return LF_ELAUNCH;
  return lf_launch(kern, dim3(nseg * pl.max_chunks, pl.n_slices), dim3(256), smem, st, (const T*)dY, (const T*)S, ds_part, db_part, M, N, R,
                   pl.n_slices, pl.group, pl.max_chunks, seg);
}

template <typename T>
static int dys_dyb_impl(const void* dY, const void* S, void* dS, void* ws, size_t limit, int M, int N, int R, const LfSegTable& seg, hipStream_t st) {
  const int nblk = n_row_blocks(M, seg);
  const int64_t rows = seg.table ? (int64_t)nblk * ROWS : M;
  const int nseg = seg.table ? seg.n_seg : 1;
  float* ds_part = (float*)ws;   // [slices][rows][R], then the dB partials [nseg * max_chunks][N][R]
  const DysRingPlan pl = dysr_plan(M, N, R, seg, limit);
  float* db_part = ds_part + (int64_t)pl.n_slices * rows * R;
  int rc;
  switch (rt_of(R)) {
    case 1: rc = dysr_launch<T, 1>(dY, S, ds_part, db_part, M, N, R, pl, nseg, seg, st); break;
    case 2: rc = dysr_launch<T, 2>(dY, S, ds_part, db_part, M, N, R, pl, nseg, seg, st); break;
    case 4: rc = dysr_launch<T, 4>(dY, S, ds_part, db_part, M, N, R, pl, nseg, seg, st); break;
    default: rc = dysr_launch<T, 8>(dY, S, ds_part, db_part, M, N, R, pl, nseg, seg, st); break;
  }
  if (rc != LF_OK) return rc;
  const int64_t n = rows * R;
  int maxrank = 0;
  for (int s = 0; s < nseg; s++) maxrank = seg.rank[s] > maxrank ? seg.rank[s] : maxrank;
  const int64_t nout = (int64_t)N * maxrank;
  const int nb_rows = (int)((n + 1023) / 1024), nb_seg = (int)((nout + 1023) / 1024);  // four outputs per thread
  return lf_launch((reduce_ds_db_kernel<T>), dim3((unsigned)(nb_rows + nb_seg * nseg)), dim3(256), 0, st, (const float*)ds_part,
                     (T*)dS, pl.n_slices, M, R, nb_rows, (const float*)db_part, N, nb_seg, pl.group, pl.max_chunks, seg);
}

int lf_launch_dys_dyb(const void* dY, const void* S, void* dS, void* ws, size_t ws_bytes, size_t limit, int M, int N, int R,
                      const LfSegTable& seg, int dtype, hipStream_t st) {
  if (!dY || !S || !dS || M <= 0 || N <= 0) return LF_EINVAL;
  if (N % 128 != 0 || R % 16 != 0 || R <= 0 || R > LF_MAX_RANK) return LF_ESHAPE;
  if (seg.table && seg.block_size_m != ROWS) return LF_ESHAPE;
  const int nseg = seg.table ? seg.n_seg : 1;
  for (int s = 0; s < nseg; s++) if (!seg.out[s] || !seg.ptr[s] || seg.rank[s] % 8 != 0 || seg.rank[s] > R) return LF_EINVAL;
  for (int s = 0; s < nseg; s++) if (((uintptr_t)seg.out[s] & 7) != 0) return LF_ESHAPE;  // 8-byte stores of dB
  if (((uintptr_t)dS & 7) != 0) return LF_ESHAPE;
  if (!ws || ws_bytes < lf_dys_dyb_workspace(M, N, R, seg, limit)) return LF_EWORKSPACE;
  if (dtype == LF_BF16) return dys_dyb_impl<__bf16>(dY, S, dS, ws, limit, M, N, R, seg, st);
  if (dtype == LF_F16) return dys_dyb_impl<_Float16>(dY, S, dS, ws, limit, M, N, R, seg, st);
  return LF_EINVAL;
}

// Ring kernel shapes by rank tiles: tiles per slice (registers: TPW * RT * 4 accumulators) and ring depth (LDS: NS
// stages of 16 KB, 24 KB with a keep-mask, plus two dS blocks of RT * 4 KB; two workgroups per CU where that fits).
constexpr int da_ns(int rt, int maskfmt) {
  if (rt == 8) return maskfmt == 1 ? 4 : 5;
  return maskfmt ? (rt == 1 ? 3 : 5) : (rt == 4 ? 3 : 4);
}
static int da_ring_smem(int rt, int maskfmt) { return da_ns(rt, maskfmt) * (TILE_BYTES + da_mask_tile_bytes(maskfmt)) + 2 * ROWS * rt * 32; }
struct DaPlan { int n_slices, group, max_chunks; double us; };
// Slices of the K axis (balanced, 2 .. TPW tiles each) x chunks of `group` row blocks per segment, by the model above.  `limit`: as for dysr_plan.
static DaPlan da_plan_of(int K, int R, int maskfmt, const int* blocks, int nseg, size_t limit) {
  const int rt = rt_of(R), T = K / 64;
  const int slots = lds_slots(da_ring_smem(rt, maskfmt));
  DaPlan best{1, 1, 1, 1e300};
  if (T < 2) return best;   // as in dysr_plan
  GroupStats stats[kNGroups];
  const int ng = all_group_stats(blocks, nseg, stats);
  double best_cost = 1e300;
  bool best_fits = false;
  for (int t = da_tpw(rt); t >= 2; t--) {   // tiles of the longest slice -> fewest slices that reach it
    const int nsl = (T + t - 1) / t;
    if (nsl > T / 2 || (T + nsl - 1) / nsl != t) continue;
    for (int k = 0; k < ng; k++) {
      const GroupStats& st = stats[k];
      const double cost = ring_us(kDaModel[maskfmt != 0][model_of(rt)], st, T, nsl, slots, false, 0.0, 4e-6 * R * K * (double)st.chunks, 2e-6 * (double)st.chunks * nsl * kGroups[k] * ROWS * R);
      const bool fits = (size_t)nseg * st.max_chunks * R * K * sizeof(float) <= limit;
      if (fits == best_fits ? cost < best_cost : fits) { best_fits = fits; best_cost = cost; best = DaPlan{nsl, kGroups[k], st.max_chunks, cost}; }
    }
  }
  return best;
}

static DaPlan da_plan(int M, int K, int R, int maskfmt, const LfSegTable& seg, size_t limit) {
  static thread_local LfMemo<DaPlan, 5 + LF_MAX_SEG / 2, 32> memo;
  int blocks[LF_MAX_SEG], nseg;
  PlanKey k;
  plan_key(k, M, K, R, maskfmt, limit, seg, blocks, nseg);
  return memo.get(k.v, [&] { return da_plan_of(K, R, maskfmt, blocks, nseg, limit); });
}

size_t lf_da_workspace(int M, int K, int R, const LfSegTable& seg, size_t limit) {
  const int nseg = seg.table ? seg.n_seg : 1;
  // the launch plans with or without a keep-mask (one byte or one bit per element): room for any
  int max_chunks = 1;
  for (int fmt = 0; fmt < 3; fmt++) max_chunks = std::max(max_chunks, da_plan(M, K, R, fmt, seg, limit).max_chunks);
  return (size_t)nseg * max_chunks * R * K * sizeof(float);
}

// One launch without a second stage: a workgroup walks all row blocks of its segment over t tiles of columns and stores the sums as
// they are.  Alone on its compute unit, it has a deeper ring and more dS buffers than the two-stage form: what a walk of one or
// two tiles per block needs to keep loads on order.  It pays where segments have few blocks (a tile costs a workgroup 0.4 us, with a
// mask 0.9, one after the other) or the partials are large (high ranks, wide inputs).  Both sides in microseconds on one scale (ring_us): over its 14100 products direct is 6.5 % off,
// the choice takes 0.3 % more than the faster form of each, 2.8 % of them more than 3 % (worst 1.5 times).
// With keep bits, two-stage -> direct: 300 x 4096 rank 16 7.9 -> 7.7, four segments of 1280 x 4096 rank 64 13.6 -> 9.9; the other side of the line: 1000 x 4096 rank 16 in one
// segment 9.3 against 13.7, without a mask 7.7 against 9.5.
// (the same choice for every mask format: dA does not depend on how the mask came)
struct DaForm { int direct_slices; double us; };   // 0: two stages
static DaForm da_form(int M, int K, int R, bool masked, const LfSegTable& seg, size_t limit) {
  const int rt = rt_of(R), T = K / 64;
  const double m = masked, two_stage = T < 2 ? 0.0 : da_plan(M, K, R, masked ? 2 : 0, seg, limit).us;
  const DaForm staged{0, two_stage};
  if (T < 2) return staged;
  int blocks[LF_MAX_SEG], nseg, live = 0, big = 0;
  seg_block_counts(M, seg, blocks, nseg);
  for (int s = 0; s < nseg; s++) live += blocks[s] > 0, big = std::max(big, blocks[s]);
  if (live == 0) return staged;
  int t = rt == 8 ? 2 : 1;   // (with a mask the ring holds three stages at least: two dS buffers allow t + 1)
  while (t <= da_tpw(rt) && ((T + t - 1) / t) * live > 256) t++;   // one round of workgroups
  if (t > da_tpw(rt)) return staged;
  const int nsl = (T + t - 1) / t;
  const double tiles = (double)big * t;
  const double direct = 3.66 + 0.40 * m + 0.20 * rt + tiles * (0.305 + 0.466 * m + 0.049 * rt) + 0.357 * big + 0.9e-3 * tiles * nsl * live;
  return direct < two_stage ? DaForm{nsl, direct} : staged;
}

// (lora_da_direct.hip)  mask_fmt: the kernel's MASK
int lf_launch_da_direct(const void* X, const uint8_t* mask, int mask_fmt, const void* dS, int M, int K, int R, int n_slices, const LfSegTable& seg, const void* dY,
                        const void* S, int N, int n_slices_b, int dtype, hipStream_t st);

template <typename T, int RT, int MASK>
static int da_ring_launch(const void* X, const uint8_t* mask, const void* dS, float* part, int M, int K, int R, const DaPlan& pl,
                          int nseg, const LfSegTable& seg, hipStream_t st) {
  auto kern = lora_da_ring_kernel<T, RT, da_tpw(RT), da_ns(RT, MASK), MASK, 2, false>;
  const int smem = da_ring_smem(RT, MASK);
  static LfLdsFlags lds_ok;
  if (!lf_allow_lds(kern, smem, lds_ok)) return LF_ELAUNCH;
  return lf_launch(kern, dim3(pl.n_slices, pl.max_chunks, nseg), dim3(256), smem, st, (const T*)X, mask, (const T*)dS, part, M, K, R,
                   pl.n_slices, pl.group, pl.max_chunks, seg, DbOperands{});
}

template <typename T>
static int da_impl(const void* X, const uint8_t* mask, int mask_bits, const void* dS, void* ws, size_t limit, int M, int K, int R, const LfSegTable& seg,
                   hipStream_t st) {
  const int nseg = seg.table ? seg.n_seg : 1;
  float* part = (float*)ws;
  int rc;
  const int fmt = mask == nullptr ? 0 : mask_bits ? 2 : 1;
  const bool off_grid = fmt == 1 && mask_off_grid(mask, 0);   // (the same split, and the same sums)
  if (const int nsl = da_form(M, K, R, mask != nullptr, seg, limit).direct_slices)
    return lf_launch_da_direct(X, mask, off_grid ? 3 : fmt, dS, M, K, R, nsl, seg, nullptr, nullptr, 0, 0,
                               std::is_same_v<T, __bf16> ? LF_BF16 : LF_F16, st);
  const DaPlan pl = da_plan(M, K, R, fmt, seg, limit);
#define LF_DA_RING(RTV)                                                                                                   \
  rc = off_grid   ? da_ring_launch<T, RTV, 3>(X, mask, dS, part, M, K, R, pl, nseg, seg, st)                              \
       : fmt == 2 ? da_ring_launch<T, RTV, 2>(X, mask, dS, part, M, K, R, pl, nseg, seg, st)                              \
       : fmt == 1 ? da_ring_launch<T, RTV, 1>(X, mask, dS, part, M, K, R, pl, nseg, seg, st)                              \
                  : da_ring_launch<T, RTV, 0>(X, mask, dS, part, M, K, R, pl, nseg, seg, st)
  switch (rt_of(R)) {
    case 1: LF_DA_RING(1); break;
    case 2: LF_DA_RING(2); break;
    case 4: LF_DA_RING(4); break;
    default: LF_DA_RING(8); break;
  }
#undef LF_DA_RING
  if (rc != LF_OK) return rc;
  int maxrank = 0;
  for (int s = 0; s < nseg; s++) maxrank = seg.rank[s] > maxrank ? seg.rank[s] : maxrank;
  const int64_t nout = (int64_t)K * maxrank;
  return lf_launch((reduce_segments_kernel<T>), dim3((unsigned)((nout + 1023) / 1024), nseg), dim3(256), 0, st, (const float*)part, K, R, 1, mask != nullptr ? 1 : 2, M, pl.group, pl.max_chunks, seg);
}

int lf_launch_da(const void* X, const uint8_t* mask, int mask_bits, const void* dS, void* ws, size_t ws_bytes, size_t limit, int M, int K, int R,
                 const LfSegTable& seg, int dtype, hipStream_t st) {
  if (!X || !dS || M <= 0 || K <= 0) return LF_EINVAL;
  if (K % 128 != 0 || R % 16 != 0 || R <= 0 || R > LF_MAX_RANK) return LF_ESHAPE;
  if (seg.table && seg.block_size_m != ROWS) return LF_ESHAPE;
  const int nseg = seg.table ? seg.n_seg : 1;
  for (int s = 0; s < nseg; s++) if (!seg.out[s] || seg.rank[s] % 8 != 0 || seg.rank[s] > R) return LF_EINVAL;
  for (int s = 0; s < nseg; s++) if (((uintptr_t)seg.out[s] & 7) != 0) return LF_ESHAPE;  // 8-byte stores of dA
  if (!ws || ws_bytes < lf_da_workspace(M, K, R, seg, limit)) return LF_EWORKSPACE;
  if (mask != nullptr && mask_bits && ((uintptr_t)mask & 3) != 0) return LF_ESHAPE;   // 4-byte loads of the keep bits
  if (dtype == LF_BF16) return da_impl<__bf16>(X, mask, mask_bits, dS, ws, limit, M, K, R, seg, st);
  if (dtype == LF_F16) return da_impl<_Float16>(X, mask, mask_bits, dS, ws, limit, M, K, R, seg, st);
  return LF_EINVAL;
}


// ---- the rank-r part of a short backward in two or three launches: dS on its own (complete, lora_stream.hip), then dA and dB side by side as sums over rows
// (lora_da_direct.hip), where dys_dyb and da take three to five.  dY is read twice; what goes is the fp32 partials of dS and dB, their second stage and the walk of
// da behind that of dys_dyb.  Behind where one workgroup walks many blocks (a tile costs it 0.4 us, with a mask 0.9).
// Both sides in microseconds on one scale (ring_us); the short side fitted to the same batches, 7 % off on those that were not.  On these the choice takes 0.914 of the two passes' time (the
// faster form of dA among them) and 0.7 % more than the best of every form; 5.7 % are more than 3 % slower than the two passes (worst 1.3 times), most of them for a launch less.  With keep bits, replayed from a graph, two
// passes -> short: 300 x 4096 x 4096 rank 16 16.3 -> 12.8, four segments of 1280 rows rank 64 26.7 -> 24.1; the line: 1000 x 4096 x 4096 rank 16 20.7 either way; the other side of it: 1500 rows
// 23.8 against 25.7, 2048 28.0 against 31.0 (without a mask 22.0 against 22.5), 3000 x 5120 x 5120 rank 128 60 against 88.
size_t lf_ds_workspace(int M, int N, int R, const LfSegTable& seg);   // (lora_stream.hip)
int lf_launch_ds(const void* dY, void* dS, void* ws, int M, int N, int R, const LfSegTable& seg, int dtype, hipStream_t st);

struct ShortGrads { int a, b; };   // slices of K and of N; 0: not this way
static ShortGrads short_grads(int M, int N, int K, int R, bool masked, const LfSegTable& seg) {
  const int rt = rt_of(R), TA = K / 64, TB = N / 64;
  if (TA < 2 || TB < 2) return {0, 0};
  int blocks[LF_MAX_SEG], nseg, live = 0, big = 0;
  seg_block_counts(M, seg, blocks, nseg);
  for (int s = 0; s < nseg; s++) live += blocks[s] > 0, big = std::max(big, blocks[s]);
  if (live == 0 || big > 64) return {0, 0};
  int t = rt == 8 ? 2 : 1;   // (as in da_form)
  auto slices = [](int T, int t) { return (T + t - 1) / t; };
  while (t <= da_tpw(rt) && (slices(TA, t) + slices(TB, t)) * live > 256) t++;   // one round of workgroups
  if (t > da_tpw(rt)) return {0, 0};
  const ShortGrads g{slices(TA, t), slices(TB, t)};
  const int64_t rows = seg.table ? (int64_t)seg.n_blocks * ROWS : M;
  const double m = masked, tiles = (double)big * t, n = N / 4096.0, full = (g.a + g.b) * live / 256.0;
  double us = 5.34 + 0.806 * rt + tiles * (0.368 + 0.517 * m) + 0.443 * big + 1.49 * t * full;
  if (R <= 32) {
    const double groups = (double)((rows + 15) / 16) / 256;
    us += n * (0.29 + 1.73 * rt + 2.47 * std::min(groups, 1.0) + 10.7 * std::max(groups - 1.0, 0.0));
  } else {
    const int sl = lf_xa_stream_slices(M, N, R, false, seg);
    const double share = (double)(((rows + 63) / 64 * sl + 255) / 256) / sl;
    us += 0.665 + n * share * 5.21 * rt + (sl > 1 ? 4e-6 * sl * (double)rows * R : 0.0);
  }
  // (one segment above rank 64: the two passes' models are 6 % high)
  const double old = (dysr_plan(M, N, R, seg, SIZE_MAX).us + da_form(M, K, R, masked, seg, SIZE_MAX).us) * (seg.table == nullptr && rt == 8 ? 0.94 : 1.0);
  // One to three launches less, whose host side is 3 us each: it counts where forward and backward take less time than the host to issue them, 130 us, and for packed batches, where the host does more.
  // 1596 rows of five adapters x 6656 x 1408 at rank 16: 25.8 us either way, the whole call 132 - 144 and 149 - 153.  (Without these the choice is 0.7 % over the best of every form.)
  const double launches = (double)M * N * K < 2.5e10 ? (seg.table != nullptr ? 3.5 : 1.5) : 0.5;
  // (longer segments gain 1 - 2 % and are as often behind; where the workgroups take almost all compute units the model is 11 % off and not 5)
  return us * (big > 8 ? 1.03 : 1.0) * (full > 0.9 ? 1.05 : 1.0) < old + launches ? g : ShortGrads{0, 0};
}
size_t lf_short_grads_workspace(int M, int N, int K, int R, const LfSegTable& seg) {
  for (const bool masked : {false, true})
    if (short_grads(M, N, K, R, masked, seg).a > 0) return lf_ds_workspace(M, N, R, seg);
  return 0;
}
// sb: B_i in ptr; sg: dB_i in ptr, dA_i in out.  The launcher's preconditions are the two passes' own (lf_launch_dys_dyb, lf_launch_da): where
// one is missing, they run and say so.  (Operands at any element's address, as there.)
bool lf_short_grads_apply(const void* dY, const void* X, const uint8_t* mask, int mask_bits, const void* S, const void* dS, const void* ws, size_t ws_bytes, size_t limit, int M,
                          int N, int K, int R, const LfSegTable& sb, const LfSegTable& sg) {
  if (!dY || !X || !S || !dS || !ws || M <= 0 || N <= 0 || K <= 0 || N % 128 != 0 || K % 128 != 0 || R % 16 != 0 || R <= 0 || R > LF_MAX_RANK) return false;
  if (sb.table && sb.block_size_m != ROWS) return false;
  uintptr_t at8 = (uintptr_t)dS;
  for (int s = 0; s < (sb.table ? sb.n_seg : 1); s++) {
    if (!sb.ptr[s] || !sg.ptr[s] || !sg.out[s] || sb.rank[s] % 8 != 0 || sb.rank[s] > R) return false;
    at8 |= (uintptr_t)sg.ptr[s] | (uintptr_t)sg.out[s];
  }
  if ((at8 & 7) != 0 || (mask != nullptr && mask_bits && ((uintptr_t)mask & 3) != 0)) return false;
  // Outputs over inputs stay with the two passes: those write dS (caller's scratch: it may lie over S) and dB once dY, S and B_i have been read, and two-stage dA
  // once X, the mask and dS have.
  struct Span { uintptr_t at, bytes; };
  const auto span = [](const void* p, int64_t bytes) { return Span{(uintptr_t)p, p != nullptr ? (uintptr_t)bytes : 0}; };
  const Span in[] = {span(dY, (int64_t)M * N * 2), span(S, (int64_t)M * R * 2), span(X, (int64_t)M * K * 2), span(mask, mask_bits ? (int64_t)M * K / 8 : (int64_t)M * K)};
  const Span ds = span(dS, (int64_t)M * R * 2);
  const auto meet = [](const Span& a, const Span& b) { return a.at < b.at + b.bytes && b.at < a.at + a.bytes; };
  for (const Span& i : in) if (meet(ds, i)) return false;
  for (int s = 0; s < (sb.table ? sb.n_seg : 1); s++) {
    const Span b = span(sb.ptr[s], (int64_t)N * sb.rank[s] * 2), db = span(sg.ptr[s], (int64_t)N * sb.rank[s] * 2), da = span(sg.out[s], (int64_t)K * sb.rank[s] * 2);
    if (meet(ds, b) || meet(ds, db) || meet(ds, da)) return false;
    for (const Span& i : in) if (meet(db, i) || meet(da, i)) return false;
  }
  if (short_grads(M, N, K, R, mask != nullptr, sb).a == 0) return false;
  return ws_bytes >= std::max(lf_ds_workspace(M, N, R, sb), std::max(lf_dys_dyb_workspace(M, N, R, sb, limit), lf_da_workspace(M, K, R, sb, limit)));
}
int lf_launch_short_grads(const void* dY, const void* X, const uint8_t* mask, int mask_bits, const void* S, void* dS, void* ws, int M, int N, int K, int R,
                          const LfSegTable& sb, const LfSegTable& sg, int dtype, hipStream_t st) {
  const int rc = lf_launch_ds(dY, dS, ws, M, N, R, sb, dtype, st);
  if (rc != LF_OK) return rc;
  const ShortGrads g = short_grads(M, N, K, R, mask != nullptr, sb);
  const int fmt = mask == nullptr ? 0 : mask_bits ? 2 : mask_off_grid(mask, 0) ? 3 : 1;
  return lf_launch_da_direct(X, mask, fmt, dS, M, K, R, g.a, sg, dY, S, N, g.b, dtype, st);
}
