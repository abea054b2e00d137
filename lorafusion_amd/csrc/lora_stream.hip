// Products of a long streamed operand with a matrix of few rows, split along the contraction, for gfx950.
//
//   D[row][c] = sum_k keep(row, k) * P[row][k] * Q[c][k]       P: many rows, read once; Q: at most 128 rows
//
// Three uses:
//   xa      : P = X, Q = A_i:             S = drop(X) A^T     (seeded_dropout + `masked_scaled_x @ lora_a.T`,
//             lorafusion/ops/lora_v1.py:111-119; the multi-adapter product, multi_lora.py:481-513)
//   forward : P = the rows of W followed by the rows of A, Q = X of at most 128 rows: one pass over the weight gives the
//             base product and the rank-r product of a short batch; a second kernel adds the slices and forms
//             Y = X W^T + scale (X A^T) B^T + bias (fused_lora_xw_sb, triton_ops/fused_lora_xw_sb.py:74-206);
//             up to 16 rows and rank 32 a kernel of its own does all of it in one launch (short16_fwd_kernel)
//   dS      : P = dY, Q = B_i transposed: dS = scale dY B_i, where dB comes with dA (lora_da_direct.hip)
//
// All are bound by the stream of P (the forward of 8 rows moves 34 MB of weights for 0.3 GFLOP), so what counts is how
// many bytes the chip has on order.  A workgroup (4 waves) owns 64 rows of P and a slice of K: the slices are what
// gives every compute unit two workgroups when P has few rows, or when Q is so tall that a workgroup which walks all of K
// (lora_xa_kernel) would read it once per 16 rows of P.  P (64 rows x 64 columns, 8 KB), Q (up to 16 KB) and the keep
// bits of a step arrive by direct-to-LDS loads in a ring of NS stages; a wave reads the rows it loaded itself, the keep
// bits are applied to the fragment in registers (every element of P belongs to exactly one lane), so the only thing the
// waves share is Q and the one barrier of a step.
#include "lf_common.h"
#include "act_math.h"
#include "rank_common.h"
#include "rank_ring.h"

namespace {

constexpr int SROWS = 64;                                              // rows of P per workgroup, 16 per wave
constexpr int st_q_bytes(int rt) { return rt == 1 ? 4096 : rt * 2048; }   // rank 16: four rows per wave, padded to a load's 1 KB
constexpr int st_bytes(int rt, int mode) { return SROWS * 128 + st_q_bytes(rt) + (mode == 2 ? 1024 : mode == 1 ? 4096 : 0); }
constexpr int st_ns(int rt, int mode) { return mode == 1 ? (rt <= 2 ? 5 : rt == 4 ? 4 : 2) : (rt <= 2 ? 6 : rt == 4 ? 4 : 3); }   // stages: two workgroups per CU
constexpr int st_smem(int rt, int mode) { return st_ns(rt, mode) * st_bytes(rt, mode) + (mode == 3 ? 4096 : 0); }

struct StreamArgs {
  const void* p0;        // rows [0, n0) of P
  const void* p1;        // rows [n0, n0 + n1) (forward: the adapter's rows), or nullptr
  int n0, n1, K, n_slices;
  int folded;            // (rank tilings of 128 columns) no memory for the slices' sums: one workgroup walks all slices and adds their sums in the order the second stage would
  const uint8_t* mask;   // keep-mask read: bits [rows, K / 8] (MODE 2) or bytes [rows, K] (MODE 1)
  uint8_t* mask_out;     //           or drawn and written (MODE 3), as bits or as bytes
  int mask_bytes;
  uint32_t seed_lo, seed_hi;
  float* part;           // xa: [slice][row][R]; forward: [slice][m][pitch]; nullptr (xa, one slice or folded): S is written directly
  int64_t pitch;
  void* S;
  int M, R;              // xa: rows given, columns of S.  forward: M = rows of Q
  const void* q;         // forward: X [M, K]
};

// grid (64-row groups of P, slices of K).  MODE: 0 no keep-mask, 1 keep bytes read, 2 keep bits read, 3 mask drawn and written, 4 bytes or bits
// read from an address that the direct loads do not take (the compiler's waits for these loads empty the ring every step).
// FWD: Q = X (the second use above), D is stored transposed, [m][row of P].  QT: Q lies transposed in memory, [K, rank] (the third: P = dY, Q = B_i).
template <typename T, int RT, int MODE, bool FWD, bool QT>
__global__ void __launch_bounds__(256, 2)
lora_stream_kernel(const StreamArgs a, const LfSegTable seg) {
  constexpr int NS = st_ns(RT, MODE), STAGE = st_bytes(RT, MODE), QB = st_q_bytes(RT);
  constexpr int NQ = RT == 1 ? 1 : RT / 2;              // loads of Q per wave and step
  constexpr int G = 2 + NQ + (MODE == 1 || MODE == 2 ? 1 : 0);       // loads per wave and step
  constexpr bool FOLDS = RT == 8 && !FWD;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  const int tid = threadIdx.x, lane = tid & 63, wave = to_sgpr(tid >> 6);
  const int li = lane & 15, qq = lane >> 4;
  const int grp = blockIdx.x, sl = blockIdx.y, K = a.K;
  // this slice (or all of them): whole pairs of steps (128 columns), balanced
  const int np = K / 128;
  auto slice_begin = [&](int i) { return (int)((int64_t)np * i / a.n_slices); };
  const int k_lo = a.folded ? 0 : slice_begin(sl), k_hi = a.folded ? np : slice_begin(sl + 1);
  const int nsteps = 2 * (k_hi - k_lo);

  int row0 = grp * SROWS, rows_all = a.n0;   // within p0 or p1
  const char* pb = (const char*)a.p0;
  const char* qb = (const char*)a.q;
  int q_rows = a.M;
  BlockInfo bi{};
  if constexpr (FWD) {
    if (row0 >= a.n0) { row0 -= a.n0; rows_all = a.n1; pb = (const char*)a.p1; }
  } else {
    bi = block_info(seg, row0 / ROWS, a.M);
    qb = (const char*)seg.ptr[bi.seg];
    q_rows = bi.rank;
  }
  const bool use_mask = MODE > 0 && bi.p > 0.f;   // (rows of a block without dropout keep everything)
  const uint32_t thr = lf_keep_threshold(bi.p);

  // loader: 8 lanes cover the 128 bytes of a row; granule g of row r goes to slot g ^ ((r >> 1) & 7)
  const int lrow = lane >> 3, slot = lane & 7;
  uint32_t pv[2], qv[NQ], mv = 0;
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int r = i * 8 + lrow;
    pv[i] = (uint32_t)(((int64_t)(wave * 16 + r) * K) * 2 + ((slot ^ ((r >> 1) & 7)) << 4));
  }
#pragma unroll
  for (int i = 0; i < NQ; i++) {
    // rank 16: a wave fetches four rows (lanes 0..31), else eight rows per load
    const int r = RT == 1 ? wave * 4 + (lrow & 3) : (wave * NQ + i) * 8 + lrow;
    qv[i] = (uint32_t)(((int64_t)r * K) * 2 + ((slot ^ ((r >> 1) & 7)) << 4));
    if (RT == 1 && lane >= 32) qv[i] = 0xffffff00u;   // beyond the window: nothing is fetched
  }
  if constexpr (QT) side_voffs<RT, NQ>(qv, q_rows, q_rows, tid);
  if constexpr (MODE == 1) mv = (uint32_t)((wave * 16 + (lane >> 2)) * (int64_t)K + (lane & 3) * 16);
  if constexpr (MODE == 2) mv = lane < 32 ? (uint32_t)((wave * 16 + (lane >> 1)) * (K >> 3) + (lane & 1) * 4) : 0xffffff00u;

  const int64_t k0 = (int64_t)k_lo * 128;
  pb += ((int64_t)row0 * K + k0) * 2;
  int64_t pleft = ((int64_t)(rows_all - row0) * K - k0) * 2;
  qb += k0 * 2 * (QT ? q_rows : 1);
  int64_t qleft = QT ? (K - k0) * q_rows * 2 : ((int64_t)q_rows * K - k0) * 2;
  const int qstep = QT ? 128 * q_rows : 128;
  const char* mb = (const char*)a.mask + (((int64_t)row0 * K + k0) >> (MODE == 2 ? 3 : 0));
  int64_t mleft = ((int64_t)(rows_all - row0) * K - k0) >> (MODE == 2 ? 3 : 0);
  int ord = 0, ist = 0;   // steps ordered so far (behind the last one: that one again, unconsumed), stage of the next
  auto issue = [&]() {
    const uint32_t st = lds0 + ist * STAGE;
    const lf_u32x4 rp = window_rsrc(pb, pleft), rq = window_rsrc(qb, qleft);
#pragma unroll
    for (int i = 0; i < 2; i++) dma16(rp, pv[i], st + wave * 2048 + i * 1024);
#pragma unroll
    for (int i = 0; i < NQ; i++) dma16(rq, qv[i], st + SROWS * 128 + (QT ? i * 4096 + wave * 1024 : (wave * NQ + i) * 1024));
    if constexpr (MODE == 1) dma16(window_rsrc(mb, mleft), mv, st + SROWS * 128 + QB + wave * 1024);
    if constexpr (MODE == 2) dma4(window_rsrc(mb, mleft), mv, st + SROWS * 128 + QB + wave * 256);
    ist = ist + 1 == NS ? 0 : ist + 1;
    if (++ord < nsteps) {
      pb += 128, pleft -= 128, qb += qstep, qleft -= qstep;
      if constexpr (MODE == 1) mb += 64, mleft -= 64;
      if constexpr (MODE == 2) mb += 8, mleft -= 8;
    }
  };
#pragma unroll 1
  for (int i = 0; i < NS - 1; i++) issue();

  lf_f32x4 acc[RT], sum[RT];
#pragma unroll
  for (int c = 0; c < RT; c++) acc[c] = sum[c] = lf_f32x4{0.f, 0.f, 0.f, 0.f};
  int fold_at = 2 * slice_begin(1), fold_next = 2;   // folded: first step of the next slice
  const int key = (li >> 1) & 7;
  char* bits_buf = lds + NS * STAGE + wave * 1024;   // MODE 3: 16 rows x 64 bytes = eight steps of this wave's keep bits
  const int64_t my_row = row0 + wave * 16 + li;
  const uint64_t ctr0 = (uint64_t)(my_row * K + k0) >> 3;

  int cst = 0;
  for (int s = 0; s < nsteps; s++) {
    wait_groups<G>(NS - 2);
    ring_barrier();   // this step's stage has landed for every wave; everyone is done with the stage refilled next
    issue();
    if (FOLDS && a.folded && s == fold_at) {
#pragma unroll
      for (int c = 0; c < RT; c++) sum[c] += acc[c], acc[c] = lf_f32x4{0.f, 0.f, 0.f, 0.f};
      fold_at = 2 * slice_begin(fold_next++);
    }
    const char* x = lds + cst * STAGE + wave * 2048;
    const char* q = lds + cst * STAGE + SROWS * 128;
    lf_u32x4 xf[2], qf[2][RT];
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int fo = ((h * 4 + qq) ^ key) << 4;
      xf[h] = *(const lf_u32x4*)(x + li * 128 + fo);
#pragma unroll
      for (int c = 0; c < RT; c++)
        if constexpr (QT) qf[h][c] = side_tr8<RT>(q, h * 32 + qq * 8 + (li >> 2), c, li & 3);
        else qf[h][c] = *(const lf_u32x4*)(RT == 1 ? q + (li >> 2) * 1024 + (li & 3) * 128 + fo : q + (c * 16 + li) * 128 + fo);
    }
    if constexpr (MODE == 1) {
      if (use_mask) {
        const char* mt = lds + cst * STAGE + SROWS * 128 + QB + wave * 1024;
#pragma unroll
        for (int h = 0; h < 2; h++) xf[h] = apply_mask8(xf[h], *(const lf_u32x2*)(mt + li * 64 + (h * 4 + qq) * 8));
      }
    }
    if constexpr (MODE == 2) {
      if (use_mask) {
        const char* mt = lds + cst * STAGE + SROWS * 128 + QB + wave * 256;
#pragma unroll
        for (int h = 0; h < 2; h++) xf[h] &= select8(*(const uint8_t*)(mt + li * 8 + h * 4 + qq));
      }
    }
    if constexpr (MODE == 4) {
      if (use_mask && my_row < rows_all) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const uint64_t el = (uint64_t)(my_row * K + k0) + (uint64_t)(s * 64 + (h * 4 + qq) * 8);
          if (a.mask_bytes) xf[h] = apply_mask8(xf[h], keep_bytes8(a.mask + el));
          else xf[h] &= select8(a.mask[el >> 3]);
        }
      }
    }
    if constexpr (MODE == 3) {
#pragma unroll
      for (int h = 0; h < 2; h++) {
        uint32_t bits = 0xffu;
        if (use_mask && thr > 0) xf[h] &= draw8(ctr0 + (uint64_t)(s * 8 + h * 4 + qq), thr, a.seed_lo, a.seed_hi, bits);
        bits_buf[li * 64 + (s & 7) * 8 + h * 4 + qq] = (char)bits;
        if (a.mask_bytes && my_row < rows_all) *(lf_u32x2*)(a.mask_out + my_row * K + k0 + s * 64 + (h * 4 + qq) * 8) = expand_keep8(bits);
      }
      if (!a.mask_bytes && ((s & 7) == 7 || s + 1 == nsteps)) {
        // (same-wave LDS traffic is ordered.)  Lane l: row l>>2, 16-byte piece l&3 = two steps
        const int r = lane >> 2, pc = lane & 3, first = s & ~7;
        const lf_u32x4 v = *(const lf_u32x4*)(bits_buf + r * 64 + pc * 16);
        const int64_t gr = row0 + wave * 16 + r;
        if (gr < rows_all && first + 2 * pc <= s) __builtin_nontemporal_store(v, (lf_u32x4*)(a.mask_out + ((gr * K + k0) >> 3) + first * 8 + pc * 16));
      }
    }
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int c = 0; c < RT; c++)
        acc[c] = FWD ? Mfma16<T>::run(qf[h][c], xf[h], acc[c]) : Mfma16<T>::run(xf[h], qf[h][c], acc[c]);
    cst = cst + 1 == NS ? 0 : cst + 1;
  }
  wait_vm<0>();   // the unconsumed loads behind the last step must not land in another workgroup's LDS
  if constexpr (FWD) {
    // lane: row li of P, rows 4 qq + e of Q
    if (row0 + wave * 16 + li < rows_all) {
      float* po = a.part + (int64_t)sl * a.M * a.pitch + grp * SROWS + wave * 16 + li;
#pragma unroll
      for (int c = 0; c < RT; c++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int m = c * 16 + qq * 4 + e;
          if (m < a.M) po[(int64_t)m * a.pitch] = acc[c][e];
        }
    }
  } else {
    // lane: column li of each 16, rows 4 qq + e of the wave
    const float mult = QT ? bi.scale : use_mask ? 1.f / (1.f - bi.p) : 1.f;
    if constexpr (FOLDS) {
#pragma unroll
      for (int c = 0; c < RT; c++) acc[c] = sum[c] + acc[c];
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int64_t row = row0 + wave * 16 + qq * 4 + e;
      if (row < rows_all) {
        const bool real = (int)(row & (ROWS - 1)) < bi.valid;
#pragma unroll
        for (int c = 0; c < RT; c++) {
          const int col = c * 16 + li;
          if (c * 16 < a.R) {
            if (a.part != nullptr) a.part[((int64_t)sl * rows_all + row) * a.R + col] = acc[c][e];
            else ((uint16_t*)a.S)[row * a.R + col] = real && col < bi.rank ? Mfma16<T>::cvt(fp32_product(acc[c][e], mult)) : (uint16_t)0;
          }
        }
      }
    }
  }
}

// Second stage of a sliced xa: S = cast(1/(1-p) * sum of the slices), zero in padded rows and beyond the rank.  (mult: 0 none, 1 1/(1-p), 2 the scale: dS)
template <typename T>
__global__ void __launch_bounds__(256)
stream_reduce_kernel(const float* __restrict__ part, T* __restrict__ S, int n_slices, int M, int R, int mult, const LfSegTable seg) {
  const int64_t rows = seg.table ? (int64_t)seg.n_blocks * ROWS : M;
  const int64_t idx = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (idx >= rows * R) return;
  const int row = (int)(idx / R), col = (int)(idx % R);
  const BlockInfo bi = block_info(seg, row / ROWS, M);
  lf_f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if (row % ROWS < bi.valid && col < bi.rank) {
    v = sum_parts(part + idx, rows * R, n_slices);
    if (mult == 1 && bi.p > 0.f) v *= 1.f / (1.f - bi.p);
    if (mult == 2) v *= bi.scale;
  }
  *(lf_u32x2*)((uint16_t*)S + idx) = pack4<T>(v);
}

// Rank-r product without a keep-mask at ranks up to 32, where the rows are few (lf_xa_rings).  A workgroup of eight waves per 16 rows of X over all of K, as
// lora_xa_kernel has it, but X and A arrive by direct loads: a wave streams its steps of both (every eighth 64 columns)
// through a ring of its own, without a barrier, and keeps NS - 1 steps on order instead of the one or two that registers hold.  Nothing needs to come
// through registers here: there is no mask to apply before the product.
// Bound by what one compute unit takes in, X and A (MI355X, replayed from a graph, rank 16: 333 x 4096 5.2 -> 4.5 us, 1000 x 4096 6.6 -> 5.3,
// 4096 x 4096 9.2 -> 8.3, 4.1 TB/s of X; whole forwards of 333 x 4096 into 4096 27.1 -> 26.1, 3000 x 8192 into 2048 at rank 32 99.6 -> 96.8).
constexpr int xr_stages(int rt) { return rt == 1 ? 4 : 3; }
// QT: A lies transposed in memory, [K, rank], and the product is scaled: dS = scale dY B_i.
template <typename T, int RT, bool QT>
__global__ void __launch_bounds__(512)
lora_xa_ring_kernel(const void* __restrict__ X, T* __restrict__ S, int M, int rows, int K, int R, const LfSegTable seg) {
  constexpr int NS = xr_stages(RT), STAGE = (1 + RT) * 2048, GL = 2 * (1 + RT);
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = to_sgpr(tid >> 6);
  const int li = lane & 15, qq = lane >> 4;
  const int row0 = blockIdx.x * 16;
  const BlockInfo bi = block_info(seg, row0 / ROWS, M);
  const char* A = (const char*)seg.ptr[bi.seg];
  const int nsteps = (K / 64 - wave + 7) / 8;   // steps wave, wave + 8, ...

  char* ring = lds + wave * NS * STAGE;
  const uint32_t ring0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)ring;
  // 8 lanes cover the 128 bytes of a row; granule c of row r at slot c ^ ((r >> 1) & 7)
  const int lrow = lane >> 3, slot = lane & 7;
  uint32_t rv[2 * RT];
#pragma unroll
  for (int i = 0; i < 2 * RT; i++) {
    const int r = i * 8 + lrow;
    rv[i] = (uint32_t)((int64_t)r * K * 2 + ((slot ^ ((r >> 1) & 7)) << 4));
  }
  uint32_t tv[2 * RT];   // QT: 64 rows of B_i
#pragma unroll
  for (int i = 0; i < 2 * RT; i++) {
    const int p = i * 64 + lane, row = side_row<RT>(p / (RT * 2)), g = (p % (RT * 2)) ^ side_key<RT>(row);
    tv[i] = (uint32_t)(row * bi.rank * 2 + (g * 8 < bi.rank ? g : 0) * 16);   // (beyond the rank: columns that are not stored)
  }
  auto issue = [&](int i) {
    const int at = i < nsteps ? i : nsteps - 1;   // (behind the last step: that one again, unconsumed)
    const int64_t ko = (int64_t)(wave + at * 8) * 128;
    const uint32_t st = ring0 + (i % NS) * STAGE;
    const lf_u32x4 rx = window_rsrc((const char*)X + (int64_t)row0 * K * 2 + ko, (int64_t)(rows - row0) * K * 2 - ko);   // (rows beyond the last and
    const int64_t qo = QT ? (int64_t)(wave + at * 8) * 128 * bi.rank : ko;                                               // beyond the rank read as zeros)
    const lf_u32x4 ra = window_rsrc(A + qo, (int64_t)bi.rank * K * 2 - qo);
#pragma unroll
    for (int q = 0; q < 2; q++) dma16(rx, rv[q], st + q * 1024);
#pragma unroll
    for (int q = 0; q < 2 * RT; q++) dma16(ra, QT ? tv[q] : rv[q], st + 2048 + q * 1024);
  };
  lf_f32x4 acc[RT];
#pragma unroll
  for (int c = 0; c < RT; c++) acc[c] = lf_f32x4{0.f, 0.f, 0.f, 0.f};
  const int key = (li >> 1) & 7;
  if (nsteps > 0) {
    for (int i = 0; i < NS - 1; i++) issue(i);
    for (int i = 0; i < nsteps; i++) {
      wait_groups<GL>(NS - 2);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // this wave has read the stage that is refilled now
      issue(i + NS - 1);
      const char* st = ring + (i % NS) * STAGE;
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const char* fr = st + li * 128 + (((h * 4 + qq) ^ key) << 4);
        const lf_u32x4 xf = *(const lf_u32x4*)fr;
#pragma unroll
        for (int c = 0; c < RT; c++)
          acc[c] = Mfma16<T>::run(xf, QT ? side_tr8<RT>(st + 2048, h * 32 + qq * 8 + (li >> 2), c, li & 3) : *(const lf_u32x4*)(fr + (1 + c) * 2048), acc[c]);
      }
    }
    wait_vm<0>();   // the unconsumed loads behind the last step
  }
  __syncthreads();
  float* part = (float*)lds;   // [8 waves][16 RT columns][16 rows]
#pragma unroll
  for (int c = 0; c < RT; c++) *(lf_f32x4*)(part + ((wave * RT + c) * 16 + li) * 16 + qq * 4) = acc[c];
  __syncthreads();
  const int col = tid >> 4, m = tid & 15;
  if (col < R && row0 + m < rows) {
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < 8; w++) v += part[w * RT * 256 + (col % (16 * RT)) * 16 + m];
    const bool real = (row0 + m) % ROWS < bi.valid && col < bi.rank;
    if constexpr (QT) v = fp32_product(v, bi.scale);
    S[(int64_t)(row0 + m) * R + col] = real ? (T)v : (T)0.f;
  }
}

// Forward of up to 16 rows at ranks up to 32 in one launch.  A workgroup owns 16 G rows of W over all of K; its NW waves deal the steps of 64
// among themselves, and each streams its steps of W, of X (16 rows) and of A through a ring of its own, so the walk has no barrier.  Every
// workgroup forms all of S for itself; the first stores it.  The waves' sums are added in a fixed order through LDS, S is rounded,
// and the workgroup's 16 G columns of Y leave complete: no partial sums in memory, no second launch.  What that costs is X and A once per
// workgroup, from L2 -- as many bytes each as W at G = 1 and rank 16.  That is why the form ends at 16 rows and rank 32, and why G is 4 (with four
// waves: the same LDS) where there are columns for it: G = 4 over G = 1 at 8192 columns 13.4 against 16.0 us, at 4096, with 64 workgroups,
// 11.1 against 9.0.  G = 2 was never ahead of both.
// Bound by the launch, the first loads and W's bytes: 6 x 4096 x 4096 at rank 16 (MI355X, W from the memory-side cache, captured back to back)
// 12.8 -> 9.0 us, 3.7 TB/s of W; 6 x 1024 x 1024 7.1 -> 3.9; 6 x 14336 x 4096 (W from HBM, 4.6 TB/s) 34.2 -> 25.6.
constexpr int short16_waves(int g) { return g == 1 ? 8 : 4; }
constexpr int short16_stages(int rt, int g) { return 160 / (short16_waves(g) * 2 * (g + 1 + rt)); }   // what 160 KiB hold: 3, 2 (G = 1, ranks to 16, 32), 3, 2
template <typename T, int RT, int G, int NW = short16_waves(G)>
__global__ void __launch_bounds__(NW * 64)
short16_fwd_kernel(const void* __restrict__ X, const void* __restrict__ W, const void* __restrict__ A, const T* __restrict__ B, float scale,
                   const uint16_t* __restrict__ bias, T* __restrict__ Y, T* __restrict__ S, int M, int N, int K, int rank, int R) {
  constexpr int NS = short16_stages(RT, G), STAGE = (G + 1 + RT) * 2048, GL = 2 * (G + 1 + RT), NT = NW * 64, COLS = 16 * G;
  static_assert(NS >= 2 && (NS - 2) * GL < 64, "");
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = to_sgpr(tid >> 6);
  const int li = lane & 15, qq = lane >> 4;
  const int col0 = blockIdx.x * COLS;
  const int nsteps = (K / 64 - wave + NW - 1) / NW;   // steps wave, wave + NW, ...
  // the row of B that this thread multiplies at the end: requested first
  const int n = tid % COLS;
  lf_u32x4 bv[RT * 2];
#pragma unroll
  for (int q = 0; q < RT * 2; q++) bv[q] = q * 8 < rank ? *(const lf_u32x4*)(B + (int64_t)(col0 + n) * rank + q * 8) : lf_u32x4{0, 0, 0, 0};

  char* ring = lds + wave * NS * STAGE;
  const uint32_t ring0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)ring;
  // 8 lanes cover the 128 bytes of a row; granule c of row r at slot c ^ ((r >> 1) & 7)
  const int lrow = lane >> 3, slot = lane & 7;
  constexpr int NV = 2 * (G > RT ? G : RT);
  uint32_t rv[NV];
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const int r = i * 8 + lrow;
    rv[i] = (uint32_t)((int64_t)r * K * 2 + ((slot ^ ((r >> 1) & 7)) << 4));
  }
  auto issue = [&](int i) {
    const int at = i < nsteps ? i : nsteps - 1;   // (behind the last step: that one again, unconsumed)
    const int64_t ko = (int64_t)(wave + at * NW) * 128;
    const uint32_t st = ring0 + (i % NS) * STAGE;
    const lf_u32x4 rw = window_rsrc((const char*)W + (int64_t)col0 * K * 2 + ko, (int64_t)COLS * K * 2 - ko);
    const lf_u32x4 rx = window_rsrc((const char*)X + ko, (int64_t)M * K * 2 - ko);   // (rows beyond M and beyond the rank read as zeros)
    const lf_u32x4 ra = window_rsrc((const char*)A + ko, (int64_t)rank * K * 2 - ko);
#pragma unroll
    for (int q = 0; q < 2 * G; q++) dma16(rw, rv[q], st + q * 1024);
#pragma unroll
    for (int q = 0; q < 2; q++) dma16(rx, rv[q], st + G * 2048 + q * 1024);
#pragma unroll
    for (int q = 0; q < 2 * RT; q++) dma16(ra, rv[q], st + (G + 1) * 2048 + q * 1024);
  };
  lf_f32x4 acc[G + RT];   // lane: column li of each group (of W's rows, then of A's), rows 4 qq + e of X
#pragma unroll
  for (int c = 0; c < G + RT; c++) acc[c] = lf_f32x4{0.f, 0.f, 0.f, 0.f};
  const int key = (li >> 1) & 7;
  if (nsteps > 0) {
    for (int i = 0; i < NS - 1; i++) issue(i);
    for (int i = 0; i < nsteps; i++) {
      wait_groups<GL>(NS - 2);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // this wave has read the stage that is refilled now
      issue(i + NS - 1);
      const char* st = ring + (i % NS) * STAGE;
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const char* fr = st + li * 128 + (((h * 4 + qq) ^ key) << 4);
        const lf_u32x4 xf = *(const lf_u32x4*)(fr + G * 2048);
#pragma unroll
        for (int c = 0; c < G + RT; c++) acc[c] = Mfma16<T>::run(xf, *(const lf_u32x4*)(fr + (c < G ? c : c + 1) * 2048), acc[c]);
      }
    }
    wait_vm<0>();   // the unconsumed loads behind the last step
  }
  __syncthreads();
  float* part = (float*)lds;                             // [NW][16 (G + RT) columns][16 rows]
  float* sv = part + NW * (G + RT) * 256;                // [16 RT][16 rows]: S, rounded
#pragma unroll
  for (int c = 0; c < G + RT; c++) *(lf_f32x4*)(part + ((wave * (G + RT) + c) * 16 + li) * 16 + qq * 4) = acc[c];
  __syncthreads();
  for (int o = tid; o < RT * 256; o += NT) {
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < NW; w++) v += part[(w * (G + RT) + G) * 256 + o];
    sv[o] = (float)(T)v;
  }
  __syncthreads();
  if (blockIdx.x == 0) {
    for (int o = tid; o < M * R; o += NT) {
      const int m = o / R, r = o % R;
      S[o] = r < rank ? (T)sv[r * 16 + m] : (T)0.f;
    }
  }
#pragma unroll
  for (int m = tid / COLS; m < 16; m += NT / COLS) {
    if (m >= M) break;
    float y = 0.f, t = 0.f;
#pragma unroll
    for (int p = 0; p < NW; p++) y += part[(p * (G + RT) * 16 + n) * 16 + m];
#pragma unroll
    for (int q = 0; q < RT * 2; q++) {
      if (q * 8 >= rank) break;   // (not zeros times zeros: S beyond the rank is the zeros of A times X, NaN where X has an infinity)
      float f[8];
      unpack8<T>(bv[q], f);
#pragma unroll
      for (int e = 0; e < 8; e++) t = __builtin_fmaf(f[e], sv[(q * 8 + e) * 16 + m], t);
    }
    y += t * scale;
    if (bias != nullptr) y += (float)__builtin_bit_cast(T, bias[col0 + n]);
    Y[(int64_t)m * N + col0 + n] = (T)y;
  }
}

// Second stage of the short forward.  grid (64-column tiles of Y, groups of 16 rows), 16 lanes per row.  A short launch is
// as long as its chain of memory round trips: the slices of Y and the rows of B are requested before the S rows that the
// workgroup needs are added up and rounded (each workgroup its own, r <= 128 columns, from L2; the first column tile
// stores them).
template <typename T>
__global__ void __launch_bounds__(256)
short_fwd_finish_kernel(const float* __restrict__ part, int64_t pitch, int n_slices, int M, int N, int rank, int R, const T* __restrict__ B,
                        float scale, const uint16_t* __restrict__ bias, T* __restrict__ Y, T* __restrict__ S) {
  __shared__ float sv[16][LF_MAX_RANK];
  const int tid = threadIdx.x, m0 = blockIdx.y * 16;
  const int mi = tid >> 4, m = m0 + mi, col = blockIdx.x * 64 + (tid & 15) * 4;   // (N % 128 == 0: no column beyond N)
  lf_f32x4 y = {0.f, 0.f, 0.f, 0.f};
  lf_u32x4 b0[4];
  if (m < M) {
    y = sum_parts(part + (int64_t)m * pitch + col, (int64_t)M * pitch, n_slices);
#pragma unroll
    for (int c = 0; c < 4; c++) b0[c] = *(const lf_u32x4*)(B + (int64_t)(col + c) * rank);
  }
  for (int o = tid; o < 4 * R; o += 256) {   // four columns of one row each
    const int r = o / (R / 4), j = o % (R / 4) * 4, sm = m0 + r;
    lf_f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (sm < M && j < rank) v = sum_parts(part + (int64_t)sm * pitch + N + j, (int64_t)M * pitch, n_slices);
    const lf_u32x2 h = pack4<T>(v);
#pragma unroll
    for (int e = 0; e < 4; e++) sv[r][j + e] = (float)(T)v[e];
    if (blockIdx.x == 0 && sm < M) *(lf_u32x2*)((uint16_t*)S + (int64_t)sm * R + j) = h;
  }
  __syncthreads();
  if (m >= M) return;
  lf_f32x4 t = {0.f, 0.f, 0.f, 0.f};
  for (int j = 0; j < rank; j += 8) {
    lf_u32x4 bn[4];
    if (j + 8 < rank) {
#pragma unroll
      for (int c = 0; c < 4; c++) bn[c] = *(const lf_u32x4*)(B + (int64_t)(col + c) * rank + j + 8);
    }
#pragma unroll
    for (int c = 0; c < 4; c++) {
      float f[8];
      unpack8<T>(b0[c], f);
#pragma unroll
      for (int e = 0; e < 8; e++) t[c] = __builtin_fmaf(f[e], sv[mi][j + e], t[c]);
      b0[c] = bn[c];
    }
  }
#pragma unroll
  for (int c = 0; c < 4; c++) {
    y[c] += t[c] * scale;
    if (bias != nullptr) y[c] += (float)__builtin_bit_cast(T, bias[col + c]);
  }
  *(lf_u32x2*)((uint16_t*)Y + (int64_t)m * N + col) = pack4<T>(y);
}

// Slices of K.  Compute units share the workgroups evenly or not at all: 65 groups in 4 slices are 260 workgroups, and four
// of the 256 compute units take twice as long as the rest.  So: the count (at most sixteen, none shorter than four
// steps) with the shortest modelled time -- the busiest compute unit's share of the walk (us per column of K: `walk`), the partial sums written and
// read back, and what a second stage costs where a single slice needs none.
// Forward: a full walk of K = 4096 takes 22 us; 6 x 4096 x 4096 (65 groups; now a single launch), first and second stage: 3 slices 12.0 us, 4: 13.3, 7: 12.5, 8: 14.0.
// xa: below K = 768 one; a walk of 4096 takes 18 - 24 us without a mask, 26 - 33 with one read and 48 - 53 with one drawn (the integer work of a workgroup that
// has a compute unit to itself); the constants are those with the smallest loss against the best count over 64 - 20000 rows, K of
// 1024 - 14336 and ranks 64 and 128 (masked 13 % -> 3.5 %, against one walk figure of 22 us for all; 9000 x 3072 at rank 64, mask drawn: one
// slice 41 us, three 27.5; 6000 x 1536 at rank 128: one 27, two 21).
struct SliceModel { double walk; bool single_is_direct; };   // single_is_direct: one slice writes no partial sums and needs no second stage (1.5 us)
constexpr SliceModel kFwdSlices = {0.0054, false}, kXaSlices = {0.008, true}, kXaMaskedSlices = {0.0105, true};
int slices_for(int64_t groups, int K, double partial_bytes, const SliceModel& m) {
  const int most = K / 256 < 1 || (m.single_is_direct && K < 768) ? 1 : K / 256 > 16 ? 16 : K / 256;
  int best = 1;
  double best_cost = 1e300;
  for (int n = 1; n <= most; n++) {
    const double share = (double)((groups * n + 255) / 256) / n;
    const double cost = share * K * m.walk + (n == 1 && m.single_is_direct ? 0.0 : n * partial_bytes / 1.5e6 + 1.5);
    if (cost < best_cost) { best_cost = cost; best = n; }
  }
  return best;
}

template <typename T, int RT, int MODE, bool FWD, bool QT = false>
int stream_launch(const StreamArgs& a, const LfSegTable& seg, int groups, hipStream_t st) {
  auto kern = lora_stream_kernel<T, RT, MODE, FWD, QT>;
  constexpr int SMEM = st_smem(RT, MODE);
  static_assert(2 * SMEM <= 160 * 1024, "two workgroups per CU");
  static LfLdsFlags lds_ok;
  if (!lf_allow_lds(kern, SMEM, lds_ok)) return LF_ELAUNCH;
  return lf_launch(kern, dim3(groups, a.folded ? 1 : a.n_slices), dim3(256), SMEM, st, a, seg);
}
template <typename T, int RT>
int stream_mode(const StreamArgs& a, const LfSegTable& seg, int groups, hipStream_t st) {
  if (a.q != nullptr) return stream_launch<T, RT, 0, true>(a, seg, groups, st);
  if (a.mask_out != nullptr) return stream_launch<T, RT, 3, false>(a, seg, groups, st);
  if (mask_off_grid(a.mask, !a.mask_bytes)) {
    if constexpr (RT == 8) return stream_launch<T, RT, 4, false>(a, seg, groups, st);
    else return LF_ESHAPE;   // (lf_xa_takes_stream)
  }
  if (a.mask != nullptr) return a.mask_bytes ? stream_launch<T, RT, 1, false>(a, seg, groups, st) : stream_launch<T, RT, 2, false>(a, seg, groups, st);
  return stream_launch<T, RT, 0, false>(a, seg, groups, st);
}
template <typename T>
int stream_rt(const StreamArgs& a, const LfSegTable& seg, int cols, int groups, hipStream_t st) {
  switch (rt_of(cols)) {
    case 1: return stream_mode<T, 1>(a, seg, groups, st);
    case 2: return stream_mode<T, 2>(a, seg, groups, st);
    case 4: return stream_mode<T, 4>(a, seg, groups, st);
    default: return stream_mode<T, 8>(a, seg, groups, st);
  }
}

template <typename T>
int xa_stream_impl(StreamArgs a, const LfSegTable& seg, float* ws, hipStream_t st) {
  const int groups = (a.n0 + SROWS - 1) / SROWS;
  a.folded = a.n_slices > 1 && ws == nullptr;
  a.part = a.n_slices > 1 ? ws : nullptr;
  int rc = stream_rt<T>(a, seg, a.R, groups, st);
  if (rc != LF_OK || a.part == nullptr) return rc;
  const int64_t n4 = ((int64_t)a.n0 * a.R + 3) / 4;
  return lf_launch((stream_reduce_kernel<T>), dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, st, (const float*)ws, (T*)a.S, a.n_slices, a.M,
                   a.R, (a.mask != nullptr || a.mask_out != nullptr) ? 1 : 0, seg);
}

}  // namespace

static int64_t xa_rows_of(int M, const LfSegTable& seg) { return seg.table ? (int64_t)seg.n_blocks * ROWS : M; }

int lf_xa_stream_slices(int M, int K, int R, bool masked, const LfSegTable& seg) {
  const int64_t groups = (xa_rows_of(M, seg) + SROWS - 1) / SROWS;
  const double slab = (double)xa_rows_of(M, seg) * R * sizeof(float);
  return slices_for(groups, K, slab, masked ? kXaMaskedSlices : kXaSlices);
}

size_t lf_xa_stream_workspace(int M, int K, int R, bool masked, const LfSegTable& seg) {
  const int n = lf_xa_stream_slices(M, K, R, masked, seg);
  return n > 1 ? (size_t)n * xa_rows_of(M, seg) * R * sizeof(float) : 0;
}

template <typename T, int RT, bool QT = false>
static int xa_ring_launch(const void* X, void* S, int M, int rows, int K, int R, const LfSegTable& seg, hipStream_t st) {
  auto kern = lora_xa_ring_kernel<T, RT, QT>;
  constexpr int SMEM = 8 * xr_stages(RT) * (1 + RT) * 2048;
  static LfLdsFlags lds_ok;
  if (!lf_allow_lds(kern, SMEM, lds_ok)) return LF_ELAUNCH;
  return lf_launch(kern, dim3((rows + 15) / 16), dim3(512), SMEM, st, X, (T*)S, M, rows, K, R, seg);
}
int lf_launch_xa_ring(const void* X, void* S, int M, int K, int R, const LfSegTable& seg, int dtype, hipStream_t st) {
  const int rows = (int)xa_rows_of(M, seg);
  if (dtype == LF_BF16) return R <= 16 ? xa_ring_launch<__bf16, 1>(X, S, M, rows, K, R, seg, st) : xa_ring_launch<__bf16, 2>(X, S, M, rows, K, R, seg, st);
  return R <= 16 ? xa_ring_launch<_Float16, 1>(X, S, M, rows, K, R, seg, st) : xa_ring_launch<_Float16, 2>(X, S, M, rows, K, R, seg, st);
}

// ws == nullptr: no room for the slices' sums (ranks above 64 or a single slice; the result is the same, bit for bit)
int lf_launch_xa_stream(const void* X, const uint8_t* mask, uint8_t* mask_out, int mask_bits, uint64_t seed, void* S, float* ws, int M, int K, int R,
                        const LfSegTable& seg, int dtype, hipStream_t st) {
  StreamArgs a{};
  a.p0 = X; a.n0 = (int)xa_rows_of(M, seg); a.K = K; a.n_slices = lf_xa_stream_slices(M, K, R, mask != nullptr || mask_out != nullptr, seg);
  a.mask = mask; a.mask_out = mask_out; a.mask_bytes = !mask_bits; a.seed_lo = (uint32_t)seed; a.seed_hi = (uint32_t)(seed >> 32);
  a.S = S; a.M = M; a.R = R;
  return dtype == LF_BF16 ? xa_stream_impl<__bf16>(a, seg, ws, st) : xa_stream_impl<_Float16>(a, seg, ws, st);
}

// ---- dS = scale dY B_i, complete: to rank 32 on the ring kernel, above in slices of N.
// ws: lf_ds_workspace bytes
size_t lf_ds_workspace(int M, int N, int R, const LfSegTable& seg) { return R <= 32 ? 0 : lf_xa_stream_workspace(M, N, R, false, seg); }
template <typename T>
static int ds_impl(const void* dY, void* dS, float* ws, int M, int N, int R, const LfSegTable& seg, hipStream_t st) {
  const int rows = (int)xa_rows_of(M, seg);
  if (R <= 32) return R <= 16 ? xa_ring_launch<T, 1, true>(dY, dS, M, rows, N, R, seg, st) : xa_ring_launch<T, 2, true>(dY, dS, M, rows, N, R, seg, st);
  StreamArgs a{};
  a.p0 = dY; a.n0 = rows; a.K = N; a.n_slices = lf_xa_stream_slices(M, N, R, false, seg); a.S = dS; a.M = M; a.R = R;
  a.part = a.n_slices > 1 ? ws : nullptr;
  const int groups = (rows + SROWS - 1) / SROWS;
  const int rc = rt_of(R) == 4 ? stream_launch<T, 4, 0, false, true>(a, seg, groups, st) : stream_launch<T, 8, 0, false, true>(a, seg, groups, st);
  if (rc != LF_OK || a.part == nullptr) return rc;
  const int64_t n4 = ((int64_t)rows * R + 3) / 4;
  return lf_launch((stream_reduce_kernel<T>), dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, st, (const float*)ws, (T*)dS, a.n_slices, M, R, 2, seg);
}
int lf_launch_ds(const void* dY, void* dS, void* ws, int M, int N, int R, const LfSegTable& seg, int dtype, hipStream_t st) {
  return dtype == LF_BF16 ? ds_impl<__bf16>(dY, dS, (float*)ws, M, N, R, seg, st) : ds_impl<_Float16>(dY, dS, (float*)ws, M, N, R, seg, st);
}

// ---- forward of a short batch (one adapter, no keep-mask)
static int short_pitch(int N, int rank) { return N + (rank + 15) / 16 * 16; }
static int short_groups(int N, int rank) { return N / SROWS + (rank + SROWS - 1) / SROWS; }

// Up to 64 rows the pass reads W at 4-5 TB/s where tiles of 64 columns leave most of the chip idle (6 x 4096 x 4096: 23.7 ->
// 12.0 us, 9.0 in one launch, 64 rows: 24.9 -> 14.5).  Up to 128 rows a workgroup fetches twice as many bytes
// of X from L2 as of W: still ahead where the output is too narrow to fill the chip with tiles (128 x 4096 x 4096: 25.3 ->
// 20.9).  What it loses is the second stage, whose workgroups (64 columns x 16 rows) form the LoRA term one column per lane, in time
// with their number and the rank, while the general path's disadvantage grows with K: the line is fitted to 620 shapes of 8 - 128 rows,
// K of 1024 - 14336, 1024 - 14336 columns and ranks 16 - 128, where the faster path is 0.4 % ahead of the chosen one on average
// (64 x 14336 over 1024: rank 16 17.2 against 14.7 us, rank 128 48.7 against 21.1; over 4096 at rank 16 38.5 against 38.3;
// 48 x 7168 over 2048: 14.6 against 16.7 at rank 16, 26.2 against 22.3 at 128).
bool lf_short_fwd_applies(int M, int N, int K, int rank) {
  if (M > 128 || (M > 64 && N > 4096)) return false;
  const double finish = (double)(N / 64) * ((M + 15) / 16) * (M > 64 ? 1.5 : 1.0);
  return finish <= 255.0 + (200.0 + 0.2 * (K - 1024)) * (28.0 / (12 + rank));
}

static int short_slices(int M, int N, int K, int rank) {
  return slices_for(short_groups(N, rank), K, (double)M * short_pitch(N, rank) * sizeof(float), kFwdSlices);
}
size_t lf_short_fwd_workspace(int M, int N, int K, int rank) {
  return (size_t)short_slices(M, N, K, rank) * M * short_pitch(N, rank) * sizeof(float);
}

template <typename T>
static int short_fwd_impl(const StreamArgs& a, const LfSegTable& seg, const void* B, float scale, const void* bias, void* Y, hipStream_t st) {
  int rc = stream_rt<T>(a, seg, a.M, short_groups(a.n0, a.n1), st);
  if (rc != LF_OK) return rc;
  return lf_launch((short_fwd_finish_kernel<T>), dim3(a.n0 / 64, (a.M + 15) / 16), dim3(256), 0, st, (const float*)a.part, a.pitch,
                   a.n_slices, a.M, a.n0, a.n1, a.R, (const T*)B, scale, (const uint16_t*)bias, (T*)Y, (T*)a.S);
}

// The one-launch form, against the two launches, over 8 widths of 128 - 14336 columns, K of 1024 - 14336, 1 - 16 rows, ranks 8 - 32.  A workgroup walks
// all of K at what one compute unit takes in, so it loses where K is long and the columns are few, and earlier at rank 32, which adds a third
// to its bytes: 16 x 1024 x 6144 rank 16 10.0 against 10.3 us, x 8192 11.4 against 11.0; 6 x 1024 x 4096 rank 32 7.7 against 8.9,
// x 5120 10.0 against 9.2.  From 3072 columns the two launches have more to stream: 16 x 3072 x 7168 rank 32 13.7 against 14.7.  In groups of 64 columns: 16 x
// 4224 x 4096 rank 16 12.8 against 13.0, rank 32 14.8 against 14.0, 6 x 8192 rank 32 14.8 against 18.9.  More than 256 groups are a second round: 6 x 17408 x 4096
// 47.3 against 40.8.
static bool short16_applies(int M, int N, int K, int rank) {
  if (M > 16 || rank > 32 || N > 256 * 64) return false;
  if (N > 4096) return K <= (rank <= 16 || N >= 8192 ? 4096 : 2048);
  return K <= (N >= 3072 ? 7168 : rank <= 16 ? 6144 : 4096);
}

template <typename T, int RT, int G>
static int short16_launch(const void* X, const void* W, const void* A, const void* B, float scale, const void* bias, void* Y, void* S, int M, int N, int K,
                          int rank, int R, hipStream_t st) {
  auto kern = short16_fwd_kernel<T, RT, G>;
  constexpr int SMEM = short16_waves(G) * short16_stages(RT, G) * (G + 1 + RT) * 2048;
  static LfLdsFlags lds_ok;
  if (!lf_allow_lds(kern, SMEM, lds_ok)) return LF_ELAUNCH;
  return lf_launch(kern, dim3(N / (16 * G)), dim3(short16_waves(G) * 64), SMEM, st, X, W, A, (const T*)B, scale, (const uint16_t*)bias, (T*)Y, (T*)S, M, N, K,
                   rank, R);
}
template <typename T>
static int short16_impl(const void* X, const void* W, const void* A, const void* B, float scale, const void* bias, void* Y, void* S, int M, int N, int K,
                        int rank, int R, hipStream_t st) {
  auto launch = rank <= 16 ? (N <= 4096 ? short16_launch<T, 1, 1> : short16_launch<T, 1, 4>) : N <= 4096 ? short16_launch<T, 2, 1> : short16_launch<T, 2, 4>;
  return launch(X, W, A, B, scale, bias, Y, S, M, N, K, rank, R, st);
}

int lf_launch_short_fwd(const void* X, const void* W, const void* A, const void* B, float scale, const void* bias, void* Y, void* S, void* ws,
                        int M, int N, int K, int rank, int R, const LfSegTable& seg, int dtype, hipStream_t st) {
  if (short16_applies(M, N, K, rank)) {
    auto one = dtype == LF_BF16 ? short16_impl<__bf16> : short16_impl<_Float16>;
    return one(X, W, A, B, scale, bias, Y, S, M, N, K, rank, R, st);
  }
  StreamArgs a{};
  a.p0 = W; a.p1 = A; a.n0 = N; a.n1 = rank; a.K = K; a.n_slices = short_slices(M, N, K, rank);
  a.part = (float*)ws; a.pitch = short_pitch(N, rank); a.S = S; a.M = M; a.R = R; a.q = X;
  return dtype == LF_BF16 ? short_fwd_impl<__bf16>(a, seg, B, scale, bias, Y, st) : short_fwd_impl<_Float16>(a, seg, B, scale, bias, Y, st);
}
