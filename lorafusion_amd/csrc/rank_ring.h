// The ring of direct-to-LDS loads that the rank-r passes with a contraction over rows stream their operand through, its LDS tile layouts, and the dA
// kernel, whose two forms are compiled in two sources (lora_skinny.hip: two stages; lora_da_direct.hip: direct) (internal).
#pragma once
#include "lf_common.h"
#include "rank_common.h"

namespace {

constexpr int TILE_BYTES = ROWS * 128;  // 128 rows x 64 columns of 16-bit

// Swizzle key of a tile row: granule g of row r sits at slot g ^ tile_key(r).  LDS serves a 16-byte read 16 lanes at
// a time and an 8-byte (transposed) read 32 lanes at a time, in both cases 256 bytes = all 64 banks.  Row fragments:
// 16 consecutive rows, one granule each -- the 8 rows of one parity need 8 different keys.  Transposed fragments:
// rows j, 8+j (j = 0..3), two neighbouring granules each -- the 4 rows of one parity (r>>1 = 0, 1, 4, 5 mod 8) need 4
// different key>>1.  The three bits of r>>1 rotated by one do both (with the bits in place, 0/1 and 4/5 share key>>1:
// every transposed read took two passes).
__device__ __forceinline__ int tile_key(int row) {
  const int x = (row >> 1) & 7;
  return ((x & 1) << 2) | (x >> 1);
}

// Row fragment: 8 consecutive columns (granule g) of `row`.
__device__ __forceinline__ lf_u32x4 tile_row_frag(const char* tile, int row, int g) {
  return *(const lf_u32x4*)(tile + row * 128 + ((g ^ tile_key(row)) << 4));
}

// Transposed fragment: rows row..row+3 and row+4..row+7 of the lane's column; `col` is the first
// of the 4 columns this lane addresses (multiple of 4).
__device__ __forceinline__ lf_u32x4 tile_tr_frag(const char* tile, int row, int col) {
  const int g = col >> 3, within = (col & 7) * 2;
  const char* p0 = tile + row * 128 + ((g ^ tile_key(row)) << 4) + within;
  const char* p1 = tile + (row + 4) * 128 + ((g ^ tile_key(row + 4)) << 4) + within;
  lf_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) lf_s16x4*)(p0));
  lf_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) lf_s16x4*)(p1));
  lf_u32x2 a = __builtin_bit_cast(lf_u32x2, lo), b = __builtin_bit_cast(lf_u32x2, hi);
  return lf_u32x4{a[0], a[1], b[0], b[1]};
}

// Blocks [b0, b1) of segment s.
__device__ __forceinline__ void segment_blocks(const LfSegTable& seg, int s, int M, int& b0, int& b1) {
  if (seg.table == nullptr) {
    b0 = 0;
    b1 = (M + ROWS - 1) / ROWS;
  } else {
    b0 = seg.first_block[s];
    b1 = (s + 1 < seg.n_seg) ? seg.first_block[s + 1] : seg.n_blocks;
  }
}

// Chunk ch of the blocks [b0, b1) when they are cut into ceil((b1 - b0) / group) chunks of nearly equal size (empty
// beyond the last chunk).
__device__ __forceinline__ void chunk_blocks(int b0, int b1, int group, int ch, int& bb0, int& bb1) {
  const int n = b1 - b0, nch = (n + group - 1) / group;
  if (n <= 0 || ch >= nch) { bb0 = bb1 = b1; return; }
  const int base = n / nch, rem = n % nch;
  bb0 = b0 + ch * base + min(ch, rem);
  bb1 = bb0 + base + (ch < rem ? 1 : 0);
}

// ------------------------------------------------------------------ streaming through a ring of direct-to-LDS loads
// A tile that waits in registers between its load and its LDS store leaves a workgroup one tile on order -- a CU 16-48 KB, half of
// what the HBM latency asks for and less.  The kernels below order their tiles as buffer loads that write LDS themselves (no
// registers, no store instructions), NS - 1 tiles ahead of the one being consumed.  (Ranks above 64, one workgroup per CU
// either way: 3000 x 5120 at rank 128, dys_dyb 33.8 -> 26.6 us and da 35.2 -> 22.0 against the register-staged form.  What bounds
// them there: 61 MB and 16 MB of fp32 partials beside 31 MB of operand, and the two or three stages that fit next to the side blocks.)
//
// A load group is waited for by count: vector memory operations complete in issue order, so "at most n younger
// operations outstanding" means the group has landed.  The loop therefore contains no other vector memory
// instruction (the compiler would count only its own and wait for everything), issues a group of the same size
// every iteration (past the end: the last tile again, unconsumed), and drains the ring before the workgroup ends.
// Rows past the end of a matrix are not clamped: every tile gets a buffer descriptor that ends where the matrix
// ends, and lanes beyond it read zeros, which add nothing to a sum over rows.
constexpr int da_tpw(int rt) { return rt >= 4 ? 8 : 16; }   // dA: tiles per slice (registers: TPW * RT * 4 accumulators)
constexpr int da_mask_tile_bytes(int fmt) { return fmt == 1 ? ROWS * 64 : fmt == 2 ? ROWS * 8 : 0; }
// Per-thread window offsets of a 128-row x 64-column tile of a 16-bit matrix with `ld` elements per row, in the LDS
// layout the fragment readers expect (position p = i*256 + tid: row p>>3, slot p&7 holds granule slot ^ tile_key(row)).
__device__ __forceinline__ void tile_voffs(uint32_t (&v)[4], int64_t ld, int tid) {
  const int srcg = (tid & 7) ^ tile_key(tid >> 3);
#pragma unroll
  for (int i = 0; i < 4; i++) v[i] = (uint32_t)((int64_t)(i * 32 + (tid >> 3)) * ld * 2 + srcg * 16);
}
__device__ __forceinline__ void tile_dma(const lf_u32x4& rsrc, const uint32_t (&v)[4], uint32_t lds_tile, int wave) {
#pragma unroll
  for (int i = 0; i < 4; i++) dma16(rsrc, v[i], lds_tile + i * 4096 + wave * 1024);
}
// keep-mask bytes of the same tile: 128 rows of 64 bytes, row-major (position p = i*256 + tid: row p>>2, 16-byte chunk p&3)
__device__ __forceinline__ void mask_voffs(uint32_t (&v)[2], int64_t ld, int tid) {
#pragma unroll
  for (int i = 0; i < 2; i++) v[i] = (uint32_t)((int64_t)(i * 64 + (tid >> 2)) * ld + (tid & 3) * 16);
}
__device__ __forceinline__ void mask_dma(const lf_u32x4& rsrc, const uint32_t (&v)[2], uint32_t lds_mask, int wave) {
#pragma unroll
  for (int i = 0; i < 2; i++) dma16(rsrc, v[i], lds_mask + i * 4096 + wave * 1024);
}
// keep-mask applied in place to a landed tile (any thread mapping; here each thread takes the positions p = i*256 + tid)
// (BITS: the mask tile holds 8 bytes per row, one bit per element)
template <bool BITS>
__device__ __forceinline__ void tile_apply_mask(char* tile, const char* mtile, int tid) {
  lf_u32x4 x[4];
  lf_u32x2 m[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {   // all reads first: behind a store the compiler would not start the next read
    const int p = i * 256 + tid, row = p >> 3, g = (p & 7) ^ tile_key(row);
    x[i] = *(const lf_u32x4*)(tile + p * 16);
    if constexpr (BITS) m[i] = expand_keep8(*(const uint8_t*)(mtile + row * 8 + g));
    else m[i] = *(const lf_u32x2*)(mtile + row * 64 + g * 8);
  }
#pragma unroll
  for (int i = 0; i < 4; i++) *(lf_u32x4*)(tile + (i * 256 + tid) * 16) = apply_mask8(x[i], m[i]);
}
// the same for a mask of bytes that is read from memory here, `mask` at the tile's first element: any address, rows of K bytes, `rows` of them
__device__ __forceinline__ void tile_apply_bytes(char* tile, const uint8_t* mask, int64_t K, int64_t rows, int tid) {
  lf_u32x4 x[4];
  lf_u32x2 m[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int p = i * 256 + tid, row = p >> 3, g = (p & 7) ^ tile_key(row);
    x[i] = *(const lf_u32x4*)(tile + p * 16);
    m[i] = lf_u32x2{0, 0};
    if (row < rows) m[i] = keep_bytes8(mask + row * K + g * 8);
  }
#pragma unroll
  for (int i = 0; i < 4; i++) *(lf_u32x4*)(tile + (i * 256 + tid) * 16) = apply_mask8(x[i], m[i]);
}

// A [rows x RT*16] side operand (S or dS block: 128 rows; B tile: 64 rows) in LDS: rows of RT*32 bytes; granule g of
// source row r at slot g ^ side_key(r) of LDS row side_row(r).  A transposed read is served 32 lanes at a time: rows
// j, 8+j (j = 0..3), 32 bytes of each, which must land on eight different 32-byte groups of the 64 banks.  At 256-byte rows
// (all start on one bank) the key tells all eight apart; at 128-byte
// rows the key separates (r>>3)&1 and (r>>1)&1 (the row's parity picks the half of the banks); at 64-byte rows
// (r>>3)&1; at 32-byte rows no key can (a row is one group): rows 8..15 of every 16 swap their halves instead.
template <int RT>
__device__ __forceinline__ int side_key(int row) {
  if constexpr (RT == 8) return ((row & 3) << 1) | (((row >> 3) & 1) << 3);
  return RT >= 4 ? ((((row >> 3) & 1) << 1) | (((row >> 1) & 1) << 2)) : RT == 2 ? ((row >> 3) & 1) << 1 : 0;
}
template <int RT>
__device__ __forceinline__ int side_row(int row) { return RT == 1 ? row ^ (((row >> 3) & 1) << 2) : row; }
// window offsets of the granules this thread fetches: position p = i*256 + tid -> row p / (2 RT), slot p % (2 RT); a
// granule beyond `cols` columns does not exist in memory: the first one is fetched instead (its products land in
// rank columns that the reduce discards)
template <int RT, int NI>
__device__ __forceinline__ void side_voffs(uint32_t (&v)[NI], int pitch_elems, int cols, int tid) {
#pragma unroll
  for (int i = 0; i < NI; i++) {
    const int p = i * 256 + tid, row = side_row<RT>(p / (RT * 2)), g = (p % (RT * 2)) ^ side_key<RT>(row);   // side_row is its own inverse
    v[i] = (uint32_t)(row * pitch_elems * 2 + (g * 8 < cols ? g : 0) * 16);
  }
}
template <int NI>
__device__ __forceinline__ void side_dma(const lf_u32x4& rsrc, const uint32_t (&v)[NI], uint32_t lds_side, int wave) {
#pragma unroll
  for (int i = 0; i < NI; i++) dma16(rsrc, v[i], lds_side + i * 4096 + wave * 1024);
}
// transposed fragment: rows row..row+3 and row+4..row+7 (row % 8 < 4) of the lane's column among columns c*16 + 4*c4 ..
template <int RT>
__device__ __forceinline__ lf_u32x4 side_tr8(const char* blk, int row, int c, int c4) {
  const int g = c * 2 + (c4 >> 1), within = (c4 & 1) * 8;
  const char* p0 = blk + side_row<RT>(row) * (RT * 32) + ((g ^ side_key<RT>(row)) << 4) + within;
  const char* p1 = blk + side_row<RT>(row + 4) * (RT * 32) + ((g ^ side_key<RT>(row + 4)) << 4) + within;
  lf_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) lf_s16x4*)(p0));
  lf_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) lf_s16x4*)(p1));
  lf_u32x2 a = __builtin_bit_cast(lf_u32x2, lo), b = __builtin_bit_cast(lf_u32x2, hi);
  return lf_u32x4{a[0], a[1], b[0], b[1]};
}

// ---- da.  grid (n_slices, max_chunks, n_seg).  Workgroup (ks, ch, s): the k-tiles of slice ks (at most TPW, at least
// two -- one in the direct form, which has no partials -- and slices are balanced) and the `group` row blocks ch*group.. of segment s; pairs (block, tile) in block-major
// order, the dS block of a row block is fetched once, with the block's first tile, into one of NSB buffers (a slice
// of nt tiles keeps at most min(NS, (NSB - 1) nt + 1) stages of the ring busy, so one block more is never on order).
//   D_j[r][k] += sum_m dS[m][r] * keep*X[m][k]   per tile j of the slice, in registers over all blocks of the chunk.
// With a keep-mask the tile is masked in place one iteration before it is consumed.
// The direct form takes dB with dA (WITH_B): the workgroups of blockIdx.y = 1 walk dY beside S without a mask, the same sum with other operands.
struct DbOperands { const void* dY; const void* S; int N, n_slices; };   // (outputs: seg.ptr)
template <typename T, int RT, int TPW, int NS, int MASK, int NSB, bool DIRECT, bool WITH_B = false>
__global__ void __launch_bounds__(256, RT >= 8 || DIRECT ? 1 : 2)
lora_da_ring_kernel(const T* __restrict__ X, const uint8_t* __restrict__ mask, const T* __restrict__ dS, float* __restrict__ part,
                    int M, int K, int R, int n_slices, int group, int max_chunks, const LfSegTable seg, const DbOperands db) {
  // MASK: 0 no keep-mask; 1 one byte per element (8 KB per tile, two loads per thread); 2 one bit per element (1 KB per
  // tile, one 4-byte load per thread); 3 one byte per element at an address that the direct loads do not take, read where it is applied (the compiler's
  // waits for those loads empty the ring every tile)
  constexpr int STAGE = TILE_BYTES + da_mask_tile_bytes(MASK);
  constexpr int SIDE = ROWS * RT * 32;
  constexpr int G = 4 + (MASK == 1 ? 2 : MASK == 2 ? 1 : 0);   // operations per load group and thread, not counting a dS block
  static_assert(NS - (MASK ? 3 : 2) <= WAIT_MOST, "every stage of the ring is used");
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  char* ring = lds;
  char* side = lds + NS * STAGE;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  const int ks = blockIdx.x, ch = DIRECT ? 0 : blockIdx.y, s = blockIdx.z;
  const bool grad_b = WITH_B && blockIdx.y != 0;
  if constexpr (WITH_B) {
    if (grad_b) X = (const T*)db.dY, dS = (const T*)db.S, K = db.N, n_slices = db.n_slices, mask = nullptr;
    if (ks >= n_slices) return;
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = to_sgpr(tid >> 6);
  const int li = lane & 15, qq = lane >> 4, j4 = li >> 2, c4 = li & 3;
  int b0, b1, bb0, bb1;
  segment_blocks(seg, s, M, b0, b1);
  chunk_blocks(b0, b1, group, ch, bb0, bb1);
  if (bb0 >= bb1) {  // this segment has fewer chunks (uniform for the whole workgroup)
    if constexpr (DIRECT) {   // no rows at all: a sum of nothing
      const int T64 = K / 64, k0 = (ks * (T64 / n_slices) + min(ks, T64 % n_slices)) * 64, nk = (T64 / n_slices + (ks < T64 % n_slices ? 1 : 0)) * 64;
      if (grad_b) for (int i = tid; i < seg.rank[s] * nk; i += 256) ((uint16_t*)seg.ptr[s])[(int64_t)k0 * seg.rank[s] + i] = 0;
      else for (int i = tid; i < seg.rank[s] * nk; i += 256) ((uint16_t*)seg.out[s])[(int64_t)(i / nk) * K + k0 + i % nk] = 0;
    }
    return;
  }
  const float p = seg.table ? (seg.block_p ? seg.block_p[b0] : 0.f) : seg.p;
  const bool use_mask = MASK && mask != nullptr && p > 0.f;
  const int64_t Mrows = seg.table ? (int64_t)seg.n_blocks * ROWS : M;
  const int T64 = K / 64;
  const int kt0 = ks * (T64 / n_slices) + min(ks, T64 % n_slices);
  const int nt = T64 / n_slices + (ks < T64 % n_slices ? 1 : 0);
  const int ns = min(NS, (NSB - 1) * nt + 1);   // stages in use

  uint32_t xv[4], mv[2], dv[RT];
  tile_voffs(xv, K, tid);
  if constexpr (MASK == 2) mv[0] = mv[1] = (uint32_t)((tid >> 1) * (K >> 3) + (tid & 1) * 4);   // row tid>>1, half tid&1 of its 8 bytes
  else mask_voffs(mv, K, tid);
  side_voffs<RT, RT>(dv, R, R, tid);

  // Load group of the next pair into stage `ist`; behind the last pair the last tile is ordered again.  The windows
  // move with the pair (byte pointers and bytes left up to the end of the matrix): a few scalar additions per group.
  int ib = bb0, ij = 0, ist = 0;
  const char* xb = (const char*)(X + (int64_t)bb0 * ROWS * K + (int64_t)kt0 * 64);
  int64_t xleft = (((int64_t)Mrows - (int64_t)bb0 * ROWS) * K - (int64_t)kt0 * 64) * 2;
  const char* sb = (const char*)(dS + (int64_t)bb0 * ROWS * R);
  int64_t sleft = ((int64_t)Mrows - (int64_t)bb0 * ROWS) * R * 2;
  // (rows of the segment's last block behind its valid ones read as zeros)
  const int64_t slast = (int64_t)to_sgpr(seg.table ? seg.table[3 * (b1 - 1) + 1] : ROWS) * R * 2;
  const int64_t xnext = (int64_t)ROWS * K * 2 - (int64_t)nt * 128;   // from behind a block's last tile to the next block's first
  auto issue = [&]() {
    tile_dma(window_rsrc(xb, xleft), xv, lds0 + ist * STAGE, wave);
    if constexpr (MASK == 1) {
      // the mask has one byte where X has two: same element offsets, half the byte offsets
      const int64_t eoff = (xb - (const char*)X) >> 1;
      mask_dma(window_rsrc(mask != nullptr ? (const char*)mask + eoff : (const char*)X, mask != nullptr ? (xleft >> 1) : 0), mv,
               lds0 + ist * STAGE + TILE_BYTES, wave);
    }
    if constexpr (MASK == 2) {
      // one bit where X has sixteen: the tile's 128 rows x 8 bytes land row-major (wave w: rows 32w .. 32w+31)
      const int64_t boff = (xb - (const char*)X) >> 4;
      dma4(window_rsrc(mask != nullptr ? (const char*)mask + boff : (const char*)X, mask != nullptr ? (xleft >> 4) : 0), mv[0],
           lds0 + ist * STAGE + TILE_BYTES + wave * 256);
    }
    if (ij == 0 && ib < bb1) side_dma<RT>(window_rsrc(sb, ib == b1 - 1 ? min(sleft, slast) : sleft), dv, lds0 + NS * STAGE + ((uint32_t)(ib - bb0) % NSB) * SIDE, wave);
    ist = ist + 1 == ns ? 0 : ist + 1;
    if (ib < bb1) {
      if (++ij < nt) {
        xb += 128, xleft -= 128;
      } else if (ib + 1 < bb1) {
        ij = 0, ib++;
        xb += 128 + xnext, xleft -= 128 + xnext;
        sb += ROWS * R * 2, sleft -= ROWS * R * 2;
      } else {
        ib = bb1;   // the cursor stays on the last tile
      }
    }
  };
#pragma unroll 1
  for (int i = 0; i < ns - 1; i++) issue();

  lf_f32x4 acc[TPW][RT];
#pragma unroll
  for (int t = 0; t < TPW; t++)
#pragma unroll
    for (int c = 0; c < RT; c++) acc[t][c] = lf_f32x4{0.f, 0.f, 0.f, 0.f};

  int cst = 0;   // stage of the pair being consumed
  auto apply_mask = [&](char* stage, int b, int t) {   // (tile t of block b)
    if constexpr (MASK == 3) {
      const int64_t row = (int64_t)b * ROWS;
      tile_apply_bytes(stage, mask + row * K + (kt0 + t) * 64, K, Mrows - row, tid);
    } else {
      tile_apply_mask<MASK == 2>(stage, stage + TILE_BYTES, tid);
    }
  };
  if constexpr (MASK) {
    wait_groups<G>(ns - 2);
    ring_barrier();
    if (use_mask) apply_mask(ring, bb0, 0);
  }
  for (int b = bb0; b < bb1; b++) {
    const char* dcur = side + ((uint32_t)(b - bb0) % NSB) * SIDE;
    lf_u32x4 df[4][RT];
#pragma unroll
    for (int t = 0; t < TPW; t++) {
      if (t < nt) {
        // MASK: the next pair's group has landed (it is masked during this iteration); else this pair's
        wait_groups<G>(MASK ? ns - 3 : ns - 2);
        ring_barrier();   // ... for every thread; and everyone is done with the previous pair's stage
        issue();
        if constexpr (MASK) {
          const int nst = cst + 1 == ns ? 0 : cst + 1;
          // (behind the last pair the last tile is there again, unconsumed: any mask of the matrix does)
          if (use_mask) apply_mask(ring + nst * STAGE, t + 1 < nt || b + 1 == bb1 ? b : b + 1, t + 1 < nt ? t + 1 : 0);
        }
        const char* xcur = ring + cst * STAGE;
        // all fragments of the tile first, then the MFMAs: with one or two waves per SIMD nothing else hides the LDS
        // latency, and read-wait-multiply in turns costs a latency per MFMA
        lf_u32x4 xt[4];
        if (t == 0) {   // the dS fragments serve every tile of the block
#pragma unroll
          for (int kk = 0; kk < 4; kk++)
#pragma unroll
            for (int c = 0; c < RT; c++) df[kk][c] = side_tr8<RT>(dcur, kk * 32 + qq * 8 + j4, c, c4);
        }
#pragma unroll
        for (int kk = 0; kk < 4; kk++) xt[kk] = tile_tr_frag(xcur, kk * 32 + qq * 8 + j4, wave * 16 + 4 * c4);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
#pragma unroll
          for (int c = 0; c < RT; c++) acc[t][c] = Mfma16<T>::run(df[kk][c], xt[kk], acc[t][c]);
        __builtin_amdgcn_sched_barrier(0);
        cst = cst + 1 == ns ? 0 : cst + 1;
      }
    }
  }
  wait_vm<0>();   // the unconsumed loads behind the last pair must not land in another workgroup's LDS
  // C layout: column (k) = lane & 15, rows (r) = 4*(lane >> 4) + e
  if constexpr (DIRECT) {   // one chunk per segment: these are the sums
    const int rank = seg.rank[s];
    if (grad_b) {   // [N, rank]: a lane has four neighbours of a row
      const float mult = seg.table ? (seg.block_scale ? seg.block_scale[b0] : 1.f) : seg.scale;
      uint16_t* out = (uint16_t*)seg.ptr[s];
#pragma unroll
      for (int t = 0; t < TPW; t++)
        if (t < nt) {
#pragma unroll
          for (int c = 0; c < RT; c++) {
            const int r = c * 16 + qq * 4;
            if (r < rank) *(lf_u32x2*)(out + (int64_t)((kt0 + t) * 64 + wave * 16 + li) * rank + r) = pack4<T>(acc[t][c] * mult);
          }
        }
      return;
    }
    const float mult = mask != nullptr && p > 0.f ? 1.f / (1.f - p) : 1.f;
    uint16_t* out = (uint16_t*)seg.out[s];
#pragma unroll
    for (int t = 0; t < TPW; t++)
      if (t < nt) {
#pragma unroll
        for (int c = 0; c < RT; c++)
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const int r = c * 16 + qq * 4 + e;
            if (r < rank) out[(int64_t)r * K + (kt0 + t) * 64 + wave * 16 + li] = Mfma16<T>::cvt(acc[t][c][e] * mult);
          }
      }
    return;
  } else {
  float* po = part + ((int64_t)s * max_chunks + ch) * R * K;
#pragma unroll
  for (int t = 0; t < TPW; t++)
    if (t < nt) {
#pragma unroll
      for (int c = 0; c < RT; c++)
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (c * 16 < R) po[(int64_t)(c * 16 + qq * 4 + e) * K + (kt0 + t) * 64 + wave * 16 + li] = acc[t][c][e];
    }
  }
}

}  // namespace
