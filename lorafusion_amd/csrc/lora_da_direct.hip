// dA of short segments in one launch, without fp32 partials: the direct form of the dA kernel (rank_ring.h), for gfx950.  The products it
// is the faster one for: da_form, and with dB beside it short_grads (both in lora_skinny.hip).
//
// With and without dB are instances of their own: in one, the operands of dB stand in the way of a launch of 5 - 8 us that has none (1441 products of packed batches 2.1 % faster apart, four
// segments of one block x 2432 at rank 16 with keep bits 6.1 -> 5.7 us; backwards level).
// A source of its own so that its 64 instances are a code object of their own; when the 32 without dB were inside that of the other rank-r kernels (3.0 MB with them, 1.7 without)
// they cost passes that never launch them: forward + backward of 2048 x 4096 x 4096 at rank 16 154.0 us with them inside, 153.5 without (three runs each,
// in turn; 153.9 before the direct form existed), with the same instructions in every kernel that runs.
#include <algorithm>
#include "rank_ring.h"

namespace {

// Alone on its compute unit: ring stages and dS buffers.  (A seventh stage without a mask, and a wait that leaves it in flight: 128 - 1000 rows x 2048 -
// 14336 at ranks 16 and 32 within 1 % either way.)
constexpr int da1_nsb(int rt) { return rt <= 2 ? 4 : rt == 4 ? 3 : 2; }
constexpr int da1_ns(int rt, int maskfmt) { return maskfmt == 1 ? (rt <= 2 ? 5 : 4) : rt <= 2 ? (maskfmt ? 7 : 6) : rt == 4 ? 6 : 5; }

template <typename T, int RT, int MASK, bool WITH_B>
int launch_form(const void* X, const uint8_t* mask, const void* dS, int M, int K, int R, int n_slices, const LfSegTable& seg, const DbOperands& db, hipStream_t st) {
  constexpr int NS = da1_ns(RT, MASK), NSB = da1_nsb(RT), smem = NS * (TILE_BYTES + da_mask_tile_bytes(MASK)) + NSB * ROWS * RT * 32;
  static_assert(smem <= 160 * 1024, "ring and dS buffers fit the LDS");
  auto kern = lora_da_ring_kernel<T, RT, da_tpw(RT), NS, MASK, NSB, true, WITH_B>;
  static LfLdsFlags lds_ok;
  if (!lf_allow_lds(kern, smem, lds_ok)) return LF_ELAUNCH;
  return lf_launch(kern, dim3(std::max(n_slices, db.n_slices), WITH_B ? 2 : 1, seg.table ? seg.n_seg : 1), dim3(256), smem, st, (const T*)X, mask, (const T*)dS, (float*)nullptr, M, K, R, n_slices,
                   1 << 20, 1, seg, db);
}
template <typename T, int RT, int MASK>
int launch(const void* X, const uint8_t* mask, const void* dS, int M, int K, int R, int n_slices, const LfSegTable& seg, const DbOperands& db, hipStream_t st) {
  return db.dY != nullptr ? launch_form<T, RT, MASK, true>(X, mask, dS, M, K, R, n_slices, seg, db, st) : launch_form<T, RT, MASK, false>(X, mask, dS, M, K, R, n_slices, seg, db, st);
}
template <typename T, int RT>
int launch_mask(const void* X, const uint8_t* mask, int fmt, const void* dS, int M, int K, int R, int n_slices, const LfSegTable& seg, const DbOperands& db, hipStream_t st) {
  switch (fmt) {
    case 0: return launch<T, RT, 0>(X, mask, dS, M, K, R, n_slices, seg, db, st);
    case 1: return launch<T, RT, 1>(X, mask, dS, M, K, R, n_slices, seg, db, st);
    case 2: return launch<T, RT, 2>(X, mask, dS, M, K, R, n_slices, seg, db, st);
    default: return launch<T, RT, 3>(X, mask, dS, M, K, R, n_slices, seg, db, st);
  }
}
template <typename T>
int launch_rank(const void* X, const uint8_t* mask, int fmt, const void* dS, int M, int K, int R, int n_slices, const LfSegTable& seg, const DbOperands& db, hipStream_t st) {
  switch (rt_of(R)) {
    case 1: return launch_mask<T, 1>(X, mask, fmt, dS, M, K, R, n_slices, seg, db, st);
    case 2: return launch_mask<T, 2>(X, mask, fmt, dS, M, K, R, n_slices, seg, db, st);
    case 4: return launch_mask<T, 4>(X, mask, fmt, dS, M, K, R, n_slices, seg, db, st);
    default: return launch_mask<T, 8>(X, mask, fmt, dS, M, K, R, n_slices, seg, db, st);
  }
}

}  // namespace

// mask_fmt: the kernel's MASK
int lf_launch_da_direct(const void* X, const uint8_t* mask, int mask_fmt, const void* dS, int M, int K, int R, int n_slices, const LfSegTable& seg, const void* dY,
                        const void* S, int N, int n_slices_b, int dtype, hipStream_t st) {
  const DbOperands db{dY, S, N, dY != nullptr ? n_slices_b : 0};
  return dtype == LF_BF16 ? launch_rank<__bf16>(X, mask, mask_fmt, dS, M, K, R, n_slices, seg, db, st)
                          : launch_rank<_Float16>(X, mask, mask_fmt, dS, M, K, R, n_slices, seg, db, st);
}
