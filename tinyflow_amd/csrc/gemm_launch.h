// Host side of the contraction kernels' in-kernel fold (gemm_core.h: Fold): the
// decision which tiles of a launch are folded, and the scratch / ticket buffers.
#pragma once

#include "gemm_core.h"
#include "internal.h"

#include <algorithm>
#include <cstdlib>

namespace tf {
namespace gemm {

// TINYFLOW_FOLD (measurements and tests): 0 no folding, 1 only short k-splits,
// 2 only the remainder round, 3 (default) both.
inline int fold_switch() {
  const char *e = getenv("TINYFLOW_FOLD");
  return e && *e ? atoi(e) : 3;
}

// Measured on the ResNet-50 batch-64 layers: folding in the kernel beats the separate
// sum pass up to five pieces (beyond that one workgroup reading all pieces of its tile
// is slower than the lane-parallel pass), and cutting the remainder round pays when a
// piece still runs at least two reduction stages (a one-stage piece is all prologue)
// of a reduction of at least eight.
constexpr int kMaxFoldedSplits = 5;
constexpr int kMinStagesPerTailPiece = 2;
constexpr int kMinStagesForTail = 8;   // shorter reductions (64 channels) lose more to the extra workgroups than they gain
constexpr int kMaxTailPieces = 8;      // 4, 8 and 16 measured the same

// Rewrites `g` (made by make_geometry for the planned number of k-splits) so that
//   * a split of 2..kMaxFoldedSplits becomes pieces of every tile, folded in the kernel;
//   * an unsplit launch of more than one round over the CUs whose last round is
//     partial folds the tiles of that round: with R leftover tiles each is cut into
//     floor(CUs / R) pieces along the reduction, about one short piece per CU,
//     instead of R whole tiles that keep R CUs busy while the rest idle.
// Depends on the shape and the CU count only, so a layer always gets the same
// summation order.
inline void plan_fold(Geometry &g, int K, int BK, int batch) {
  const int mode = fold_switch();
  const int tiles = g.tiles();
  const int k_steps = (K + BK - 1) / BK;
  if (g.splits > 1) {
    if (!(mode & 1) || g.splits > kMaxFoldedSplits || (int64_t)tiles * batch > kFoldTicketSlots) return;
    g.fold_first_tile = 0;
    g.fold_pieces = g.splits;
    g.fold_k_per_piece = g.k_per_split;
    g.splits = 1;
    return;
  }
  if (!(mode & 2) || batch != 1) return;
  const int cus = num_cus();
  if (tiles <= cus) return;
  const int rest = tiles % cus;
  if (rest == 0) return;
  if (k_steps < kMinStagesForTail) return;
  int pieces = std::min(std::min(cus / rest, k_steps / kMinStagesPerTailPiece), kMaxTailPieces);
  if (pieces < 2) return;
  const int steps_per_piece = (k_steps + pieces - 1) / pieces;
  pieces = (k_steps + steps_per_piece - 1) / steps_per_piece;  // no empty piece
  if (pieces < 2) return;
  g.fold_first_tile = tiles - rest;
  g.fold_pieces = pieces;
  g.fold_k_per_piece = steps_per_piece * BK;
}

struct FoldBuffers {
  float *scratch = nullptr;
  unsigned *tickets = nullptr;
  size_t bytes = 0;
  hipStream_t stream = nullptr;
};

// Scratch and tickets for the folded tiles of `g`, entered into `g`: 0 ok (also when
// nothing is folded), 1 when the scratch cannot be had (fb.bytes = size wanted), -1 on error.
inline int acquire_fold(Geometry &g, int bm, int bn, int batch, hipStream_t s, FoldBuffers &fb) {
  if (g.fold_pieces <= 1) return 0;
  fb.bytes = g.fold_scratch_bytes(bm, bn, batch);
  fb.tickets = fold_tickets(s);
  if (!fb.tickets) {
    fprintf(stderr, "[tinyflow_amd] no memory for the fold counters\n");
    return -1;
  }
  fb.stream = s;
  fb.scratch = (float *)device_alloc(fb.bytes, s);
  g.fold_scratch = fb.scratch;
  g.fold_ticket_words = fb.tickets;
  return fb.scratch ? 0 : 1;
}
inline void release_fold(FoldBuffers &fb) {
  if (fb.scratch) device_free(fb.scratch, fb.stream);  // stream-ordered reuse
  fb.scratch = nullptr;
}

// ---- cost model of the split engine (gemm_split.h) ------------------------------------------
struct SplitTraffic {
  int which = 0;                         // 0 forward or a plain product, 1 grad-data, 2 grad-filter
  double in_bytes = 0, out_bytes = 0;    // the operand that is not a filter, and the result
  double gather = 1.0;                   // time of a reduction step next to that of one fetched by vectors
  bool scatter = false;                  // the result goes to every u-th row and v-th column, zeros between
};

// Microseconds, fitted to sweeps of every tile and split over 300 layers (ResNet-50 at batch 8 to 128 and 64 to 224
// pixels, random ones of 48 - 512 channels and 1x1 to 7x7 filters): rms error 11 %, its picks within 1.1 % of the
// sweeps' best on average.
//   workgroup time   = a(tile) * gather * (k per split + o(tile)); a tile's start and end cost as much as 70 - 80 steps
//   rounds           = workgroups / CUs, rounded up three quarters of the way
//   latency hiding   = a CU that only ever holds 1 / 2 workgroups runs them at 0.73 / 0.92 of the rate
//   bytes            = nothing runs faster than 5.6 TB/s over operand and result, and 5.8 us a launch
//   split-sum pass   = 7.75 TB/s over the partial results, folds in the kernel 3.8 TB/s
// The 64 x 128 tile had two workgroups a CU in those sweeps; with the three that it has now it takes 4 - 17 % less time than its constants say.
inline double predict_split_us(int M, int N, int K, int bm, int bn, int splits, int stage, const SplitTraffic &t) {
  const Geometry g = make_geometry(M, N, K, bm, bn, splits, stage);
  const double a = bm == 128 ? 0.0316 : bn == 128 ? 0.0223 : 0.0126;
  const double o = bm == 128 ? 69.0 : bn == 128 ? 70.0 : 81.0;
  const double per_cu = (double)g.blocks() / num_cus();
  const double whole = std::ceil(per_cu);
  const double rounds = per_cu <= 1.0 ? 1.0 : std::min(whole, per_cu + 0.75);
  const double hiding = whole <= 1 ? 0.725 : whole <= 2 ? 0.918 : 1.0;
  const bool second_pass = g.splits > kMaxFoldedSplits;
  double us = rounds * a * t.gather * (g.k_per_split + o) / hiding;
  us = std::max(us, (t.out_bytes * (second_pass ? g.splits : 1) + t.in_bytes) / 5.6e6) + 5.8;
  if (second_pass) us += (2.0 * g.splits + 1.0) * t.out_bytes / 7.75e6 + 0.8;
  else if (g.splits > 1) us += (g.splits + 1.0) * t.out_bytes / 3.8e6;
  if (t.scatter) us += t.out_bytes / 14.9e6;
  return us;
}

// Batched products of the transformed domain (`batch` of them; V and M stream by, the time of the transforms and of the sum
// over k-splits is the caller's): the same form with constants of their own, from sweeps over 29 layers of VGG-16 at batch 32 and
// ResNet-50 at batch 64 and 8.  us, measured / model: 256 channels, 6 272 tiles, 128 x 128 178 / 176; 512, 512 tiles 68 / 64, 64 x 128
// 66 / 69; 128, 3 136 tiles 36 / 33; grad-filter 256, 6 272 tiles in 8 pieces 169 / 161; 64 channels 49.5 / 48.  Grad-data's
// filter comes eight bytes a lane on tiles of 64 rows: 1.2 times the time.
inline double predict_split_batched_us(int M, int N, int K, int bm, int bn, int splits, int stage, int which, int batch) {
  const Geometry g = make_geometry(M, N, K, bm, bn, splits, stage);
  const double a = (bm == 128 ? 0.0345 : bn == 128 ? 0.0232 : 0.0141) * (which == 2 ? 1.04 : which == 1 && bm == 64 ? 1.2 : 1.0);
  const double o = bm == 128 ? 109.0 : bn == 128 ? 85.0 : 102.0;
  const double per_cu = (double)g.blocks() * batch / num_cus();
  const double whole = std::ceil(per_cu);
  const double rounds = per_cu <= 1.0 ? 1.0 : std::min(whole, per_cu + 0.75);
  const double hiding = whole <= 1 ? 0.725 : whole <= 2 ? 0.918 : 1.0;
  return rounds * a * (g.k_per_split + o) / hiding;
}

}  // namespace gemm
}  // namespace tf
