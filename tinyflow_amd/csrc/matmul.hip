// DLGpuMatrixMultiply: C = op(A) * op(B) on the fp32 MFMA tile engine.
//
// Replaces the cublasSgemm call of the reference (src/gpu_op.cu:1166-1199).
// The same entry point serves the forward product and both gradients the
// autodiff emits for it (dA = dY * B^T, dB = A^T * dY,
// pycode/tinyflow/autodiff.py:477-506), so all four transpose combinations are
// first-class: a transposed operand only changes which loader reads it.
//
// Skinny problems (few output tiles, long reduction - e.g. a batch-32 fully
// connected layer) are split along k into partial products that a second,
// fixed-order pass adds up, so results do not depend on scheduling.
#include "gemm_core.h"
#include "gemm_launch.h"
#include "gemm_split.h"
#include "internal.h"

#include <algorithm>

using namespace tf;
using namespace tf::gemm;

namespace {

template <int V>
using IC = std::integral_constant<int, V>;
typedef float f32x4 __attribute__((ext_vector_type(4)));

// out[i] = sum_s partial[s * count + i] for 16-byte aligned data with count % 4 == 0, with the
// splits dealt round-robin to SG lane groups of a workgroup so that a small output with
// many splits still has enough loads in flight.  Group g adds splits g, g+SG,
// ... in that order, then group 0 adds the SG group sums in index order: the
// order of additions depends on (splits, SG) only, never on timing.
template <int SG>
__global__ __launch_bounds__(256) void split_sum_vec_kernel(const f32x4 *__restrict__ partial,
                                                           f32x4 *__restrict__ out, int64_t count4, int splits) {
  constexpr int COLS = 256 / SG;
  __shared__ f32x4 part[SG][COLS];
  const int col = threadIdx.x % COLS, g = threadIdx.x / COLS;
  const int64_t i = (int64_t)blockIdx.x * COLS + col;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  if (i < count4) {
    int k = g;
    for (; k + 3 * SG < splits; k += 4 * SG) {
      const f32x4 v0 = __builtin_nontemporal_load(partial + (int64_t)k * count4 + i);
      const f32x4 v1 = __builtin_nontemporal_load(partial + (int64_t)(k + SG) * count4 + i);
      const f32x4 v2 = __builtin_nontemporal_load(partial + (int64_t)(k + 2 * SG) * count4 + i);
      const f32x4 v3 = __builtin_nontemporal_load(partial + (int64_t)(k + 3 * SG) * count4 + i);
      acc = (((acc + v0) + v1) + v2) + v3;
    }
    for (; k < splits; k += SG) acc += __builtin_nontemporal_load(partial + (int64_t)k * count4 + i);
  }
  if (SG == 1) {
    if (i < count4) out[i] = acc;
    return;
  }
  part[g][col] = acc;
  __syncthreads();
  if (g == 0 && i < count4) {
    f32x4 total = part[0][col];
#pragma unroll
    for (int j = 1; j < SG; ++j) total += part[j][col];
    out[i] = total;
  }
}

// Any other output: one lane per element adds the splits in index order.  Bound by the loads' latency: that lane has
// kOrderedDepth of them in flight.  Many splits of few elements go through LDS (sum_through_lds): a workgroup fetches 512 splits of four
// elements at a time, each lane eight values, while four lanes add the ones before.
constexpr int kOrderedDepth = 32;
__global__ __launch_bounds__(64) void split_sum_ordered_kernel(const float *__restrict__ partial,
                                                              float *__restrict__ out, int64_t count, int splits) {
  const int64_t i = (int64_t)blockIdx.x * 64 + threadIdx.x;
  if (i >= count) return;
  float s = partial[i];
  int k = 1;
  for (; k + kOrderedDepth <= splits; k += kOrderedDepth) {
    float v[kOrderedDepth];
#pragma unroll
    for (int e = 0; e < kOrderedDepth; ++e) v[e] = __builtin_nontemporal_load(partial + (int64_t)(k + e) * count + i);
#pragma unroll
    for (int e = 0; e < kOrderedDepth; ++e) s += v[e];
  }
#pragma unroll 4
  for (; k < splits; ++k) s += __builtin_nontemporal_load(partial + (int64_t)k * count + i);
  out[i] = s;
}

// Whether LDS is the better way.  us, one lane an element / through LDS: 150 values in 392 pieces 6.0 / 4.6, 1 021 17.9 / 9.5; 601 in 129
// 3.9 / 3.6; 1 350 in 257 7.3 / 6.5; 2 402 in 513 13.2 / 12.9.  Past the line: 601 in 65 2.8 / 3.4, 1 350 in 129 4.4 / 4.7, 2 402 in 257
// 7.5 / 7.7, 4 801 in 513 13.3 / 18.1 (a wave reads 16 bytes of a line), 65 533 in 33 3.7 / 21.4 and in 1 021 62 / 334.
bool sum_through_lds(int64_t count, int splits) {
  return splits > 4 * kOrderedDepth && count <= std::min(2048, 5 * splits);
}

__global__ __launch_bounds__(256) void split_sum_tiles_kernel(const float *__restrict__ partial, float *__restrict__ out,
                                                            int64_t count, int splits) {
  constexpr int COLS = 4, DEPTH = 8, ROUND = 256 / COLS * DEPTH;  // splits a round
  __shared__ float tile[2][ROUND][COLS];
  const int tid = threadIdx.x, col = tid % COLS, row = tid / COLS;
  const int64_t i = (int64_t)blockIdx.x * COLS + col;
  const float *p = partial + min(i, count - 1);
  float v[DEPTH], s = 0.f;
  auto fetch = [&](int k0) {
#pragma unroll
    for (int e = 0; e < DEPTH; ++e)
      v[e] = __builtin_nontemporal_load(p + (int64_t)min(k0 + e * (256 / COLS) + row, splits - 1) * count);
  };
  fetch(0);
  int buf = 0;
  for (int k0 = 0; k0 < splits; k0 += ROUND, buf ^= 1) {
#pragma unroll
    for (int e = 0; e < DEPTH; ++e) tile[buf][e * (256 / COLS) + row][col] = v[e];
    if (k0 + ROUND < splits) fetch(k0 + ROUND);
    __syncthreads();  // one a round: the buffer written next was read before the last of them
    if (tid < COLS) {
      const int n = min(ROUND, splits - k0);
      int k = 0;
      if (k0 == 0) s = tile[0][k++][col];
#pragma unroll 16
      for (; k < n; ++k) s += tile[buf][k][col];
    }
  }
  if (tid < COLS && i < count) out[i] = s;
}

template <int BM, int BN, int BK, class AL, class BL>
void launch(const AL &al, const BL &bl, const StoreRowMajor &ep, int K, const Geometry &g, hipStream_t s) {
  hipLaunchKernelGGL((gemm_kernel<BM, BN, BK, AL, BL, StoreRowMajor>), dim3(g.blocks()), dim3(THREADS), 0, s,
                     al, bl, ep, K, g.k_per_split, g.tiles_m, g.tiles_n, g.fold());
}

constexpr int64_t kFlatMinWeights = (1 << 22) + 1;  // elements: more than 16 MiB

// 16-byte loads when both operands allow them (alignment, leading dimension and
// the extent along each operand's contiguous direction multiples of 4)
bool vec_operands(const float *A, bool tA, int lda, const float *B, bool tB, int ldb, int M, int N, int K) {
  return vec4_ok(A, lda, tA ? M : K) && vec4_ok(B, ldb, tB ? K : N);
}

template <int BM, int BN, int BK>
void dispatch(const float *A, bool tA, int lda, uint32_t a_bytes, const float *B, bool tB, int ldb,
              uint32_t b_bytes, const StoreRowMajor &ep, int M, int N, int K, const Geometry &g, hipStream_t s) {
  const FastDiv whole(ONE_SEGMENT);
  if (BM == 32 || vec_operands(A, tA, lda, B, tB, ldb, M, N, K)) {  // the caller takes the 32-row tile only with both
    if (!tA && !tB) {
      Across4<BM, BK> al{A, a_bytes, lda, M, K, whole, 0};
      Along4<BN, BK> bl{B, b_bytes, ldb, N, K, whole, 0};
      launch<BM, BN, BK>(al, bl, ep, K, g, s);
    } else if (tA && !tB) {
      Along4<BM, BK> al{A, a_bytes, lda, M, K, whole, 0};
      Along4<BN, BK> bl{B, b_bytes, ldb, N, K, whole, 0};
      launch<BM, BN, BK>(al, bl, ep, K, g, s);
    } else if (!tA && tB) {
      Across4<BM, BK> al{A, a_bytes, lda, M, K, whole, 0};
      Across4<BN, BK> bl{B, b_bytes, ldb, N, K, whole, 0};
      launch<BM, BN, BK>(al, bl, ep, K, g, s);
    } else {
      Along4<BM, BK> al{A, a_bytes, lda, M, K, whole, 0};
      Across4<BN, BK> bl{B, b_bytes, ldb, N, K, whole, 0};
      launch<BM, BN, BK>(al, bl, ep, K, g, s);
    }
    return;
  }
  if constexpr (BM != 32) {
    if (!tA && !tB) {
      PlainAcross<BM, BK> al{A, a_bytes, lda, M, K};
      PlainAlong<BN, BK> bl{B, b_bytes, ldb, N, K};
      launch<BM, BN, BK>(al, bl, ep, K, g, s);
    } else if (tA && !tB) {
      PlainAlong<BM, BK> al{A, a_bytes, lda, M, K};
      PlainAlong<BN, BK> bl{B, b_bytes, ldb, N, K};
      launch<BM, BN, BK>(al, bl, ep, K, g, s);
    } else if (!tA && tB) {
      PlainAcross<BM, BK> al{A, a_bytes, lda, M, K};
      PlainAcross<BN, BK> bl{B, b_bytes, ldb, N, K};
      launch<BM, BN, BK>(al, bl, ep, K, g, s);
    } else {
      PlainAlong<BM, BK> al{A, a_bytes, lda, M, K};
      PlainAcross<BN, BK> bl{B, b_bytes, ldb, N, K};
      launch<BM, BN, BK>(al, bl, ep, K, g, s);
    }
  }
}

template <int BM, int BN, int BK, bool RAGGED>
void dispatch_split(const float *A, bool tA, int lda, uint32_t a_bytes, const float *B, bool tB, int ldb,
                    uint32_t b_bytes, const StoreRowMajor &ep, int M, int N, int K, const Geometry &g, hipStream_t s) {
  const FastDiv whole(ONE_SEGMENT);
  auto go = [&](const auto &al, const auto &bl) {
    using AL = std::decay_t<decltype(al)>;
    using BL = std::decay_t<decltype(bl)>;
    hipLaunchKernelGGL((split::gemm_kernel<BM, BN, BK, AL, BL, StoreRowMajor>), dim3(g.blocks()), dim3(THREADS), 0, s, al,
                       bl, ep, K, g.k_per_split, g.tiles_m, g.tiles_n, g.fold());
  };
  const split::SplitAcross4<BM, BK, RAGGED> a_across{A, a_bytes, lda, M, K, whole, 0, K};
  const split::SplitAcross4<BN, BK, RAGGED> b_across{B, b_bytes, ldb, N, K, whole, 0, K};
  const split::SplitAlong4<BM, BK> a_along{A, a_bytes, lda, M, K, whole, 0};
  const split::SplitAlong4<BN, BK> b_along{B, b_bytes, ldb, N, K, whole, 0};
  if (!tA && !tB) go(a_across, b_along);
  else if (tA && !tB) go(a_along, b_along);
  else if (!tA && tB) go(a_across, b_across);
  else go(a_along, b_across);
}

}  // namespace

namespace tf {

int launch_split_sum(const float *partial, float *out, int64_t count, int splits, hipStream_t s) {
  const bool vec = count % 4 == 0 && ((reinterpret_cast<uintptr_t>(partial) | reinterpret_cast<uintptr_t>(out)) & 15u) == 0;
  if (vec) {
    const int64_t count4 = count / 4;
    const f32x4 *p4 = reinterpret_cast<const f32x4 *>(partial);
    f32x4 *o4 = reinterpret_cast<f32x4 *>(out);
    // enough lane groups that about 64 K lanes are busy, as long as each group
    // still has a few splits to add
    int sg = 1;
    while (sg < 16 && count4 * sg < 65536 && splits >= 8 * sg) sg *= 4;
    const unsigned blocks = (unsigned)((count4 + 256 / sg - 1) / (256 / sg));
    if (sg == 1) hipLaunchKernelGGL(split_sum_vec_kernel<1>, dim3(blocks), dim3(256), 0, s, p4, o4, count4, splits);
    else if (sg == 4) hipLaunchKernelGGL(split_sum_vec_kernel<4>, dim3(blocks), dim3(256), 0, s, p4, o4, count4, splits);
    else hipLaunchKernelGGL(split_sum_vec_kernel<16>, dim3(blocks), dim3(256), 0, s, p4, o4, count4, splits);
  } else {
    if (sum_through_lds(count, splits))
      hipLaunchKernelGGL(split_sum_tiles_kernel, dim3((unsigned)((count + 3) / 4)), dim3(256), 0, s, partial, out, count,
                         splits);
    else
      hipLaunchKernelGGL(split_sum_ordered_kernel, dim3((unsigned)((count + 63) / 64)), dim3(64), 0, s, partial, out, count,
                         splits);
  }
  return 0;
}

// Number of k-splits that brings `tiles` output tiles up to about two
// workgroups per CU without making a split shorter than `min_k` reduction steps.
int choose_splits(int tiles, int K, int min_k) {
  const int target = 2 * num_cus();
  if (tiles >= target) return 1;
  int splits = (target + tiles - 1) / tiles;
  const int max_splits = K / min_k;
  if (splits > max_splits) splits = max_splits;
  return splits < 1 ? 1 : splits;
}

}  // namespace tf

namespace {

struct Plan {
  int tile, splits;  // square tile that the reduction is planned for, k-splits asked for
  Geometry g;        // of that tile
  bool flat;         // launched on 32 x 128 tiles
  bool split;        // on the split engine (gemm_split.h)
};

// Products of more than 256 rows, columns and reduction steps run on the split engine (1000 x 1537 x 777 and both its
// gradients 117 us on the fp32 engine, 86 here; 4096^3 1000 and 690).  With fewer of one the time is mostly that of
// streaming the largest operand or of the launch (256 x 256 x 12544: 22 against 21 us, 128 x 784 x 256 11.5 against 10).
// A line on sizes, no more: it keeps the rounding of classifiers under a batch-norm head (see may_use_split in conv.hip) as
// long as the batch or a layer's width is at most 256.  TINYFLOW_SPLIT=0 / 1 forces the fp32 / the split engine.
bool product_on_split(int M, int N, int K) {
  const char *e = getenv("TINYFLOW_SPLIT");
  if (e && *e) return atoi(e) != 0;
  return M > 256 && N > 256 && K > 256;
}
constexpr int split_stage(int tile) { return tile == 128 ? 16 : 32; }

// Two 64 x 64 tiles of at most 32 rows side by side are one 32 x 128 tile, with as many floats to fold.  Every
// output element keeps the pieces of the reduction that it has on the 64 x 64 tiles and the order in which they
// are summed, so the tile does not show in the bits of the result.
void to_flat_tiles(Geometry &g, int N) {
  g.tiles_n = cdiv(N, 128);
  g.fold_first_tile /= 2;
}

Plan plan_product(int M, int N, int K, bool vec) {
  Plan p;
  p.split = product_on_split(M, N, K);
  if (p.split) {
    SplitTraffic t;
    t.in_bytes = 4.0 * ((double)M * K + (double)K * N);
    t.out_bytes = 4.0 * (double)M * N;
    double best = 1e30;
    for (int tile : {128, 64}) {
      if (tile == 128 && (M <= 64 || N <= 64)) continue;
      for (int splits : {1, 2, 3, 4, 6, 8, 12, 16}) {
        if (splits > 1 && K / splits < 64) break;
        const double us = predict_split_us(M, N, K, tile, tile, splits, split_stage(tile), t);
        if (us < best) {
          best = us;
          p.tile = tile;
          p.splits = splits;
        }
      }
    }
    p.g = make_geometry(M, N, K, p.tile, p.tile, p.splits, split_stage(p.tile));
    plan_fold(p.g, K, split_stage(p.tile), 1);
    p.flat = false;
    return p;
  }
  p.tile = M > 64 && N > 64 && cdiv(M, 128) * cdiv(N, 128) >= num_cus() ? 128 : 64;
  p.splits = choose_splits(cdiv(M, p.tile) * cdiv(N, p.tile), K, 256);
  p.g = make_geometry(M, N, K, p.tile, p.tile, p.splits);
  plan_fold(p.g, K, p.tile == 128 ? 16 : 32, 1);
  // At most 32 rows: a tile of one MFMA's height.  On the 64-row tile half of the matrix instructions work on
  // padding, which for weights that come from memory costs as much as reading them.  64-row against 32-row tile, us:
  // 32 x 25088 x 4096 124 / 92 (4.5 TB/s), 32 x 4096 x 25088 with transposed weights 143 / 98, 6 x 4608 x 4096
  // 27 / 20, 6 x 3200 x 2048 16.2 / 12.5; but 32 x 2048 x 2048, 2^22 weights, 11.7 / 12.0, and smaller ones likewise:
  // their time is the launch's and the sum of the splits.
  p.flat = M <= 32 && vec && (int64_t)N * K >= kFlatMinWeights && p.g.fold_first_tile % 2 == 0;
  return p;
}

}  // namespace

extern "C" int DLGpuMatrixMultiplyDescribe(int M, int N, int K, bool vec, int *tile_rows, int *tile_cols, int *pieces,
                                           int *first_folded_tile) {
  TF_REQUIRE(M > 0 && N > 0 && K > 0 && tile_rows && tile_cols && pieces && first_folded_tile, "bad arguments");
  Plan p = plan_product(M, N, K, vec);
  if (p.flat) to_flat_tiles(p.g, N);
  *tile_rows = p.flat ? 32 : p.tile;
  *tile_cols = p.flat ? 128 : p.tile;
  *pieces = p.g.fold_pieces > 1 ? p.g.fold_pieces : p.g.splits;
  *first_folded_tile = p.g.fold_pieces > 1 ? p.g.fold_first_tile : -1;
  return 0;
}

extern "C" int DLGpuMatrixMultiply(const DLArrayHandle matA, bool transposeA, const DLArrayHandle matB,
                                   bool transposeB, DLArrayHandle matC, void **handle, void **stream) {
  announce_write(matC);
  (void)handle;
  TF_REQUIRE(on_gpu(matA) && on_gpu(matB) && on_gpu(matC), "arrays must live on the GPU");
  TF_REQUIRE(matA->ndim == 2 && matB->ndim == 2 && matC->ndim == 2, "operands must be 2-D");
  const int64_t M = matA->shape[transposeA ? 1 : 0], K = matA->shape[transposeA ? 0 : 1];
  const int64_t Kb = matB->shape[transposeB ? 1 : 0], N = matB->shape[transposeB ? 0 : 1];
  TF_REQUIRE(K == Kb, "inner dimensions differ (%lld vs %lld)", (long long)K, (long long)Kb);
  TF_REQUIRE(matC->shape[0] == M && matC->shape[1] == N, "output must be %lld x %lld", (long long)M,
             (long long)N);
  const int64_t a_bytes = numel(matA) * 4, b_bytes = numel(matB) * 4;
  TF_REQUIRE(a_bytes < (1ll << 31) && b_bytes < (1ll << 31) && M * N * 4 < (1ll << 31),
             "operands and results of 2 GiB or more are not supported");
  // the epilogue forms 32-bit byte offsets for every row of a tile, including the rows
  // of the last tile that lie past M (the buffer bound drops them only if the offset
  // has not wrapped)
  TF_REQUIRE((M + 128) * N * 4 < (1ll << 32), "result too wide: (rows + 128) * columns * 4 must stay below 4 GiB");
  hipStream_t s = stream_of(stream);
  if (M == 0 || N == 0) return 0;
  if (K == 0) return DLGpuArraySet(matC, 0.f, stream);

  const int lda = (int)matA->shape[1], ldb = (int)matB->shape[1];
  const Plan plan = plan_product((int)M, (int)N, (int)K,
                                 vec_operands((const float *)matA->data, transposeA, lda, (const float *)matB->data,
                                              transposeB, ldb, (int)M, (int)N, (int)K));
  Geometry g = plan.g;
  FoldBuffers fb;
  if (acquire_fold(g, plan.tile, plan.tile, 1, s, fb) != 0) {  // no scratch (this entry point cannot report it): no fold
    release_fold(fb);
    g = make_geometry((int)M, (int)N, (int)K, plan.tile, plan.tile, plan.splits, plan.split ? split_stage(plan.tile) : 32);
  }

  float *dst = (float *)matC->data;
  float *partial = nullptr;
  if (g.splits > 1) {
    partial = (float *)device_alloc((size_t)g.splits * M * N * sizeof(float), s);
    if (!partial) {  // no scratch: fall back to one pass over the whole reduction
      g = make_geometry((int)M, (int)N, (int)K, plan.tile, plan.tile, 1);
    } else {
      dst = partial;
    }
  }
  if (plan.flat) to_flat_tiles(g, (int)N);
  StoreRowMajor ep{dst, (int)N, (int)M, (int)N, M * N};
  if (plan.split) {
    auto run = [&](auto tile, auto ragged) {
      constexpr int T = decltype(tile)::value;
      dispatch_split<T, T, split_stage(T), decltype(ragged)::value>(
          (const float *)matA->data, transposeA, lda, (uint32_t)a_bytes, (const float *)matB->data, transposeB, ldb,
          (uint32_t)b_bytes, ep, (int)M, (int)N, (int)K, g, s);
    };
    const bool ragged = K % 4 != 0;  // the last vector along the reduction holds other elements behind it
    if (plan.tile == 128 && ragged) run(IC<128>{}, std::true_type{});
    else if (plan.tile == 128) run(IC<128>{}, std::false_type{});
    else if (ragged) run(IC<64>{}, std::true_type{});
    else run(IC<64>{}, std::false_type{});
  } else if (plan.tile == 128)
    dispatch<128, 128, 16>((const float *)matA->data, transposeA, lda, (uint32_t)a_bytes, (const float *)matB->data,
                       transposeB, ldb, (uint32_t)b_bytes, ep, (int)M, (int)N, (int)K, g, s);
  else if (plan.flat)
    dispatch<32, 128, 32>((const float *)matA->data, transposeA, lda, (uint32_t)a_bytes, (const float *)matB->data,
                          transposeB, ldb, (uint32_t)b_bytes, ep, (int)M, (int)N, (int)K, g, s);
  else
    dispatch<64, 64, 32>((const float *)matA->data, transposeA, lda, (uint32_t)a_bytes, (const float *)matB->data,
                     transposeB, ldb, (uint32_t)b_bytes, ep, (int)M, (int)N, (int)K, g, s);
  if (partial) {
    launch_split_sum(partial, (float *)matC->data, M * N, g.splits, s);
    device_free(partial, s);
  }
  release_fold(fb);
  return finish(s, "DLGpuMatrixMultiply");
}
