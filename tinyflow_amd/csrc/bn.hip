// Batch normalisation forward (training) and backward with gamma = 1, beta = 0,
// eps = 1e-5 and biased variance -- the only configuration the reference uses
// (src/gpu_op.cu:4224-4458: scale/bias are rebuilt as ones/zeros on every call,
// the scale/bias gradients cuDNN returns are discarded, there are no running
// statistics).
//
// per-activation mode (what every reference model graph passes): one statistic
//   per (c,h,w) position over the batch.  x is an [N, L] matrix, L = C*H*W; a lane
//   owns one column, keeps its N values in registers, and the whole op is a
//   single pass: forward reads x and writes y (8 B/element), backward reads x, dy
//   and writes dx (12 B/element).  Lanes of a wave read 64 consecutive columns,
//   so every access is a full 256-byte line.
// spatial mode: one statistic per channel over (N,H,W).  Per-(channel, image-chunk)
//   partial sums (fp32 per lane, fp64 across lanes and chunks), and a streaming
//   normalise pass over the flat tensor (12 B/element forward, 20 backward).  The chunks
//   of a channel are folded in a fixed order, by the workgroups of the second pass
//   themselves or, where that costs more than a launch, by a small kernel in between.
//   A channel that fits a workgroup's registers needs no second pass (8 B/element forward,
//   12 backward), and its ReLU joins it there.
//
// Saved statistics protocol (as the reference): forward allocates mean and
// inverse-std buffers and publishes them through *mean_p / *Variance_p; backward
// consumes and releases them.
#include "gemm_core.h"
#include "internal.h"

#include <algorithm>
#include <type_traits>

using namespace tf;
using tf::gemm::FastDiv;

namespace {

constexpr int kThreads = 256;
constexpr float kEps = 1e-5f;
constexpr int kNonTemporal = 2;  // cache-policy operand of a buffer access: a stream that is read once
typedef float f32x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- per-activation

// NREG >= N values of one column live in registers.  The three tensors are addressed
// through buffer descriptors: one per-lane column offset (a VGPR computed once) plus a
// uniform row offset (a scalar) per access, instead of a 64-bit vector address per
// access -- the address arithmetic was more than half of the kernel's instructions and
// cost as many registers as a quarter of the data.  A descriptor covers exactly the N
// rows, so rows N..NREG-1 read as zero and their stores are dropped by the bounds
// check: no per-row branch.  Needs NREG * L * 4 < 2^32 (the row offsets are 32-bit).
// RELU: y = max(bn(x), 0) in the same pass (the fused entry points below).
// BOTH: also bn(x) itself, to `plain`: 12 bytes per element where batch norm and ReLU apart move 16.
// FULL: N == NREG, no row needs masking in the variance.
template <int NREG, bool RELU, bool BOTH, bool FULL>
__global__ __launch_bounds__(kThreads) void bn_pa_forward_kernel(const float *__restrict__ x,
                                                                float *__restrict__ y, float *__restrict__ plain,
                                                                float *__restrict__ save_mean,
                                                                float *__restrict__ save_istd, int N, uint32_t L) {
  const uint32_t l = blockIdx.x * kThreads + threadIdx.x;
  if (l >= L) return;
  const uint32_t col = l * 4u, row = L * 4u;
  const __amdgpu_buffer_rsrc_t rx = gemm::make_rsrc(x, (uint32_t)N * row), ry = gemm::make_rsrc(y, (uint32_t)N * row);
  const __amdgpu_buffer_rsrc_t rp = BOTH ? gemm::make_rsrc(plain, (uint32_t)N * row) : ry;
  float v[NREG];
#pragma unroll
  for (int n = 0; n < NREG; ++n)
    v[n] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, (int)col, (int)(n * row), kNonTemporal));
  float s = 0.f;
#pragma unroll
  for (int n = 0; n < NREG; ++n) s += v[n];
  const float mean = s / (float)N;
  float q = 0.f;
#pragma unroll
  for (int n = 0; n < NREG; ++n) {
    const float dlt = (FULL || n < N) ? v[n] - mean : 0.f;
    q += dlt * dlt;
  }
  const float istd = 1.0f / sqrtf(q / (float)N + kEps);
  save_mean[l] = mean;
  save_istd[l] = istd;
#pragma unroll
  for (int n = 0; n < NREG; ++n) {
    const float out = (v[n] - mean) * istd;
    if (BOTH) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, out), rp, (int)col, (int)(n * row), 0);
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, (RELU && out < 0.f) ? 0.f : out), ry, (int)col,
                                          (int)(n * row), 0);
  }
}

// One lane per column, three sweeps over it, for few rows of more columns than the register kernels address: lanes
// enough and no chain worth mentioning, so nothing but the bytes counts, where a tile of 64 rows would be mostly
// padding.  67 M columns of 2 rows 578 us against 1926 in tiles, 34 M of 8 rows 950 against 1177; 16 rows 1947
// against 1643, and the tiles are faster from there on.
constexpr int kFewRows = 12;

template <bool RELU>
__global__ __launch_bounds__(kThreads) void bn_pa_forward_stream_kernel(const float *__restrict__ x,
                                                                       float *__restrict__ y,
                                                                       float *__restrict__ save_mean,
                                                                       float *__restrict__ save_istd, int N,
                                                                       int64_t L) {
  const int64_t l = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (l >= L) return;
  float s = 0.f;
  for (int n = 0; n < N; ++n) s += x[(int64_t)n * L + l];
  const float mean = s / (float)N;
  float q = 0.f;
  for (int n = 0; n < N; ++n) {
    const float dlt = x[(int64_t)n * L + l] - mean;
    q += dlt * dlt;
  }
  const float istd = 1.0f / sqrtf(q / (float)N + kEps);
  save_mean[l] = mean;
  save_istd[l] = istd;
  for (int n = 0; n < N; ++n) {
    const float out = (x[(int64_t)n * L + l] - mean) * istd;
    y[(int64_t)n * L + l] = (RELU && out < 0.f) ? 0.f : out;
  }
}

// More rows than registers: a workgroup owns COLS columns and walks them three times (the second
// and third walk hit the cache) in tiles of 4096 elements.  All lanes fetch a tile and put it into
// LDS, then lane c adds column c from there in row order while the fetch of the next tile is in
// flight.  What bounds a narrow tensor is the chain of additions in a column, and the order stays
// that chain's; taken straight from memory, each link waited for a load: the ten logits of a
// batch of 1000 took 290 us forward and 250 us backward, now 29 and 27.  Rows past N enter the sums as +0, which
// changes none.
// COLS is 64 (a 256-byte line per row) where that gives every CU two workgroups, else 16.  16 against 64 columns, us,
// forward and backward: 130 rows of 4096 columns 8 / 13 and 7 / 11, of 16384 9.9 / 13.7 and 12.5 / 11.2, of 33000
// 27 / 23 and 35 / 25; 1000 rows of 16384 77 / 115 and 92 / 107, of 33000 182 / 156 and 236 / 223.
constexpr int kTile = 4096, kTileRegs = kTile / kThreads;
constexpr int kWideCols = 64, kNarrowCols = 16;

// Calls fetch(row) -> T for the lane's elements of every tile, then add(T) in lane c < COLS for
// every row of column c in row order.
template <int COLS, class T, class Fetch, class Add>
__device__ inline void walk_column(T (*tile)[COLS], int N, const Fetch &fetch, const Add &add) {
  constexpr int ROWS = kTile / COLS, STEP = kThreads / COLS;
  const int col = threadIdx.x % COLS, r0 = threadIdx.x / COLS;
  T v[kTileRegs];
#pragma unroll
  for (int e = 0; e < kTileRegs; ++e) v[e] = fetch(r0 + e * STEP);
  for (int n0 = 0; n0 < N; n0 += ROWS) {
#pragma unroll
    for (int e = 0; e < kTileRegs; ++e) tile[r0 + e * STEP][col] = v[e];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kTileRegs; ++e) v[e] = fetch(n0 + ROWS + r0 + e * STEP);
    if (threadIdx.x < COLS) {
#pragma unroll 16
      for (int r = 0; r < ROWS; ++r) add(tile[r][col]);
    }
    __syncthreads();
  }
}

template <int COLS, bool RELU>
__global__ __launch_bounds__(kThreads) void bn_pa_forward_tiles_kernel(const float *__restrict__ x,
                                                                      float *__restrict__ y,
                                                                      float *__restrict__ save_mean,
                                                                      float *__restrict__ save_istd, int N,
                                                                      int64_t L) {
  __shared__ float tile[kTile / COLS][COLS];
  __shared__ float stat[COLS];
  const int col = threadIdx.x % COLS;
  const int64_t l = (int64_t)blockIdx.x * COLS + col;
  const int rows = l < L ? N : 0;  // a lane beyond L fetches and writes nothing but meets every barrier
  float s = 0.f;
  walk_column<COLS>(tile, N, [&](int n) { return n < rows ? x[(int64_t)n * L + l] : 0.f; }, [&](float v) { s += v; });
  if (threadIdx.x < COLS) stat[col] = s / (float)N;
  __syncthreads();
  const float mean = stat[col];
  float q = 0.f;
  walk_column<COLS>(tile, N, [&](int n) { return n < rows ? x[(int64_t)n * L + l] - mean : 0.f; },
                    [&](float dlt) { q += dlt * dlt; });
  // every lane has read the mean before the walk's first barrier
  if (threadIdx.x < COLS) {
    stat[col] = 1.0f / sqrtf(q / (float)N + kEps);
    if (l < L) {
      save_mean[l] = mean;
      save_istd[l] = stat[col];
    }
  }
  __syncthreads();
  const float istd = stat[col];
#pragma unroll 4
  for (int n = threadIdx.x / COLS; n < rows; n += kThreads / COLS) {
    const float out = (x[(int64_t)n * L + l] - mean) * istd;
    y[(int64_t)n * L + l] = (RELU && out < 0.f) ? 0.f : out;
  }
}

// dx = istd/N * (N*dy - sum(dy) - xhat * sum(dy*xhat))
// RELU: dy is first masked with bn(x) > 0, i.e. the gradient of max(bn(x), 0).
// BOTH: the masked dy goes to `masked` as well: 16 bytes per element where the two gradients apart move 20.
// Addressing as in the forward kernel; a row beyond N reads dy = 0 and adds nothing.
template <int NREG, bool RELU, bool BOTH>
__global__ __launch_bounds__(kThreads) void bn_pa_backward_kernel(const float *__restrict__ x,
                                                                 const float *__restrict__ dy,
                                                                 float *__restrict__ dx, float *__restrict__ masked,
                                                                 const float *__restrict__ save_mean,
                                                                 const float *__restrict__ save_istd, int N,
                                                                 uint32_t L) {
  const uint32_t l = blockIdx.x * kThreads + threadIdx.x;
  if (l >= L) return;
  const uint32_t col = l * 4u, row = L * 4u, all = (uint32_t)N * row;
  const __amdgpu_buffer_rsrc_t rx = gemm::make_rsrc(x, all), rg = gemm::make_rsrc(dy, all),
                               ro = gemm::make_rsrc(dx, all), rm = BOTH ? gemm::make_rsrc(masked, all) : ro;
  const float mean = save_mean[l], istd = save_istd[l];
  float xh[NREG], g[NREG];
#pragma unroll
  for (int n = 0; n < NREG; ++n) {
    xh[n] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, (int)col, (int)(n * row), kNonTemporal));
    g[n] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rg, (int)col, (int)(n * row), kNonTemporal));
  }
  float s1 = 0.f, s2 = 0.f;
#pragma unroll
  for (int n = 0; n < NREG; ++n) {
    xh[n] = (xh[n] - mean) * istd;
    if (RELU) g[n] = xh[n] > 0.f ? g[n] : 0.f;
    if (BOTH) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, g[n]), rm, (int)col, (int)(n * row), 0);
    s1 += g[n];
    s2 += g[n] * xh[n];
  }
  const float m = (float)N;
  const float scale = istd / m;
#pragma unroll
  for (int n = 0; n < NREG; ++n)
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, scale * (m * g[n] - s1 - xh[n] * s2)), ro, (int)col,
                                          (int)(n * row), 0);
}

// One lane per column, as in forward; it walks the column twice.  From six workgroups per CU on the lanes hide the
// loads' latency, and the tiles' detour over LDS and its barriers cost more than they give.  This against tiles, us:
// 130 rows of 262144 columns 171 / 144, of 393216 182 / 212, of 524288 237 / 289; 300 rows 383 / 321, 466 / 474 and
// 562 / 682.
template <bool RELU>
__global__ __launch_bounds__(kThreads) void bn_pa_backward_stream_kernel(const float *__restrict__ x,
                                                                        const float *__restrict__ dy,
                                                                        float *__restrict__ dx,
                                                                        const float *__restrict__ save_mean,
                                                                        const float *__restrict__ save_istd,
                                                                        int N, int64_t L) {
  const int64_t l = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (l >= L) return;
  const float mean = save_mean[l], istd = save_istd[l];
  float s1 = 0.f, s2 = 0.f;
  for (int n = 0; n < N; ++n) {
    const float xh = (x[(int64_t)n * L + l] - mean) * istd;
    float g = dy[(int64_t)n * L + l];
    if (RELU) g = xh > 0.f ? g : 0.f;
    s1 += g;
    s2 += g * xh;
  }
  const float m = (float)N;
  const float scale = istd / m;
  for (int n = 0; n < N; ++n) {
    const float xh = (x[(int64_t)n * L + l] - mean) * istd;
    float g = dy[(int64_t)n * L + l];
    if (RELU) g = xh > 0.f ? g : 0.f;
    dx[(int64_t)n * L + l] = scale * (m * g - s1 - xh * s2);
  }
}

struct GradPair {
  float g, xh;
};

template <int COLS, bool RELU>
__global__ __launch_bounds__(kThreads) void bn_pa_backward_tiles_kernel(const float *__restrict__ x,
                                                                       const float *__restrict__ dy,
                                                                       float *__restrict__ dx,
                                                                       const float *__restrict__ save_mean,
                                                                       const float *__restrict__ save_istd,
                                                                       int N, int64_t L) {
  __shared__ GradPair tile[kTile / COLS][COLS];
  __shared__ float sums[2][COLS];
  const int col = threadIdx.x % COLS;
  const int64_t l = (int64_t)blockIdx.x * COLS + col;
  const int rows = l < L ? N : 0;
  const float mean = l < L ? save_mean[l] : 0.f, istd = l < L ? save_istd[l] : 0.f;
  auto fetch = [&](int n) {
    if (n >= rows) return GradPair{0.f, 0.f};
    const float xh = (x[(int64_t)n * L + l] - mean) * istd;
    const float g = dy[(int64_t)n * L + l];
    return GradPair{RELU && !(xh > 0.f) ? 0.f : g, xh};
  };
  float s1 = 0.f, s2 = 0.f;
  walk_column<COLS>(tile, N, fetch, [&](GradPair p) {
    s1 += p.g;
    s2 += p.g * p.xh;
  });
  if (threadIdx.x < COLS) {
    sums[0][col] = s1;
    sums[1][col] = s2;
  }
  __syncthreads();
  s1 = sums[0][col];
  s2 = sums[1][col];
  const float m = (float)N;
  const float scale = istd / m;
#pragma unroll 4
  for (int n = threadIdx.x / COLS; n < rows; n += kThreads / COLS) {
    const GradPair p = fetch(n);
    dx[(int64_t)n * L + l] = scale * (m * p.g - s1 - p.xh * s2);
  }
}

// Whether one lane per column gives every CU six workgroups.
bool many_columns(int64_t L) { return L >= (int64_t)num_cus() * kThreads * 6; }

// Whether COLS = kWideCols gives every CU two workgroups.
bool wide_column_blocks(int64_t L) { return L >= (int64_t)num_cus() * kWideCols * 2; }

template <bool RELU>
void bn_pa_forward_tiles(hipStream_t s, const float *x, float *y, float *mean, float *istd, int N, int64_t L) {
  if (wide_column_blocks(L))
    hipLaunchKernelGGL((bn_pa_forward_tiles_kernel<kWideCols, RELU>), dim3(cdiv(L, kWideCols)), dim3(kThreads), 0, s,
                       x, y, mean, istd, N, L);
  else
    hipLaunchKernelGGL((bn_pa_forward_tiles_kernel<kNarrowCols, RELU>), dim3(cdiv(L, kNarrowCols)), dim3(kThreads), 0,
                       s, x, y, mean, istd, N, L);
}

template <bool RELU>
void bn_pa_backward_tiles(hipStream_t s, const float *x, const float *dy, float *dx, const float *mean, const float *istd,
                         int N, int64_t L) {
  if (wide_column_blocks(L))
    hipLaunchKernelGGL((bn_pa_backward_tiles_kernel<kWideCols, RELU>), dim3(cdiv(L, kWideCols)), dim3(kThreads), 0, s,
                       x, dy, dx, mean, istd, N, L);
  else
    hipLaunchKernelGGL((bn_pa_backward_tiles_kernel<kNarrowCols, RELU>), dim3(cdiv(L, kNarrowCols)), dim3(kThreads), 0,
                       s, x, dy, dx, mean, istd, N, L);
}

// ------------------------------------------------------------------------ spatial

__device__ inline double lane_value(double v, int lane) {
  const int2 h = __builtin_bit_cast(int2, v);
  return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_readlane(h.x, lane), __builtin_amdgcn_readlane(h.y, lane)));
}
// Adds the value of the lane OFF further on, of the same sixteen (zero past them).
template <int OFF>
__device__ inline double add_row_lane(double v) {
  constexpr int kRowShiftLeft = 0x100;
  const int2 h = __builtin_bit_cast(int2, v);
  return v + __builtin_bit_cast(double, make_int2(__builtin_amdgcn_mov_dpp(h.x, kRowShiftLeft + OFF, 0xf, 0xf, true),
                                                  __builtin_amdgcn_mov_dpp(h.y, kRowShiftLeft + OFF, 0xf, 0xf, true)));
}
// Sum over a wave, valid in lane 0.  The steps inside a row of lanes stay off the LDS, which sixteen waves share.
__device__ inline double wave_sum_d(double v) {
  v += __shfl_down(v, 32, 64);
  v += __shfl_down(v, 16, 64);
  v = add_row_lane<8>(v);
  v = add_row_lane<4>(v);
  v = add_row_lane<2>(v);
  return add_row_lane<1>(v);
}

// Sum of a pair over the 256 lanes of a block, valid in thread 0.
__device__ inline void block_sum2(double &a, double &b, double (*smem)[2]) {
  a = wave_sum_d(a);
  b = wave_sum_d(b);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    smem[wave][0] = a;
    smem[wave][1] = b;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    a = (smem[0][0] + smem[1][0]) + (smem[2][0] + smem[3][0]);
    b = (smem[0][1] + smem[1][1]) + (smem[2][1] + smem[3][1]);
  }
}

// One unit of the spatial kernels: a 16-byte vector (feature maps whose size is a
// multiple of 4) or a single float.
template <bool VEC>
struct Unit;
template <>
struct Unit<true> {
  static constexpr int W = 4;
  static __device__ inline void load(const float *p, float (&v)[4]) {
    const f32x4 t = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(p));
    v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
  }
  static __device__ inline void store(float *p, const float (&v)[4]) {
    const f32x4 t = {v[0], v[1], v[2], v[3]};
    *reinterpret_cast<f32x4 *>(p) = t;
  }
};
template <>
struct Unit<false> {
  static constexpr int W = 1;
  static __device__ inline void load(const float *p, float (&v)[1]) { v[0] = *p; }
  static __device__ inline void store(float *p, const float (&v)[1]) { *p = v[0]; }
};

// x viewed as [N, C, HW]; block (c, chunk) sums images [chunk*ipc, ...) of channel c.
// FWD: partial = (sum (x - p), sum (x - p)^2) with the pivot p = the channel's first
// element (image 0, pixel 0): sums of shifted values lose nothing to cancellation
// when |mean| is much larger than the standard deviation, where sum x^2 - m*mean^2
// in fp32 would.  BWD: partial = (sum dy, sum dy*xhat).
// The (image, pixel) pairs of a chunk are walked as one flat index so that small
// feature maps (7x7) keep all lanes busy; VEC: 16-byte loads when HW is a multiple
// of 4.  Lanes accumulate in fp32 (a few hundred terms each), the block and the
// chunks are combined in fp64.  The fused steps are explicit, as in bn_sp_one_kernel, which has the same bits.
template <bool BWD, bool VEC>
__global__ __launch_bounds__(kThreads) void bn_sp_partial_kernel(const float *__restrict__ x,
                                                                const float *__restrict__ dy,
                                                                const float *__restrict__ save_mean,
                                                                const float *__restrict__ save_istd,
                                                                double *__restrict__ partial,
                                                                float *__restrict__ pivots, int N, int C, int HW,
                                                                int images_per_chunk, FastDiv div_row) {
  __shared__ double smem[4][2];
  const int c = blockIdx.x;
  const int n0 = blockIdx.y * images_per_chunk;
  int n1 = n0 + images_per_chunk;
  if (n1 > N) n1 = N;
  const float mean = BWD ? save_mean[c] : 0.f, istd = BWD ? save_istd[c] : 0.f;
  const float pivot = BWD ? 0.f : x[(int64_t)c * HW];
  constexpr int W = Unit<VEC>::W;
  const uint32_t row_units = (uint32_t)HW / W;                 // div_row divides by this
  const uint32_t total = (uint32_t)(n1 - n0) * row_units;
  float a0 = 0.f, b0 = 0.f;
  for (uint32_t idx = threadIdx.x; idx < total; idx += kThreads) {
    uint32_t img, unit;
    div_row.divmod(idx, img, unit);
    const int64_t at = ((int64_t)(n0 + (int)img) * C + c) * HW + (int64_t)unit * W;
    float xv[W], gv[W] = {};
    Unit<VEC>::load(x + at, xv);
    if (BWD) Unit<VEC>::load(dy + at, gv);
#pragma unroll
    for (int k = 0; k < W; ++k) {
      if (BWD) {
        a0 += gv[k];
        b0 = __builtin_fmaf(gv[k], (xv[k] - mean) * istd, b0);
      } else {
        const float t = xv[k] - pivot;
        a0 += t;
        b0 = __builtin_fmaf(t, t, b0);
      }
    }
  }
  double a = (double)a0, b = (double)b0;
  block_sum2(a, b, smem);
  if (threadIdx.x == 0) {
    partial[((int64_t)blockIdx.y * C + c) * 2 + 0] = a;
    partial[((int64_t)blockIdx.y * C + c) * 2 + 1] = b;
    if (!BWD && blockIdx.y == 0) pivots[c] = pivot;  // for the apply pass, which may overwrite x
  }
}

// What the apply pass needs of a channel, from the sums of its chunk partials: forward (mean,
// 1/sqrt(var + eps)), which are also the saved statistics; backward (sum dy, sum dy*xhat).
template <bool BWD>
__device__ inline void channel_floats(double s, double q, double m, float pivot, float &f0, float &f1) {
  f0 = (float)s;
  f1 = (float)q;
  if (BWD) return;
  const double shifted_mean = s / m;  // mean of x - pivot; the variance does not depend on the pivot
  double var = q / m - shifted_mean * shifted_mean;
  if (var < 0.0) var = 0.0;
  f0 = (float)((double)pivot + shifted_mean);
  f1 = (float)(1.0 / sqrt(var + (double)kEps));
}

// Folds the chunk partials of every channel, in chunk order.  A workgroup takes CH channels; all lanes fetch, 256 / CH
// chunks of a channel at a time, so that the chain of additions runs out of LDS:
// 1024 chunks of one channel took 77 us with a lane per channel that reads them from memory, and take 4 so.
template <bool BWD>
__global__ __launch_bounds__(kThreads) void bn_sp_finish_kernel(const double *__restrict__ partial,
                                                               const float *__restrict__ pivots,
                                                               float *__restrict__ out0, float *__restrict__ out1,
                                                               int C, int chunks, double m, int log_ch) {
  __shared__ double part[2][kThreads];
  const int tid = threadIdx.x, ch = 1 << log_ch, depth = kThreads >> log_ch;
  const int local = tid & (ch - 1), c = blockIdx.x * ch + local;
  const int sums_of = tid >> log_ch;  // 0: first sum of the pair, 1: second, beyond: fetches only
  double sum = 0.0;
  for (int k0 = 0; k0 < chunks; k0 += depth) {
    const int n = min(depth, chunks - k0);
    if ((tid >> log_ch) < n && c < C) {
      const double *p = partial + ((int64_t)(k0 + (tid >> log_ch)) * C + c) * 2;
      part[0][tid] = p[0];
      part[1][tid] = p[1];
    }
    __syncthreads();
    if (sums_of < 2 && c < C) {
#pragma unroll 8
      for (int k = 0; k < n; ++k) sum += part[sums_of][(k << log_ch) + local];
    }
    __syncthreads();
  }
  if (sums_of < 2) part[sums_of][local] = sum;
  __syncthreads();
  if (sums_of == 0 && c < C) channel_floats<BWD>(part[0][local], part[1][local], m, BWD ? 0.f : pivots[c], out0[c], out1[c]);
}

// Channels per workgroup of the kernel above, as a power of two: as many as leave lanes for all chunks of each.
int finish_log_channels(int chunks) {
  int log_ch = 6;  // at least four lanes per channel
  while (log_ch > 0 && (kThreads >> log_ch) < chunks) --log_ch;
  return log_ch;
}

// Apply pass over the flat tensor, one contiguous run of 1024 units (16 KiB when
// VEC) per workgroup as in the elementwise engine; a unit (float4 or float) lies
// inside one (image, channel) row, whose channel is (unit / units per row) % C.
// FOLD: each workgroup first folds, in chunk order, the chunk partials of the channels of its
// rows: a few KB from the L2 while its elements are on their way (fold_in_apply says when).
// Else p0, p1 hold what bn_sp_finish_kernel made of them.
// FWD: y = (x - mean) * istd; with FOLD also the saved statistics, by the workgroup that holds the
// first unit of the channel's row in image 0.  BWD: dx = istd/m * (m*dy - s1 - xhat*s2).
template <bool BWD, bool VEC, bool FOLD>
__global__ __launch_bounds__(kThreads) void bn_sp_apply_kernel(const float *__restrict__ x,
                                                              const float *__restrict__ dy,
                                                              float *__restrict__ out,
                                                              const double *__restrict__ partial,
                                                              const float *__restrict__ pivot, int chunks, double m,
                                                              const float *__restrict__ p0,
                                                              const float *__restrict__ p1,
                                                              float *__restrict__ save_mean,
                                                              float *__restrict__ save_istd, FastDiv div_row,
                                                              FastDiv div_c, uint32_t units) {
  constexpr int W = Unit<VEC>::W;
  constexpr int kUnroll = 4;
  __shared__ float fold[2][FOLD ? kThreads * kUnroll : 1];  // per row: FWD mean, istd; BWD sum dy, sum dy*xhat
  const uint32_t first = blockIdx.x * (kThreads * kUnroll), base = first + threadIdx.x;
  float xv[kUnroll][W], gv[kUnroll][W];
  uint32_t row_of[kUnroll], ch[kUnroll];
#pragma unroll
  for (int u = 0; u < kUnroll; ++u) {
    const uint32_t unit = min(base + u * kThreads, units - 1u);  // no branch between the loads
    uint32_t img;
    row_of[u] = div_row.div(unit);
    div_c.divmod(row_of[u], img, ch[u]);
    Unit<VEC>::load(x + (int64_t)unit * W, xv[u]);
    if (BWD) Unit<VEC>::load(dy + (int64_t)unit * W, gv[u]);
  }
  const uint32_t first_row = div_row.div(first);
  if (FOLD) {
    const uint32_t last_row = div_row.div(min(first + kThreads * kUnroll, units) - 1u);
    for (uint32_t row = first_row + threadIdx.x; row <= last_row; row += kThreads) {
      uint32_t img, c;
      div_c.divmod(row, img, c);
      double s = 0.0, q = 0.0;
#pragma unroll 4
      for (int k = 0; k < chunks; ++k) {
        s += partial[((int64_t)k * div_c.d + c) * 2 + 0];
        q += partial[((int64_t)k * div_c.d + c) * 2 + 1];
      }
      float f0, f1;
      channel_floats<BWD>(s, q, m, BWD ? 0.f : pivot[c], f0, f1);
      if (!BWD && img == 0 && row * div_row.d >= first) {
        save_mean[c] = f0;
        save_istd[c] = f1;
      }
      fold[0][row - first_row] = f0;
      fold[1][row - first_row] = f1;
    }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < kUnroll; ++u) {
    const uint32_t unit = base + u * kThreads;
    if (unit >= units) continue;
    const uint32_t c = ch[u];
    const float f0 = FOLD ? fold[0][row_of[u] - first_row] : p0[c];
    const float f1 = FOLD ? fold[1][row_of[u] - first_row] : p1[c];
    float r[W];
    if (BWD) {
      const float mean = save_mean[c], istd = save_istd[c];
      const float scale = istd / (float)m;
#pragma unroll
      for (int k = 0; k < W; ++k) {
        const float xh = (xv[u][k] - mean) * istd;
        r[k] = scale * ((float)m * gv[u][k] - f0 - xh * f1);
      }
    } else {
#pragma unroll
      for (int k = 0; k < W; ++k) r[k] = (xv[u][k] - f0) * f1;
    }
    Unit<VEC>::store(out + (int64_t)unit * W, r);
  }
}

// Both passes in one launch where a workgroup holds a whole channel in registers: at small batches the launches and the
// latency of each bound the two, not the bytes.  The chunks, the lanes of a chunk and the order of every sum are those of
// the two passes, so the bits are too: 256 lanes take a chunk, up to four chunks go side by side, and unit slot i of a
// lane's chunk j is register slot j * lane_units + i.  At most four slots (64 KB of x a workgroup): a channel's
// chain of loads stays short, and what is larger has workgroups enough in two passes.  With the host's 4 us a call, two passes /
// here, forward then backward: 8 images of 256 channels of 10 x 10 9.3 / 6.7 and 9.4 / 6.3 us, of 64 of 40 x 40 10.0 / 9.0 and
// 10.1 / 8.4, of 256 of 40 x 40 14.9 / 10.7 and 16.1 / 10.4; 2 of 4096 of 40 x 40 35.7 / 24.6 and 49.7 / 32.2; 16 of 64 of
// 32 x 32 (sixteen chunks, four slots: the most that is taken) 10.9 / 10.5 and 10.8 / 9.8.  Short rows: see sp_one.
// ResNet-50 on 8 images of 160 x 160: 212 launches of batch norm and 66 of their ReLUs become 110, 3.92 ms a step 3.44.
// JOIN: forward also max(y, 0) to `second`; backward masks dy with bn(x) > 0 first and writes that to `second`.
constexpr int kOneSlots = 4, kOneGroups = 4;

template <bool BWD, bool VEC, int SLOTS, bool JOIN>
__global__ __launch_bounds__(kThreads * kOneGroups) void bn_sp_one_kernel(const float *__restrict__ x,
                                                                         const float *__restrict__ dy, float *out,
                                                                         float *second, float *__restrict__ save_mean,
                                                                         float *__restrict__ save_istd, int N, int C,
                                                                         int HW, int images_per_chunk, int chunks,
                                                                         int lane_units, double m, FastDiv div_row) {
  __shared__ double part[kOneSlots * kOneGroups][4][2];
  constexpr int W = Unit<VEC>::W;
  const int c = blockIdx.x, lane = threadIdx.x & (kThreads - 1), groups = blockDim.x / kThreads;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), group = wave >> 2;
  const uint32_t row_units = (uint32_t)HW / W;
  const float mean = BWD ? save_mean[c] : 0.f, istd = BWD ? save_istd[c] : 0.f;
  const float pivot = BWD ? 0.f : x[(int64_t)c * HW];
  float xv[SLOTS][W], gv[SLOTS][W];
  int64_t at[SLOTS];  // -1: no unit
  int chunk = group, i = 0;
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
    const int n0 = chunk * images_per_chunk, n1 = min(n0 + images_per_chunk, N);
    const uint32_t total = chunk < chunks ? (uint32_t)(n1 - n0) * row_units : 0u, idx = lane + i * kThreads;
    uint32_t img, unit;
    div_row.divmod(idx, img, unit);
    at[s] = idx < total ? ((int64_t)(n0 + (int)img) * C + c) * HW + (int64_t)unit * W : -1;
#pragma unroll
    for (int k = 0; k < W; ++k) xv[s][k] = gv[s][k] = 0.f;
    if (at[s] >= 0) {
      Unit<VEC>::load(x + at[s], xv[s]);
      if (BWD) Unit<VEC>::load(dy + at[s], gv[s]);
    }
    if (++i == lane_units) {
      i = 0;
      chunk += groups;
    }
  }
  chunk = group;
  i = 0;
  float a0 = 0.f, b0 = 0.f;  // b0 by explicit fused steps: unrolled, the first two would fuse the other way round
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
    if (at[s] >= 0) {
#pragma unroll
      for (int k = 0; k < W; ++k) {
        if (BWD) {
          const float xh = (xv[s][k] - mean) * istd;
          if (JOIN) gv[s][k] = xh > 0.f ? gv[s][k] : 0.f;
          a0 += gv[s][k];
          b0 = __builtin_fmaf(gv[s][k], xh, b0);
        } else {
          const float t = xv[s][k] - pivot;
          a0 += t;
          b0 = __builtin_fmaf(t, t, b0);
        }
      }
      if (BWD && JOIN) Unit<VEC>::store(second + at[s], gv[s]);
    }
    if (++i == lane_units) {
      if (chunk < chunks) {
        const double a = wave_sum_d((double)a0), b = wave_sum_d((double)b0);
        if ((lane & 63) == 0) {
          part[chunk][wave & 3][0] = a;
          part[chunk][wave & 3][1] = b;
        }
      }
      a0 = b0 = 0.f;
      i = 0;
      chunk += groups;
    }
  }
  __syncthreads();
  // lane k folds chunk k, every wave for itself; the chain over the chunks takes the lanes' values in their order
  const int of = min(lane & 63, chunks - 1);
  const double c0 = (part[of][0][0] + part[of][1][0]) + (part[of][2][0] + part[of][3][0]);
  const double c1 = (part[of][0][1] + part[of][1][1]) + (part[of][2][1] + part[of][3][1]);
  double s0 = 0.0, s1 = 0.0;
  for (int k = 0; k < chunks; ++k) {
    s0 += lane_value(c0, k);
    s1 += lane_value(c1, k);
  }
  float f0, f1;
  channel_floats<BWD>(s0, s1, m, pivot, f0, f1);
  if (!BWD && threadIdx.x == 0) {
    save_mean[c] = f0;
    save_istd[c] = f1;
  }
  const float scale = istd / (float)m;
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
    if (at[s] < 0) continue;
    float r[W];
#pragma unroll
    for (int k = 0; k < W; ++k) {
      if (BWD) {
        const float xh = (xv[s][k] - mean) * istd;
        r[k] = scale * ((float)m * gv[s][k] - f0 - xh * f1);
      } else {
        r[k] = (xv[s][k] - f0) * f1;
      }
    }
    Unit<VEC>::store(out + at[s], r);
    if (!BWD && JOIN) {
#pragma unroll
      for (int k = 0; k < W; ++k) r[k] = r[k] < 0.f ? 0.f : r[k];
      Unit<VEC>::store(second + at[s], r);
    }
  }
}

template <int NREG, bool RELU, bool BOTH>
void pa_forward(dim3 grid, dim3 block, hipStream_t s, const float *x, float *y, float *plain, float *mean, float *istd,
                int N, uint32_t L) {
  if (N == NREG)
    hipLaunchKernelGGL((bn_pa_forward_kernel<NREG, RELU, BOTH, true>), grid, block, 0, s, x, y, plain, mean, istd, N, L);
  else
    hipLaunchKernelGGL((bn_pa_forward_kernel<NREG, RELU, BOTH, false>), grid, block, 0, s, x, y, plain, mean, istd, N, L);
}

// The register kernels address row n at the 32-bit byte offset n * L * 4.
bool pa_rows_addressable(int nreg, int64_t L) { return (int64_t)nreg * L * 4 < ((int64_t)1 << 32); }

// Rows of the register kernel that takes N rows of L columns, 0 where none does.
int pa_registers(int N, int64_t L) {
  const int nreg = N <= 32 ? 32 : N <= 64 ? 64 : 128;
  return N <= 128 && pa_rows_addressable(nreg, L) ? nreg : 0;
}

int sp_chunks(int N, int C) {
  // about four workgroups per CU in the partial pass
  int chunks = cdiv((int64_t)num_cus() * 4, C);
  if (chunks > N) chunks = N;
  return chunks < 1 ? 1 : chunks;
}

// Whether the apply pass folds the chunks itself.  That saves a launch of about 3 us, but every workgroup pays the
// lanes' chain of additions straight from the L2 and, forward, a square root in fp64 that costs as much as eight of
// them: with few rounds of workgroups and short chains.  Folding in the apply pass / before it, us forward: 32 images
// of 256 channels of 14 x 14 8.3 / 11.9, 8 of 64 of 56 x 56 8.8 / 9.4, 512 of 32 of 14 x 14 12.6 / 12.7, 300 of 16 of
// 112 x 112 141 / 119, 1000 of 1 of 224 x 224 449 / 113, 100000 of 64 of one pixel 88 / 48, 65536 of 1 of one pixel
// 138 / 22.
bool fold_in_apply(int chunks, int units_per_row, uint32_t units) {
  const int lane_rows = cdiv(cdiv(kThreads * 4 - 1, units_per_row) + 1, kThreads);  // rows that a lane folds
  const int64_t per_cu = units / (kThreads * 4) / num_cus();
  return lane_rows * (chunks + 8) * (4 + per_cu) <= 384;
}

// A channel's workgroup writes its rows in pieces of a line where they are short, the second of two passes whole lines; from 3 MB on the
// pieces of 32 images and more cost more than the second launch.  us of both directions, two passes / one: 512 images of 8192 channels of
// one pixel 82 / 139; 128 of 8192 of 1 x 3 66 / 90; 64 of 4096 of 2 x 2 28.6 / 34.3.  Not past the line: 16 of 4096 of 3 x 3 19.3 / 13.3, 64
// of 1024 of 4 x 4 (64 bytes a row) 14.8 / 7.7, 64 of 2048 of 2 x 2 (2 MB) 19.8 / 17.1.  Of 714 shapes of up to 36 pixels and 32 MB
// four stay slower in one launch, by up to 7 %; the 714 together take 0.70 of two passes' time.
constexpr int kShortRow = 16, kManyRows = 32;
constexpr int64_t kShortRowElements = 3 << 18;

// Whether bn_sp_one_kernel takes the tensor, and how: `slots` 0 where it does not.
struct SpOne {
  bool vec;
  int chunks, images_per_chunk, groups, lane_units, slots;
};
SpOne sp_one(const BNDesc *d, uintptr_t addresses) {
  SpOne o = {};
  if (d->mode != 1 || d->two_passes || d->N < 1 || d->C < 1 || d->HW < 1) return o;
  o.vec = d->HW % 4 == 0 && (addresses & 15u) == 0;
  o.images_per_chunk = cdiv(d->N, sp_chunks(d->N, d->C));
  o.chunks = cdiv(d->N, o.images_per_chunk);
  o.groups = std::min(o.chunks, kOneGroups);
  const int64_t units = (int64_t)o.images_per_chunk * (o.vec ? d->HW / 4 : d->HW);
  const int64_t slots = (units + kThreads - 1) / kThreads * cdiv(o.chunks, o.groups);
  if (slots > kOneSlots) return o;
  if (d->HW < kShortRow && d->N >= kManyRows && (int64_t)d->N * d->C * d->HW > kShortRowElements) return o;
  o.lane_units = (int)((units + kThreads - 1) / kThreads);
  o.slots = (int)slots;
  return o;
}

template <bool BWD, bool JOIN>
void launch_sp_one(const BNDesc *d, const SpOne &o, hipStream_t s, const float *x, const float *dy, float *out, float *second,
                   float *mean, float *istd) {
  auto go = [&](auto vec_c, auto slots_c) {
    constexpr bool VEC = decltype(vec_c)::value;
    hipLaunchKernelGGL((bn_sp_one_kernel<BWD, VEC, decltype(slots_c)::value, JOIN>), dim3(d->C), dim3(kThreads * o.groups), 0,
                       s, x, dy, out, second, mean, istd, d->N, d->C, d->HW, o.images_per_chunk, o.chunks, o.lane_units,
                       (double)d->N * (double)d->HW, FastDiv((uint32_t)(d->HW / (VEC ? 4 : 1))));
  };
  auto by_slots = [&](auto vec_c) {
    if (o.slots == 1) go(vec_c, std::integral_constant<int, 1>{});
    else if (o.slots == 2) go(vec_c, std::integral_constant<int, 2>{});
    else go(vec_c, std::integral_constant<int, kOneSlots>{});
  };
  if (o.vec) by_slots(std::true_type{}); else by_slots(std::false_type{});
}

uintptr_t address(const void *p) { return reinterpret_cast<uintptr_t>(p); }

int check_bn_arrays(const BNDesc *d, const DLArray *a, const DLArray *b) {
  TF_REQUIRE(on_gpu(a) && on_gpu(b), "arrays must live on the GPU");
  const int64_t n = (int64_t)d->N * d->C * d->HW;
  TF_REQUIRE(numel(a) == n && numel(b) == n, "arrays do not match the descriptor");
  // the spatial kernels index units with 32-bit fast division
  TF_REQUIRE(d->mode == 0 || n < (int64_t(1) << 31), "spatial mode supports fewer than 2^31 elements");
  return 0;
}

}  // namespace

extern "C" int DLGpuBatchNormalizationGetCudnnlist(const int *input_shapes, int sizeofshape, int dataformat,
                                                   int batchNormMode, void **mean_p, void **Variance_p,
                                                   void ***list) {
  (void)mean_p;
  (void)Variance_p;
  TF_REQUIRE(input_shapes && list, "null argument");
  TF_REQUIRE(sizeofshape >= 2 && sizeofshape <= 5, "rank %d not supported", sizeofshape);
  TF_REQUIRE(dataformat == 0, "only NCHW (dataformat 0) is implemented");
  TF_REQUIRE(batchNormMode == 0 || batchNormMode == 1, "unknown batch-norm mode %d", batchNormMode);
  int64_t hw = 1;
  for (int i = 0; i < sizeofshape; ++i) {
    TF_REQUIRE(input_shapes[i] >= 0, "negative extent");
    if (i >= 2) hw *= input_shapes[i];
    TF_REQUIRE(hw <= INT32_MAX, "spatial extent too large");
  }
  BNDesc *d = new BNDesc();
  d->magic = kMagicBN;
  d->mode = batchNormMode;
  d->N = input_shapes[0];
  d->C = input_shapes[1];
  d->HW = (int)hw;
  d->stat_count = batchNormMode == 0 ? (int64_t)d->C * d->HW : d->C;
  // TINYFLOW_SPATIAL_ONE_LAUNCH=0 in the environment keeps a descriptor to two passes (tests: both have the same bits)
  const char *one_launch = getenv("TINYFLOW_SPATIAL_ONE_LAUNCH");
  d->two_passes = one_launch && *one_launch && atoi(one_launch) == 0;
  d->saved_mean = d->saved_istd = nullptr;
  void **slots = (void **)malloc(sizeof(void *) * 3);
  slots[0] = slots[1] = slots[2] = d;
  *list = slots;
  return 0;
}

static int bn_forward_impl(const DLArrayHandle input, DLArrayHandle output, int batchNormMode, int n,
                           void **mean_p, void **Variance_p, void ***list, void **handle, int *memorytoSaving,
                           void **stream, bool relu, float *plain, const char *what) {
  (void)handle;
  (void)n;  // would weight running statistics, which the reference never keeps
  BNDesc *d = desc_from_list<BNDesc>(list, kMagicBN);
  TF_REQUIRE(d, "descriptor list was not created by DLGpuBatchNormalizationGetCudnnlist");
  TF_REQUIRE(d->mode == batchNormMode, "mode differs from the descriptor");
  TF_REQUIRE(mean_p && Variance_p, "null statistics cell");
  TF_REQUIRE(!relu || d->mode == 0 || plain, "the fused batch-norm + ReLU entry points implement per-activation mode only");
  if (check_bn_arrays(d, input, output) != 0) return -1;
  const SpOne one = sp_one(d, address(input->data) | address(output->data) | address(plain));
  hipStream_t s = stream_of(stream);
  const size_t stat_bytes = (size_t)d->stat_count * sizeof(float);
  if (d->saved_mean) {  // a forward whose backward never ran: recycle its statistics
    device_free(d->saved_mean, d->saved_on);
    device_free(d->saved_istd, d->saved_on);
    d->saved_mean = d->saved_istd = nullptr;
  }
  // Everything this call allocates, which is what it reports when any of it cannot be had:
  // a caller that makes that much room must be able to repeat the call.
  const int sp_real_chunks = (d->mode == 0 || numel(input) == 0 || one.slots) ? 0 : cdiv(d->N, cdiv(d->N, sp_chunks(d->N, d->C)));
  // chunk partials of every channel and, behind them, the channels' pivots
  const size_t sp_partial_bytes = sp_real_chunks ? (size_t)d->C * (sp_real_chunks * 2 * sizeof(double) + sizeof(float)) : 0;
  const size_t all_bytes = 2 * block_bytes(stat_bytes) + (sp_partial_bytes ? block_bytes(sp_partial_bytes) : 0);
  float *mean = (float *)device_alloc(stat_bytes, s);
  float *istd = mean ? (float *)device_alloc(stat_bytes, s) : nullptr;
  if (!mean || !istd) {
    if (mean) device_free(mean, s);
    if (memorytoSaving) *memorytoSaving = shortfall(all_bytes);
    return 0;
  }
  *mean_p = d->saved_mean = mean;
  *Variance_p = d->saved_istd = istd;
  d->saved_on = s;
  const float *x = (const float *)input->data;
  float *y = (float *)output->data;
  if (numel(input) == 0) return 0;
  if (d->mode == 0) {
    const int64_t L = d->stat_count;
    const dim3 grid(cdiv(L, kThreads)), block(kThreads);  // one lane per column
    auto run = [&](auto relu_c, auto both_c) {
      constexpr bool RELU = decltype(relu_c)::value, BOTH = decltype(both_c)::value;
      const uint32_t l32 = (uint32_t)L;
      const int nreg = pa_registers(d->N, L);
      if (nreg == 32)
        pa_forward<32, RELU, BOTH>(grid, block, s, x, y, plain, mean, istd, d->N, l32);
      else if (nreg == 64)
        pa_forward<64, RELU, BOTH>(grid, block, s, x, y, plain, mean, istd, d->N, l32);
      else if (nreg == 128)
        pa_forward<128, RELU, BOTH>(grid, block, s, x, y, plain, mean, istd, d->N, l32);
      else if (d->N < kFewRows)
        hipLaunchKernelGGL(bn_pa_forward_stream_kernel<RELU>, grid, block, 0, s, x, y, mean, istd, d->N, L);
      else
        bn_pa_forward_tiles<RELU>(s, x, y, mean, istd, d->N, L);
    };
    if (plain) run(std::true_type{}, std::true_type{});  // the caller has checked that a register kernel takes it
    else if (relu) run(std::true_type{}, std::false_type{});
    else run(std::false_type{}, std::false_type{});
  } else if (one.slots) {
    if (plain) launch_sp_one<false, true>(d, one, s, x, nullptr, plain, y, mean, istd);
    else launch_sp_one<false, false>(d, one, s, x, nullptr, y, nullptr, mean, istd);
  } else {
    const int chunks = sp_chunks(d->N, d->C);
    const int ipc = cdiv(d->N, chunks);
    const int real_chunks = sp_real_chunks;
    double *partial = (double *)device_alloc(sp_partial_bytes, s);
    if (!partial) {
      device_free(mean, s);
      device_free(istd, s);
      *mean_p = d->saved_mean = nullptr;
      *Variance_p = d->saved_istd = nullptr;
      if (memorytoSaving) *memorytoSaving = shortfall(all_bytes);
      return 0;
    }
    float *pivots = reinterpret_cast<float *>(partial + (size_t)real_chunks * d->C * 2);
    const bool vec = d->HW % 4 == 0 && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 15u) == 0;
    const int W = vec ? 4 : 1;
    const FastDiv div_row((uint32_t)(d->HW / W)), div_c((uint32_t)d->C);
    const uint32_t units = (uint32_t)((int64_t)d->N * d->C * d->HW / W);
    const dim3 pgrid(d->C, real_chunks), agrid((units + kThreads * 4 - 1) / (kThreads * 4));
    auto run = [&](auto vec_c) {
      constexpr bool VEC = decltype(vec_c)::value;
      hipLaunchKernelGGL((bn_sp_partial_kernel<false, VEC>), pgrid, dim3(kThreads), 0, s, x, (const float *)nullptr,
                         (const float *)nullptr, (const float *)nullptr, partial, pivots, d->N, d->C, d->HW, ipc, div_row);
      const double m = (double)d->N * (double)d->HW;
      if (fold_in_apply(real_chunks, div_row.d, units)) {
        hipLaunchKernelGGL((bn_sp_apply_kernel<false, VEC, true>), agrid, dim3(kThreads), 0, s, x,
                           (const float *)nullptr, y, (const double *)partial, (const float *)pivots, real_chunks, m,
                           (const float *)nullptr, (const float *)nullptr, mean, istd, div_row, div_c, units);
      } else {
        const int log_ch = finish_log_channels(real_chunks);
        hipLaunchKernelGGL(bn_sp_finish_kernel<false>, dim3(cdiv(d->C, 1 << log_ch)), dim3(kThreads), 0, s,
                           (const double *)partial, (const float *)pivots, mean, istd, d->C, real_chunks, m, log_ch);
        hipLaunchKernelGGL((bn_sp_apply_kernel<false, VEC, false>), agrid, dim3(kThreads), 0, s, x,
                           (const float *)nullptr, y, (const double *)nullptr, (const float *)nullptr, 0, m,
                           (const float *)mean, (const float *)istd, mean, istd, div_row, div_c, units);
      }
    };
    if (vec) run(std::true_type{}); else run(std::false_type{});
    device_free(partial, s);
  }
  return finish(s, what);
}

extern "C" int DLGpuBatchNormalizationForward(const DLArrayHandle input, DLArrayHandle output,
                                              int batchNormMode, int n, void **mean_p, void **Variance_p,
                                              void ***list, void **handle, int *memorytoSaving,
                                              void **stream) {
  announce_write(output);
  return bn_forward_impl(input, output, batchNormMode, n, mean_p, Variance_p, list, handle, memorytoSaving, stream,
                         false, nullptr, "DLGpuBatchNormalizationForward");
}

// No counterpart in the reference: y = max(bn(x), 0) in one pass over x (8 bytes per
// element instead of 16 for the two ops), per-activation mode.  Same statistics
// protocol as the plain forward; pairs with DLGpuBatchNormalizationReluBackward.
extern "C" int DLGpuBatchNormalizationReluForward(const DLArrayHandle input, DLArrayHandle output,
                                                  int batchNormMode, int n, void **mean_p, void **Variance_p,
                                                  void ***list, void **handle, int *memorytoSaving,
                                                  void **stream) {
  announce_write(output);
  return bn_forward_impl(input, output, batchNormMode, n, mean_p, Variance_p, list, handle, memorytoSaving, stream,
                         true, nullptr, "DLGpuBatchNormalizationReluForward");
}

static int bn_backward_impl(const DLArrayHandle input, const DLArrayHandle doutput, DLArrayHandle dinput,
                            int batchNormMode, void **mean_p, void **Variance_p, void ***list, void **handle,
                            int *memorytoSaving, void **stream, bool relu, float *masked, const char *what) {
  (void)handle;
  BNDesc *d = desc_from_list<BNDesc>(list, kMagicBN);
  TF_REQUIRE(d, "descriptor list was not created by DLGpuBatchNormalizationGetCudnnlist");
  TF_REQUIRE(d->mode == batchNormMode, "mode differs from the descriptor");
  // the cells start out pointing at host integers, so "non-null" proves nothing:
  // they must hold exactly what the last forward published
  TF_REQUIRE(mean_p && Variance_p && d->saved_mean && *mean_p == d->saved_mean &&
                 *Variance_p == d->saved_istd,
             "no saved statistics: backward needs the forward pass of the same step");
  TF_REQUIRE(!relu || d->mode == 0 || masked, "the fused batch-norm + ReLU entry points implement per-activation mode only");
  if (check_bn_arrays(d, input, doutput) != 0) return -1;
  TF_REQUIRE(on_gpu(dinput) && numel(dinput) == numel(input), "dinput must have the input's shape");
  hipStream_t s = stream_of(stream);
  const float *x = (const float *)input->data, *dy = (const float *)doutput->data;
  float *dx = (float *)dinput->data;
  const float *mean = (const float *)*mean_p, *istd = (const float *)*Variance_p;
  const SpOne one = sp_one(d, address(x) | address(dy) | address(dx) | address(masked));
  if (numel(input) != 0) {
    if (d->mode == 0) {
      const int64_t L = d->stat_count;
      const dim3 grid(cdiv(L, kThreads)), block(kThreads);  // one lane per column
      auto run = [&](auto relu_c, auto both_c) {
        constexpr bool RELU = decltype(relu_c)::value, BOTH = decltype(both_c)::value;
        const uint32_t l32 = (uint32_t)L;
        const int nreg = pa_registers(d->N, L);
        if (nreg == 32)
          hipLaunchKernelGGL((bn_pa_backward_kernel<32, RELU, BOTH>), grid, block, 0, s, x, dy, dx, masked, mean, istd,
                             d->N, l32);
        else if (nreg == 64)
          hipLaunchKernelGGL((bn_pa_backward_kernel<64, RELU, BOTH>), grid, block, 0, s, x, dy, dx, masked, mean, istd,
                             d->N, l32);
        else if (nreg == 128)
          hipLaunchKernelGGL((bn_pa_backward_kernel<128, RELU, BOTH>), grid, block, 0, s, x, dy, dx, masked, mean, istd,
                             d->N, l32);
        else if (many_columns(L))
          hipLaunchKernelGGL(bn_pa_backward_stream_kernel<RELU>, grid, block, 0, s, x, dy, dx, mean, istd, d->N, L);
        else
          bn_pa_backward_tiles<RELU>(s, x, dy, dx, mean, istd, d->N, L);
      };
      if (masked) run(std::true_type{}, std::true_type{});  // as in the forward pass
      else if (relu) run(std::true_type{}, std::false_type{});
      else run(std::false_type{}, std::false_type{});
    } else if (one.slots) {
      float *stat0 = const_cast<float *>(mean), *stat1 = const_cast<float *>(istd);
      if (masked) launch_sp_one<true, true>(d, one, s, x, dy, dx, masked, stat0, stat1);
      else launch_sp_one<true, false>(d, one, s, x, dy, dx, nullptr, stat0, stat1);
    } else {
      const int chunks = sp_chunks(d->N, d->C);
      const int ipc = cdiv(d->N, chunks);
      const int real_chunks = cdiv(d->N, ipc);
      // chunk partials of every channel and, behind them, the channels' two sums
      const size_t pbytes = (size_t)d->C * (real_chunks * 2 * sizeof(double) + 2 * sizeof(float));
      double *partial = (double *)device_alloc(pbytes, s);
      if (!partial) {
        if (memorytoSaving) *memorytoSaving = shortfall(pbytes);
        return 0;  // statistics stay published so the call can be repeated
      }
      float *sums = reinterpret_cast<float *>(partial + (size_t)real_chunks * d->C * 2);
      const bool vec = d->HW % 4 == 0 &&
                       ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(dy) |
                         reinterpret_cast<uintptr_t>(dx)) & 15u) == 0;
      const int W = vec ? 4 : 1;
      const FastDiv div_row((uint32_t)(d->HW / W)), div_c((uint32_t)d->C);
      const uint32_t units = (uint32_t)((int64_t)d->N * d->C * d->HW / W);
      const dim3 pgrid(d->C, real_chunks), agrid((units + kThreads * 4 - 1) / (kThreads * 4));
      auto run = [&](auto vec_c) {
        constexpr bool VEC = decltype(vec_c)::value;
        hipLaunchKernelGGL((bn_sp_partial_kernel<true, VEC>), pgrid, dim3(kThreads), 0, s, x, dy, mean, istd, partial,
                           (float *)nullptr, d->N, d->C, d->HW, ipc, div_row);
        const double m = (double)d->N * (double)d->HW;
        float *stat0 = const_cast<float *>(mean), *stat1 = const_cast<float *>(istd);
        if (fold_in_apply(real_chunks, div_row.d, units)) {
          hipLaunchKernelGGL((bn_sp_apply_kernel<true, VEC, true>), agrid, dim3(kThreads), 0, s, x, dy, dx,
                             (const double *)partial, (const float *)nullptr, real_chunks, m, (const float *)nullptr,
                             (const float *)nullptr, stat0, stat1, div_row, div_c, units);
        } else {
          const int log_ch = finish_log_channels(real_chunks);
          hipLaunchKernelGGL(bn_sp_finish_kernel<true>, dim3(cdiv(d->C, 1 << log_ch)), dim3(kThreads), 0, s,
                             (const double *)partial, (const float *)nullptr, sums, sums + d->C, d->C, real_chunks, m,
                             log_ch);
          hipLaunchKernelGGL((bn_sp_apply_kernel<true, VEC, false>), agrid, dim3(kThreads), 0, s, x, dy, dx,
                             (const double *)nullptr, (const float *)nullptr, 0, m, (const float *)sums,
                             (const float *)(sums + d->C), stat0, stat1, div_row, div_c, units);
        }
      };
      if (vec) run(std::true_type{}); else run(std::false_type{});
      device_free(partial, s);
    }
  }
  // the saved statistics are consumed (stream-ordered release)
  device_free(d->saved_mean, s);
  device_free(d->saved_istd, s);
  *mean_p = d->saved_mean = nullptr;
  *Variance_p = d->saved_istd = nullptr;
  return finish(s, what);
}

extern "C" int DLGpuBatchNormalizationBackward(const DLArrayHandle input, const DLArrayHandle doutput,
                                               DLArrayHandle dinput, int batchNormMode, void **mean_p,
                                               void **Variance_p, void ***list, void **handle,
                                               int *memorytoSaving, void **stream) {
  announce_write(dinput);
  return bn_backward_impl(input, doutput, dinput, batchNormMode, mean_p, Variance_p, list, handle, memorytoSaving,
                          stream, false, nullptr, "DLGpuBatchNormalizationBackward");
}

// No counterpart in the reference: gradient of max(bn(x), 0) with respect to x.
// doutput is the gradient of the ReLU output; the ReLU mask bn(x) > 0 is rebuilt
// from x and the saved statistics, so neither bn(x) nor the ReLU output is read
// (12 bytes per element instead of 24 for the two ops).
extern "C" int DLGpuBatchNormalizationReluBackward(const DLArrayHandle input, const DLArrayHandle doutput,
                                                   DLArrayHandle dinput, int batchNormMode, void **mean_p,
                                                   void **Variance_p, void ***list, void **handle,
                                                   int *memorytoSaving, void **stream) {
  announce_write(dinput);
  return bn_backward_impl(input, doutput, dinput, batchNormMode, mean_p, Variance_p, list, handle, memorytoSaving,
                          stream, true, nullptr, "DLGpuBatchNormalizationReluBackward");
}

// Whether one pass over the tensor does both: the per-activation register kernels (up to 128 images), and spatial
// mode's where a workgroup holds a channel.
static bool joint_pass(const BNDesc *d, int batchNormMode, uintptr_t addresses) {
  if (d->mode != batchNormMode) return false;
  return d->mode == 0 ? pa_registers(d->N, d->stat_count) != 0 : sp_one(d, addresses).slots != 0;
}

// bn_output = bn(x) and relu_output = max(bn(x), 0): one pass where there is one for the tensor, else the two calls that
// this stands for, with the same bytes.
extern "C" int DLGpuBatchNormalizationAndReluForward(const DLArrayHandle input, DLArrayHandle bn_output,
                                                     DLArrayHandle relu_output, int batchNormMode, int n, void **mean_p,
                                                     void **Variance_p, void ***list, void ***activation_list,
                                                     void **handle, int *memorytoSaving, void **stream) {
  const BNDesc *d = desc_from_list<BNDesc>(list, kMagicBN);
  TF_REQUIRE(d, "descriptor list was not created by DLGpuBatchNormalizationGetCudnnlist");
  if (check_bn_arrays(d, input, bn_output) != 0 || check_bn_arrays(d, input, relu_output) != 0) return -1;
  if (joint_pass(d, batchNormMode, address(input->data) | address(bn_output->data) | address(relu_output->data)) &&
      bn_output->data != relu_output->data) {
    announce_write(bn_output);
    announce_write(relu_output);
    return bn_forward_impl(input, relu_output, batchNormMode, n, mean_p, Variance_p, list, handle, memorytoSaving, stream,
                           true, (float *)bn_output->data, "DLGpuBatchNormalizationAndReluForward");
  }
  int wanted = 0;
  const int rc = DLGpuBatchNormalizationForward(input, bn_output, batchNormMode, n, mean_p, Variance_p, list, handle,
                                                &wanted, stream);
  if (memorytoSaving && wanted) *memorytoSaving = wanted;
  return rc || wanted ? rc : DLGpuActivationForward(bn_output, relu_output, 1, activation_list, handle, stream);
}

// drelu = doutput where bn(x) > 0, else 0, and dinput = the batch norm's gradient of it: one pass under the same rule
// (the mask rebuilt from x and the saved statistics, which has bn_output's bits), else the two calls.
extern "C" int DLGpuBatchNormalizationAndReluBackward(const DLArrayHandle input, const DLArrayHandle bn_output,
                                                      const DLArrayHandle relu_output, const DLArrayHandle doutput,
                                                      DLArrayHandle drelu, DLArrayHandle dinput, int batchNormMode,
                                                      void **mean_p, void **Variance_p, void ***list,
                                                      void ***activation_list, void **handle, int *memorytoSaving,
                                                      void **stream) {
  const BNDesc *d = desc_from_list<BNDesc>(list, kMagicBN);
  TF_REQUIRE(d, "descriptor list was not created by DLGpuBatchNormalizationGetCudnnlist");
  if (check_bn_arrays(d, input, doutput) != 0 || check_bn_arrays(d, drelu, dinput) != 0) return -1;
  // in place the two calls read what they have written
  const void *const read[] = {input->data, doutput->data};
  const bool apart = drelu->data != dinput->data && drelu->data != read[0] && dinput->data != read[1];
  if (joint_pass(d, batchNormMode, address(read[0]) | address(read[1]) | address(dinput->data) | address(drelu->data)) &&
      apart) {
    announce_write(drelu);
    announce_write(dinput);
    return bn_backward_impl(input, doutput, dinput, batchNormMode, mean_p, Variance_p, list, handle, memorytoSaving,
                            stream, true, (float *)drelu->data, "DLGpuBatchNormalizationAndReluBackward");
  }
  const int rc = DLGpuActivationBackward(bn_output, drelu, relu_output, doutput, 1, activation_list, handle, stream);
  return rc ? rc : DLGpuBatchNormalizationBackward(input, drelu, dinput, batchNormMode, mean_p, Variance_p, list, handle,
                                                   memorytoSaving, stream);
}
