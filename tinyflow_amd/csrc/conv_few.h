// Forward and stride-1 grad-data of convolutions with few output channels, on the vector units.
//
// The tile engine's 64 rows are mostly padding for a handful of channels, and every element of the pixel operand is
// gathered with an address of its own: 6 <- 16 channels, 5x5, 1 000 images of 14 x 14 took 118 us for 0.9 GFLOP.  Here a lane
// owns one output pixel and all channels of it.  The source pixels of a workgroup's range of outputs lie in LDS, zeros
// around them, so a tap is one LDS read at a constant offset, shared by all channels, and the filter comes through
// scalar loads.  What bounds it is the latency of those, covered by other waves only: that layer 51 us, forward of its first,
// 1 -> 6 channels, 59 -> 19; fetching the next row's filter values ahead spills scalar registers and is slower
// (82 and 30 us).
//
// The sums are the tile engine's, bit for bit: its matrix instruction is a chain of fused multiply-adds in the order of the
// reduction (channel, tap row, tap column), which is what a lane does here; where the engine's plan cuts the reduction into
// pieces (Fold in gemm_core.h) the pieces are summed apart and added in order.
#pragma once

#include "gemm_core.h"

namespace tf {
namespace few {

using gemm::FastDiv;

struct Conv {
  int N, M, C;                 // images, output channels, source channels
  int Hs, Ws, OW, OHW;         // source plane, output row and plane
  int R, u, v;                 // tap rows; strides (1 for grad-data)
  int row0, col0;              // source position of LDS (0, 0) for output row 0
  int images, span, ranges;    // a workgroup: `images` whole planes, or (images = 1) one of `ranges` spans of a plane
  int rows, width;             // LDS plane of one image and channel
  int chunk;                   // source channels in LDS at a time
  int piece, tile, first_tile; // reduction steps a piece (0: uncut) in tiles of `tile` output columns from first_tile on
  FastDiv div_ow, div_ohw, div_width, div_rows, div_chunk, div_ranges, div_tile;
};

constexpr int kThreads = 256;

template <int MT, int S, bool DGRAD>
__global__ __launch_bounds__(kThreads) void gemm_kernel(const float *__restrict__ src, const float *__restrict__ w,
                                                              float *__restrict__ out, const Conv p) {
  extern __shared__ float lds[];  // [image][channel][rows][width]
  uint32_t block_image, range;
  p.div_ranges.divmod(blockIdx.x, block_image, range);
  const int image0 = (int)block_image * p.images;
  const int first = (int)range * p.span;  // first output of the range (0 for whole planes)
  // this lane's output
  uint32_t g = 0, pixel = (uint32_t)first + threadIdx.x;
  bool valid;
  if (p.images > 1) {
    p.div_ohw.divmod(threadIdx.x, g, pixel);
    valid = (int)g < p.images && image0 + (int)g < p.N;
  } else {
    valid = (int)threadIdx.x < p.span && (int)pixel < p.OHW;
  }
  if (!valid) g = 0, pixel = (uint32_t)first;
  uint32_t oh, ow;
  p.div_ow.divmod(pixel, oh, ow);
  const int oh0 = (int)p.div_ow.div((uint32_t)first);
  const int plane = p.rows * p.width;
  // LDS position of tap (0, 0); taps go down and right (forward) or up and left
  const int at = (int)g * p.chunk * plane + (DGRAD ? ((int)oh - oh0 + p.R - 1) * p.width + (int)ow + S - 1
                                                   : ((int)oh - oh0) * p.u * p.width + (int)ow * p.v);
  const int src_row0 = p.row0 + (DGRAD ? oh0 : oh0 * p.u);
  const bool cut = p.piece > 0 && (int)p.div_tile.div((uint32_t)((image0 + (int)g) * p.OHW + (int)pixel)) >= p.first_tile;

  float acc[MT], total[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = total[m] = 0.f;
  int k = 0, boundary = p.piece > 0 ? p.piece : 0x7fffffff;
  for (int c0 = 0; c0 < p.C; c0 += p.chunk) {
    if (c0) __syncthreads();
    const int fill = p.images * p.chunk * plane;
    for (int i = threadIdx.x; i < fill; i += kThreads) {
      uint32_t t, col, row, c, gi;
      p.div_width.divmod((uint32_t)i, t, col);
      p.div_rows.divmod(t, t, row);
      p.div_chunk.divmod(t, gi, c);
      const int y = src_row0 + (int)row, x = p.col0 + (int)col, image = image0 + (int)gi, ch = c0 + (int)c;
      const bool inside = (uint32_t)y < (uint32_t)p.Hs && (uint32_t)x < (uint32_t)p.Ws && image < p.N && ch < p.C;
      lds[i] = inside ? src[(((int64_t)image * p.C + ch) * p.Hs + y) * p.Ws + x] : 0.f;
    }
    __syncthreads();
    const int channels = min(p.chunk, p.C - c0);
    for (int c = 0; c < channels; ++c) {
      for (int r = 0; r < p.R; ++r) {
        // the S taps of this row for every output channel; past the last channel the last one again
        const float *row = lds + at + c * plane + (DGRAD ? -r : r) * p.width;
        float tap[S], f[MT][S];
#pragma unroll
        for (int s = 0; s < S; ++s) tap[s] = row[DGRAD ? -s : s];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const int mm = min(m, p.M - 1);
          const int64_t base = DGRAD ? (((int64_t)(c0 + c) * p.M + mm) * p.R + r) * S
                                     : (((int64_t)mm * p.C + c0 + c) * p.R + r) * S;
#pragma unroll
          for (int s = 0; s < S; ++s) f[m][s] = w[base + s];
        }
        if (k + S <= boundary) {
#pragma unroll
          for (int s = 0; s < S; ++s)
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[m] = __builtin_fmaf(f[m][s], tap[s], acc[m]);
        } else {
#pragma unroll
          for (int s = 0; s < S; ++s) {
            if (k + s == boundary) {
              boundary += p.piece;
#pragma unroll
              for (int m = 0; m < MT; ++m) {
                total[m] = cut ? total[m] + acc[m] : total[m];
                acc[m] = cut ? 0.f : acc[m];
              }
            }
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[m] = __builtin_fmaf(f[m][s], tap[s], acc[m]);
          }
        }
        k += S;
      }
    }
  }
  if (!valid) return;
  float *dst = out + ((int64_t)(image0 + (int)g) * p.M) * p.OHW + pixel;
#pragma unroll
  for (int m = 0; m < MT; ++m)
    if (m < p.M) dst[(int64_t)m * p.OHW] = cut ? total[m] + acc[m] : acc[m];
}

}  // namespace few
}  // namespace tf
