// Several elementwise nodes of a step graph in one launch: every result is written, as the calls that a group stands
// for write it, with the same arithmetic; a step that reads what an earlier one of the group made takes it from
// registers.
//
// Bound by the launch: the arrays of small networks are a few KB, a call costs the host 3.6 us and the device 2 us
// whatever they hold, and a fully connected layer has five such calls (bias broadcast, sum and ReLU; the ReLU's gradient
// and the sum with zeros that the bias's adjoint brings).  MLP step at batch 128: 36 launches -> 25, 180 -> 154 us; LeNet-5 at batch 64:
// 63 -> 46, 282 -> 245.  Arrays of millions of elements move as many bytes as the separate calls with their joins and
// kept sign bits (LeNet-5 at batch 1 000: 579 us both ways).
#include "ew_core.h"
#include "gemm_core.h"
#include "internal.h"

#include <algorithm>

using namespace tf;
using namespace tf::ew;
using tf::gemm::FastDiv;

namespace {

constexpr int kMaxSteps = 6;   // operands are picked by a chain of scalar moves, fifteen of them for the sixth step

struct Step {
  int kind;
  float value;
  int from_a, from_b;            // the step of the group that made the operand, -1: memory
  const float *a, *b;
  float *out;
  uint32_t n;
  FastDiv inner, channels;       // kGroupBroadcast: out[i] = a[i / inner % channels]
};
struct Group {
  Step s[kMaxSteps];
  int steps;
};

// VEC: four consecutive elements a lane, every array 16-byte aligned, every length a multiple of four (or one).
template <bool VEC>
__global__ __launch_bounds__(kThreads) void group_kernel(const Group g, uint32_t n) {
#pragma clang fp contract(off)  // a product and a sum of two nodes are rounded apart
  constexpr int W = VEC ? 4 : 1;
  const uint32_t i = (blockIdx.x * kThreads + threadIdx.x) * W;
  if (i >= n) return;
  float r[kMaxSteps][W];
#pragma unroll
  for (int k = 0; k < kMaxSteps; ++k) {
    if (k >= g.steps) break;   // uniform
    const Step &s = g.s[k];
    const bool one = s.n == 1;
    if (one ? i != 0 : i >= s.n) continue;
    float a[W], b[W];
    auto fetch = [&](const float *p, int from, float (&v)[W]) {
      if (from < 0) {
        if (p == nullptr) {
#pragma unroll
          for (int e = 0; e < W; ++e) v[e] = 0.f;
        } else if (VEC && !one) {
          const f32x4 q = *reinterpret_cast<const f32x4 *>(p + i);
          v[0] = q.x;
          if constexpr (VEC) {
            v[1] = q.y;
            v[2] = q.z;
            v[3] = q.w;
          }
        } else {
          v[0] = p[i];
        }
      }
#pragma unroll
      for (int j = 0; j < k; ++j)
        if (from == j) {
#pragma unroll
          for (int e = 0; e < W; ++e) v[e] = r[j][e];
        }
    };
    if (s.kind == kGroupBroadcast) {
#pragma unroll
      for (int e = 0; e < W; ++e) {
        uint32_t q, c;
        s.channels.divmod(s.inner.div(i + e), q, c);
        r[k][e] = s.a[c];
      }
    } else {
      fetch(s.a, s.from_a, a);
      fetch(s.b, s.from_b, b);
#pragma unroll
      for (int e = 0; e < W; ++e) {
        float v = s.value;                                              // kGroupSet
        if (s.kind == kGroupAdd) v = a[e] + b[e];
        else if (s.kind == kGroupAddConst) v = a[e] + s.value;
        else if (s.kind == kGroupMul) v = a[e] * b[e];
        else if (s.kind == kGroupMulConst) v = a[e] * s.value;
        else if (s.kind == kGroupRelu) v = a[e] < 0.f ? 0.f : a[e];
        else if (s.kind == kGroupReluGradient) v = a[e] > 0.f ? b[e] : 0.f;
        r[k][e] = v;
      }
    }
    if (VEC && !one) {
      if constexpr (VEC) *reinterpret_cast<f32x4 *>(s.out + i) = f32x4{r[k][0], r[k][1], r[k][2], r[k][3]};
    } else {
      s.out[i] = r[k][0];
    }
  }
}

bool overlap(const float *a, int64_t na, const float *b, int64_t nb) { return a < b + nb && b < a + na; }

}  // namespace

extern "C" int DLGpuElementwiseGroup(const DLGroupStep *steps, int n_steps, int ordered, void **stream) {
  TF_REQUIRE(steps && n_steps >= 1 && n_steps <= kMaxSteps, "a group has 1 to %d steps", kMaxSteps);
  for (int k = 0; k < n_steps; ++k) announce_write(steps[k].out);
  Group g;
  g.steps = n_steps;
  int64_t n = 0;
  for (int k = 0; k < n_steps; ++k) {
    const DLGroupStep &in = steps[k];
    TF_REQUIRE(in.kind >= kGroupSet && in.kind <= kGroupBroadcast, "unknown kind %d", in.kind);
    const bool has_a = in.kind != kGroupSet;
    const bool has_b = in.kind == kGroupAdd || in.kind == kGroupMul || in.kind == kGroupReluGradient;
    TF_REQUIRE(on_gpu(in.out) && (!has_a || on_gpu(in.a)) && (!has_b || on_gpu(in.b)), "arrays must live on the GPU");
    n = std::max(n, numel(in.out));
  }
  TF_REQUIRE(n < ((int64_t)1 << 31), "tensors of 2^31 elements or more are not supported");
  bool vec = true;
  auto fits = [&](const DLArray *x) {
    const int64_t m = numel(x);
    if (m != 1) vec = vec && m % 4 == 0 && aligned16(x->data);
  };
  for (int k = 0; k < n_steps; ++k) {
    const DLGroupStep &in = steps[k];
    Step &s = g.s[k];
    const bool has_a = in.kind != kGroupSet;
    const bool has_b = in.kind == kGroupAdd || in.kind == kGroupMul || in.kind == kGroupReluGradient;
    const int64_t m = numel(in.out);
    s.kind = in.kind;
    s.value = in.value;
    s.out = (float *)in.out->data;
    s.n = (uint32_t)m;
    s.a = has_a ? (const float *)in.a->data : nullptr;
    s.b = has_b ? (const float *)in.b->data : nullptr;
    s.from_a = s.from_b = -1;
    // an array of one element beside longer ones is on its own: lanes other than the first have no value of it
    TF_REQUIRE(m == n || m == 1, "the steps of a group have one length");
    fits(in.out);
    if (in.kind == kGroupBroadcast) {
      // what DLGpuBroadcastTo0 and 1 take
      int64_t inner = 1;
      for (int i = 2; in.per_channel && i < in.out->ndim; ++i) inner *= in.out->shape[i];
      const int64_t channels = numel(in.a);
      if (in.per_channel) {
        TF_REQUIRE(in.a->ndim == 1 && in.out->ndim >= 2 && channels == in.out->shape[1], "input must be (C,) and output (N, C, ...)");
      } else if (!(in.a->ndim == 1 && channels == 1)) {
        TF_REQUIRE(in.a->ndim <= in.out->ndim, "input has more dims than output");
        for (int i = 0; i < in.a->ndim; ++i)
          TF_REQUIRE(in.a->shape[in.a->ndim - 1 - i] == in.out->shape[in.out->ndim - 1 - i],
                     "input must match the trailing dims of the output");
      }
      TF_REQUIRE(channels > 0 && inner > 0, "empty operand");
      s.inner = FastDiv((uint32_t)inner);
      s.channels = FastDiv((uint32_t)channels);
      for (int j = 0; j < k; ++j) TF_REQUIRE(g.s[j].out != s.a, "an operand that is spread cannot come from the group");
    } else {
      TF_REQUIRE((!has_a || same_shape(in.a, in.out)) && (!has_b || same_shape(in.b, in.out)), "shape mismatch");
      for (int j = 0; j < k; ++j) {  // the whole of what a step makes: lanes have no more of it
        if (has_a && g.s[j].out == s.a && g.s[j].n == m) s.from_a = j;
        if (has_b && g.s[j].out == s.b && g.s[j].n == m) s.from_b = j;
      }
      if (has_a && s.from_a < 0) fits(in.a);
      if (has_b && s.from_b < 0) fits(in.b);
    }
  }
  // what is read from memory is read at any time: nothing of the group may write it, nor two steps the same bytes
  for (int k = 0; k < n_steps; ++k)
    for (int j = 0; j < n_steps; ++j) {
      const Step &s = g.s[j];
      const float *out = g.s[k].out;
      const int64_t m = g.s[k].n;
      TF_REQUIRE(j == k || !overlap(out, m, s.out, s.n), "two steps write the same array");
      TF_REQUIRE(!s.a || s.from_a >= 0 || !overlap(out, m, s.a, numel(steps[j].a)), "a step writes what another one reads");
      TF_REQUIRE(!s.b || s.from_b >= 0 || !overlap(out, m, s.b, numel(steps[j].b)), "a step writes what another one reads");
    }
  if (n == 0) return 0;
  hipStream_t s = stream_of(stream);
  if (ordered && wait_for_other_streams(s) != 0) return -1;
  if (n == 1) vec = false;
  const dim3 grid((unsigned)cdiv(vec ? cdiv(n, 4) : n, kThreads)), block(kThreads);
  if (vec) hipLaunchKernelGGL(group_kernel<true>, grid, block, 0, s, g, (uint32_t)n);
  else hipLaunchKernelGGL(group_kernel<false>, grid, block, 0, s, g, (uint32_t)n);
  const int rc = finish(s, "DLGpuElementwiseGroup");
  if (ordered) order_others_behind(s);
  return rc;
}
