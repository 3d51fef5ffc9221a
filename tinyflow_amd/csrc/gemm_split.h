// The tile engine of gemm_core.h on the bf16 matrix instruction: fp32 in, fp32 out, for
// contractions whose time is the multiplications'.
//
// The fp32 matrix instruction runs at a sixteenth of the bf16 one's rate, so each fp32
// operand element is split into three bf16 numbers, x = h + m + l.  With every slice the
// nearest bf16 of what is left this is exact: h keeps 8 of the 24 significant bits, the rest
// x - h (exact in fp32) has at most 16 and a sign, m keeps 8 of those, and what then remains
// fits l.  A product of two elements is the sum of nine slice products; the engine
// computes the six largest,
//   h h'   and   (h m' + m h') + (m m' + h l' + l h'),
// each exact in the multiplier, accumulated in fp32 by v_mfma_f32_32x32x16_bf16.  What
// is left out (m l', l m', l l') is at most 2^-24 of the product, an fp32 rounding (|m| up to 2^-8, |l| up to 2^-17 of a value
// near 1; more than 2^-26 for one pair of random operands in 36).  Six such instructions for 16 reduction steps cost 192
// cycles where the eight fp32 ones cost 512.
//
// The h h' products and the smaller ones have accumulators of their own, added at the end: a sum of h h' is rounded
// once where the fp32 instruction rounds eight times, and the roundings of the others do not
// show.  (In one accumulator the instruction's own rounding adds up to a bias: error against float64 of
// 4096^3 from 8.1e-7 of the fp32 instruction to 9.4e-7, with two 3.2e-7; 256 x 64 x 200704: 1.05e-7, 1.08e-7, 4.1e-8.)
//
// Every element is multiplied by 2^23 before it is split, and the sums by 2^-46 at the end: all slices of every
// fp32 number, subnormal ones included, are then normal bf16 numbers.  (Unscaled, the slices below 2^-133 are lost: error
// against float64 of K = 264 with operands of 1e-36 2.7e-5, of 1e-40 0.26; scaled 6.7e-8, fp32 engine 2.9e-7.)
//
// Where the split does not hold - an infinity (its rest is not a number), a value or a sum that
// the scaling takes past the largest number (from 2^104 and 2^82 on) - some accumulator ends
// up infinite or NaN.  A workgroup that finds one computes its tile again with
// the fp32 instruction, so such problems have the results of a plain fp32 product.
//
// Operand tiles are fetched as in gemm_core.h, split in registers (thirteen vector
// instructions for two elements) and staged through
// double-buffered LDS as planes [slice][k / 8][row] of 16-byte units: a unit is the eight
// reduction elements that one lane feeds to one MFMA.  Per MFMA a lane supplies
// A[m = lane%32][k = 8*(lane/32) + 0..7], the same of B, and owns 16 accumulators
// D[8*(v/4) + 4*(lane/32) + v%4][lane%32], as with the fp32 instruction, so the epilogues are shared.
//
// What bounds it, for long reductions: power.  4096^3 runs at 195 to 205 TFLOP/s by card (fp32 engine: 137), with zeros for data
// at 300; the matrix instructions alone, out of LDS, at 324.  Short reductions (the 1x1 layers of a ResNet: 120 to 150) are
// bound by a tile's start and end, as long as 70 to 80 reduction steps and not overlapped with another tile's
// multiplications: the matrix pipes are busy in 0.3 to 0.5 of their cycles.  The work beside the matrix instructions counts:
// the splitting (104 of the 114 vector instructions
// of a 128 x 128 stage) sits between the matrix instructions, addresses are a lane's constant plus a scalar, and
// the LDS layouts have no bank conflicts.
#pragma once

#include "gemm_core.h"

namespace tf {
namespace gemm {
namespace split {

// ---- bf16 slices and their LDS planes ------------------------------------------------
typedef float f32x2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2v __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));

// Two fp32 values as two bf16 (nearest, ties to even): the first in the low half.
__device__ inline uint32_t pack_bf16(float a, float b) {
  const f32x2v v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
constexpr float kScale = 0x1p23f, kUnscale = 0x1p-46f;  // of an element, of a sum of products

// The three slices of two neighbouring reduction elements: thirteen instructions.
__device__ inline void split_pair(float a, float b, uint32_t (&slice)[3]) {
  a *= kScale;
  b *= kScale;
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    slice[s] = pack_bf16(a, b);
    if (s < 2) {
      a -= __builtin_bit_cast(float, slice[s] << 16);
      b -= __builtin_bit_cast(float, slice[s] & 0xffff0000u);
    }
  }
}

// LDS planes of one operand and one stage.  ROWS rows of the tile lie in VW blocks of
// ROWS / VW units, row d in block d % VW: a lane that fetched VW consecutive rows of one
// reduction index then writes to the same place of every block, next to its neighbour
// lanes (no bank conflict), and the padding between the blocks keeps eight lanes that
// read eight consecutive rows on distinct banks.
// The slices are SLICE bytes apart, the groups of eight reduction elements GROUP bytes.
template <int ROWS, int BK, int VW, int PAD>
struct Planes {
  static constexpr int BLOCK = ROWS / VW + PAD;  // units
  static constexpr int GROUP = (VW == 1 ? BLOCK : VW * BLOCK - PAD) * 16;
  static constexpr int SLICE = BK / 8 * GROUP;
  static constexpr int BYTES = 3 * SLICE;
  static __device__ inline int row(int d) { return ((d % VW) * BLOCK + d / VW) * 16; }
};

// N consecutive reduction elements (2, 4 or a multiple of 8, the first a multiple of N) of one row.
template <class P, int N>
__device__ inline void put_run(char *planes, int row_off, int k, const float *v) {
  static_assert(N == 2 || N == 4 || N % 8 == 0, "run length");
  uint32_t w[3][N / 2];
#pragma unroll
  for (int i = 0; i < N / 2; ++i) {
    uint32_t s[3];
    split_pair(v[2 * i], v[2 * i + 1], s);
#pragma unroll
    for (int q = 0; q < 3; ++q) w[q][i] = s[q];
  }
  char *at = planes + row_off + (k / 8) * P::GROUP + (k % 8) * 2;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    if constexpr (N == 2) {
      *reinterpret_cast<uint32_t *>(at + q * P::SLICE) = w[q][0];
    } else if constexpr (N == 4) {
      *reinterpret_cast<u32x2v *>(at + q * P::SLICE) = u32x2v{w[q][0], w[q][1]};
    } else {
#pragma unroll
      for (int g = 0; g < N / 8; ++g)
        *reinterpret_cast<u32x4v *>(at + q * P::SLICE + g * P::GROUP) =
            u32x4v{w[q][4 * g], w[q][4 * g + 1], w[q][4 * g + 2], w[q][4 * g + 3]};
    }
  }
}

// ---- loaders ----------------------------------------------------------------------------
// A loader fetches EPT elements of a D x BK operand tile per lane:
//   init(st, origin, tid)            the lane's part of the addresses; origin: first row of the tile
//   load(st, k0, k_limit, reg)       the stage that starts at k0; indices from k_limit on read as zero
//   put(st, planes, reg)             splits them into the LDS planes (its type Layout)
//   each(st, reg, f)                 f(k in the stage, row in the tile, value), for the fp32 pass
//
// "Along" lanes: the 256 lanes run along the tile's rows, every lane holds a run of
// consecutive reduction elements of one row, and one load instruction of a wave reads 64
// consecutive rows for a single, wave-uniform k.
template <int D, int BK>
struct AlongRuns {
  static_assert(D == 64 || D == 128, "tile extent");
  static constexpr int EPT = BK * D / THREADS;  // elements per lane per stage
  using Layout = Planes<D, BK, 1, 0>;
  int d_local;                               // position along the tile extent
  int k_first;                               // wave-uniform
  __device__ inline void init(int tid) {
    d_local = tid % D;
    k_first = __builtin_amdgcn_readfirstlane(tid / D) * EPT;
  }
  __device__ inline int k_of(int e) const { return k_first + e; }
  __device__ inline void put(char *planes, const float (&reg)[EPT]) const {
    put_run<Layout, EPT>(planes, Layout::row(d_local), k_first, reg);
  }
  template <class F>
  __device__ inline void each(const float (&reg)[EPT], F &&f) const {
#pragma unroll
    for (int e = 0; e < EPT; ++e) f(k_of(e), d_local, reg[e]);
  }
};

// "Across" lanes: BK / 4 lanes run along the reduction, the contiguous direction of
// the operand in memory, and every lane holds runs of four elements of EPT / 4 rows.
template <int D, int BK>
struct AcrossRuns {
  static constexpr int LPR = BK / 4;            // lanes per row of the tile
  static constexpr int DSTEP = THREADS / LPR;
  static constexpr int VPT = D / DSTEP;         // runs per lane per stage
  static constexpr int EPT = VPT * 4;
  static_assert(VPT >= 1 && VPT * DSTEP == D, "tile shape");
  using Layout = Planes<D, BK, 1, 128 / BK>;    // the lanes of one store cover every bank once
  int k_local;
  int d_first;
  __device__ inline void init(int tid) {
    k_local = (tid % LPR) * 4;
    d_first = tid / LPR;
  }
  __device__ inline int d_of(int e) const { return d_first + e * DSTEP; }
  __device__ inline void put(char *planes, const float (&reg)[EPT]) const {
#pragma unroll
    for (int e = 0; e < VPT; ++e) put_run<Layout, 4>(planes, Layout::row(d_of(e)), k_local, &reg[4 * e]);
  }
  template <class F>
  __device__ inline void each(const float (&reg)[EPT], F &&f) const {
#pragma unroll
    for (int e = 0; e < EPT; ++e) f(k_local + e % 4, d_of(e / 4), reg[e]);
  }
};

// ---- matrix operands: 8- and 16-byte loads ---------------------------------------------
// One load instruction per lane fetches several consecutive elements: a quarter of
// the load instructions and of the address arithmetic of one-element loads.
// Addressing is segmented so that the same two loaders serve plain
// matrices and the NCHW tensors of 1x1 / stride-1 convolutions (pixels of one image
// and channel are contiguous, images are `outer` elements apart):
//   SplitAlong4 :  element(d, k) = base[(d / inner) * outer + d % inner + k * ld]
//   SplitAcross4:  element(d, k) = base[d * ld + (k / inner) * outer + k % inner]
// A plain matrix is the case inner = 2^31 (one segment), outer = 0; an Across operand of one segment has
// SEGMENTS = false and no division per stage.
// `inner` is a multiple of 4 (or the whole extent); nothing else needs to be: such loads
// want no more than 4-byte alignment from global memory.
//
// Ragged segments: a segment whose real length is not a multiple of 4 (the 49 pixels
// of a 7x7 map) is addressed with `inner` rounded up to the next multiple of 4 while
// `outer` stays the real distance between segments.  The last vector of a segment, and
// that of a row of a matrix whose extent is no multiple of 4,
// then also fetches up to three elements that belong to what follows it in memory.
// For SplitAlong4 they land in
// tile rows that exist only in the padded index space, or past the extent, and are dropped by the
// epilogue; for SplitAcross4 they would enter the reduction, so its RAGGED form zeroes
// every element whose position in the segment is `seg_valid` or more.
__device__ inline f32x4v buf_load4_at(__amdgpu_buffer_rsrc_t r, uint32_t byte_off, uint32_t uniform_off) {
  return __builtin_bit_cast(f32x4v, __builtin_amdgcn_raw_buffer_load_b128(r, (int)byte_off, (int)uniform_off, 0));
}
__device__ inline f32x2v buf_load2_at(__amdgpu_buffer_rsrc_t r, uint32_t byte_off, uint32_t uniform_off) {
  return __builtin_bit_cast(f32x2v, __builtin_amdgcn_raw_buffer_load_b64(r, (int)byte_off, (int)uniform_off, 0));
}

template <int D, int BK>
struct SplitAlong4 {
  static constexpr bool kSplit = true;
  static constexpr int EPT = BK * D / THREADS;
  static constexpr int VW = EPT >= 8 ? 4 : 2;   // rows per load
  static constexpr int KPL = EPT / VW;          // consecutive reduction elements per lane
  static constexpr int LPU = 8 / KPL;           // lanes that share the units of VW rows
  static_assert(KPL == 2 || KPL == 4, "tile shape");
  using Layout = Planes<D, BK, VW, VW == 4 ? 4 : 8>;
  const float *base;
  uint32_t bytes;
  int ld, d_extent, k_extent;
  FastDiv div_inner;
  int outer;

  struct State {
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t d_off;       // byte offset of this lane's first d, or OOB
    uint32_t off[KPL];    // of its elements in the stage at k = 0
    int d_local, k_first;
  };
  __device__ inline void init(State &st, int origin, int tid) const {
    st.rsrc = make_rsrc(base, bytes);
    st.d_local = (tid / LPU) % (D / VW) * VW;
    st.k_first = tid / (LPU * D / VW) * 8 + (tid % LPU) * KPL;
    const int d = origin + st.d_local;
    uint32_t seg, rem;
    div_inner.divmod((uint32_t)(d < d_extent ? d : 0), seg, rem);
    st.d_off = d < d_extent ? (seg * (uint32_t)outer + rem) * 4u : OOB;
#pragma unroll
    for (int e = 0; e < KPL; ++e)
      st.off[e] = (st.d_off + (uint32_t)(st.k_first + e) * (uint32_t)ld * 4u) | (st.d_off & OOB);
  }
  __device__ inline void load(const State &st, int k0, int k_limit, float (&reg)[EPT]) const {
    const uint32_t stage_off = (uint32_t)min(k0, k_limit) * (uint32_t)ld * 4u;  // uniform, inside the buffer
#pragma unroll
    for (int e = 0; e < KPL; ++e) {
      const uint32_t off = st.k_first < k_limit - k0 - e ? st.off[e] : OOB;
      if constexpr (VW == 4) {
        const f32x4v v = buf_load4_at(st.rsrc, off, stage_off);
#pragma unroll
        for (int i = 0; i < 4; ++i) reg[i * KPL + e] = v[i];
      } else {
        const f32x2v v = buf_load2_at(st.rsrc, off, stage_off);
#pragma unroll
        for (int i = 0; i < 2; ++i) reg[i * KPL + e] = v[i];
      }
    }
  }
  __device__ inline void put(const State &st, char *planes, const float (&reg)[EPT]) const {
#pragma unroll
    for (int i = 0; i < VW; ++i)
      put_run<Layout, KPL>(planes, Layout::row(st.d_local) + i * Layout::BLOCK * 16, st.k_first, &reg[i * KPL]);
  }
  template <class F>
  __device__ inline void each(const State &st, const float (&reg)[EPT], F &&f) const {
#pragma unroll
    for (int e = 0; e < EPT; ++e) f(st.k_first + e % KPL, st.d_local + e / KPL, reg[e]);
  }
};

template <int D, int BK, bool RAGGED = false, bool SEGMENTS = false>
struct SplitAcross4 {
  using Map = AcrossRuns<D, BK>;
  using Layout = typename Map::Layout;
  static constexpr bool kSplit = true;
  static constexpr int EPT = Map::EPT;
  const float *base;
  uint32_t bytes;
  int ld, d_extent, k_extent;
  FastDiv div_inner;
  int outer;
  int seg_valid = 0;  // RAGGED: real length of a segment

  struct State {
    Map map;
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t row_off[Map::VPT];  // byte offset of (row d, first element of a stage at k = 0), or OOB
  };
  __device__ inline void init(State &st, int origin, int tid) const {
    st.rsrc = make_rsrc(base, bytes);
    st.map.init(tid);
#pragma unroll
    for (int e = 0; e < Map::VPT; ++e) {
      const int d = origin + st.map.d_of(e);
      st.row_off[e] = d < d_extent ? ((uint32_t)d * (uint32_t)ld + (uint32_t)st.map.k_local) * 4u : OOB;
    }
  }
  __device__ inline void load(const State &st, int k0, int k_limit, float (&reg)[EPT]) const {
    const int k = k0 + st.map.k_local;
    uint32_t seg = 0, rem = (uint32_t)k, lane_off = 0, stage_off = (uint32_t)min(k0, k_limit) * 4u;
    if (SEGMENTS) {
      div_inner.divmod((uint32_t)min(k, k_limit - 1), seg, rem);
      lane_off = (seg * (uint32_t)outer + rem - (uint32_t)st.map.k_local) * 4u;  // the row's offset holds k_local
      stage_off = 0;
    }
    const uint32_t k_bad = k < k_limit ? 0u : OOB;
#pragma unroll
    for (int e = 0; e < Map::VPT; ++e) {
      const uint32_t off = SEGMENTS ? (st.row_off[e] + lane_off) | (st.row_off[e] & OOB) | k_bad : st.row_off[e] | k_bad;
      const f32x4v v = buf_load4_at(st.rsrc, off, stage_off);
#pragma unroll
      for (int i = 0; i < 4; ++i) reg[4 * e + i] = (RAGGED && (int)rem + i >= seg_valid) ? 0.f : v[i];
    }
  }
  __device__ inline void put(const State &st, char *planes, const float (&reg)[EPT]) const { st.map.put(planes, reg); }
  template <class F>
  __device__ inline void each(const State &st, const float (&reg)[EPT], F &&f) const {
    st.map.each(reg, f);
  }
};

// ---- the kernel ----------------------------------------------------------------------
// Operands of many problems (the transformed domain) say so.
template <class L, class = void>
struct leaves_early : std::false_type {};
template <class L>
struct leaves_early<L, std::enable_if_t<L::kBatched>> : std::true_type {};

// Work decomposition, fold and epilogue are those of the fp32 kernel.
// Workgroups a CU: two of the 128 x 128 tile (its registers and no more).  Three of the 64 x 128 tile, whose LDS has room for
// them; left to itself the compiler takes six registers too many for the third (1x1, 256 -> 64 channels, 56 x 56, batch 64: 76 -> 66 us,
// 64 -> 256 104 -> 86, 512 -> 2048 at 7 x 7 54 -> 52).  LDS holds two of the 64 x 64 tile.
template <int BM, int BN, int BK, class ALoader, class BLoader, class Epilogue>
__global__ __launch_bounds__(THREADS, BM *BN == 128 * 128 ? 2 : BN == 128 ? 3 : 1) void gemm_kernel(const ALoader al, const BLoader bl, const Epilogue ep,
                                                      int k_extent, int k_per_split, int tiles_m, int tiles_n,
                                                      const Fold fold) {
  // four waves, 2 x 2 over the tile
  constexpr int WM = BM / 2, WN = BN / 2;  // wave tile
  constexpr int TM = WM / 32, TN = WN / 32;
  static_assert(TM >= 1 && TN >= 1, "tile too small for the wave grid");
  using PA = typename ALoader::Layout;
  using PB = typename BLoader::Layout;
  constexpr int LDA = BM + 4, LDB = BN + 4;  // rows of the fp32 pass's planes, floats
  __shared__ __align__(16) char lds[2 * (PA::BYTES + PB::BYTES)];
  __shared__ unsigned flag;
  constexpr int STAGE = PA::BYTES + PB::BYTES;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m_wave = wave % 2 * WM, n_wave = wave / 2 * WN;  // this wave's part of the tile

  const int tiles = tiles_m * tiles_n;
  const TileWork work = tile_work(bl, k_extent, k_per_split, tiles, fold);
  const int k_begin = work.k_begin, k_end = work.k_end;
  const int m0 = work.tile % tiles_m * BM, n0 = work.tile / tiles_m * BN;

  typename ALoader::State sa;
  typename BLoader::State sb;
  al.init(sa, m0, tid);
  bl.init(sb, n0, tid);

  f32x16 acc[TM][TN], low[TM][TN];  // sums of h h', and of everything smaller
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = low[i][j][v] = 0.f;

  // Two sets of fetched values: while a stage is multiplied, the next one (fetched during the stage before)
  // is split into the other planes and the one after it is on its way.
  float ra[2][ALoader::EPT], rb[2][BLoader::EPT];
  al.load(sa, k_begin, k_end, ra[0]);
  bl.load(sb, k_begin, k_end, rb[0]);
  al.load(sa, k_begin + BK, k_end, ra[1]);
  bl.load(sb, k_begin + BK, k_end, rb[1]);
  if (tid == 0) flag = 0u;
  // Transformed-domain products: a workgroup that fetches anything infinite or NaN for its first stage leaves its tile to the fp32 pass at
  // once, which for them keeps two stages in LDS and one chain of sums, as the fp32 kernel does.  VGG-16, batch 32, steps on nothing but
  // NaN: 18.2 ms with all of the slices' work before that pass and one stage in it, now 14.2, with the fp32 kernel 13.7; finite steps are
  // as fast as without the look.
  constexpr bool LEAVES = leaves_early<BLoader>::value;
  __shared__ unsigned lost[4];
  if (LEAVES) {
    float largest = 0.f;  // propagates NaN
#pragma unroll
    for (int e = 0; e < ALoader::EPT; ++e) largest = __builtin_elementwise_maximum(largest, __builtin_fabsf(ra[0][e]));
#pragma unroll
    for (int e = 0; e < BLoader::EPT; ++e) largest = __builtin_elementwise_maximum(largest, __builtin_fabsf(rb[0][e]));
    const bool any = __any(!(largest < __builtin_inff()));
    if (lane == 0) lost[wave] = any;
  }
  al.put(sa, lds, ra[0]);
  bl.put(sb, lds + PA::BYTES, rb[0]);
  __syncthreads();

  const int lhalf = lane >> 5;  // which eight of the sixteen reduction elements of an MFMA this lane feeds
  const int lcol = lane & 31;
  int a_off[TM], b_off[TN];     // this lane's units in the planes of the first stage
#pragma unroll
  for (int i = 0; i < TM; ++i) a_off[i] = lhalf * PA::GROUP + PA::row(m_wave + 32 * i + lcol);
#pragma unroll
  for (int j = 0; j < TN; ++j) b_off[j] = PA::BYTES + lhalf * PB::GROUP + PB::row(n_wave + 32 * j + lcol);

  // One stage out of the planes of buffer `cur`.  Past the end of the range every offset is
  // out of bounds, so the last fetches cost no memory traffic and the stage has no branch.
  auto stage = [&](auto cur_c, int k0) {
    constexpr int cur = decltype(cur_c)::value;
    al.load(sa, k0 + 2 * BK, k_end, ra[cur]);
    bl.load(sb, k0 + 2 * BK, k_end, rb[cur]);
    // keep the fetches ahead of the multiply: without this fence the scheduler
    // sinks them next to their use and their latency is no longer hidden
    __builtin_amdgcn_sched_barrier(0);
    const char *planes = lds + cur * STAGE;
#pragma unroll
    for (int g = 0; g < BK / 16; ++g) {
      bf16x8 a[3][TM], b[3][TN];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
          a[q][i] = *reinterpret_cast<const bf16x8 *>(planes + a_off[i] + q * PA::SLICE + 2 * g * PA::GROUP);
#pragma unroll
        for (int j = 0; j < TN; ++j)
          b[q][j] = *reinterpret_cast<const bf16x8 *>(planes + b_off[j] + q * PB::SLICE + 2 * g * PB::GROUP);
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0][i], b[0][j], acc[i][j], 0, 0, 0);
      constexpr int qa[5] = {0, 1, 1, 0, 2}, qb[5] = {1, 0, 1, 2, 0};
#pragma unroll
      for (int p = 0; p < 5; ++p)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            low[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[qa[p]][i], b[qb[p]][j], low[i][j], 0, 0, 0);
    }
    al.put(sa, lds + (cur ^ 1) * STAGE, ra[cur ^ 1]);
    bl.put(sb, lds + (cur ^ 1) * STAGE + PA::BYTES, rb[cur ^ 1]);
    // Interleave: the first matrix instructions need the highest slices only; the splitting of the next stage's
    // values (some 6.5 vector instructions an element) goes between the others, which leave the issue port free.  A sixth
    // of them first: 5x5 stride 2 layer with both gradients 144 us, with a third 149; groups of 9 an element on the 64 x 64
    // tile: 1000 x 1537 x 777 with both gradients 86 us, of 7 92, which the other tiles like better.
    constexpr int MFMAS = 6 * TM * TN * (BK / 16);
    constexpr int SPLIT = (BM == 64 && BN == 64 ? 9 : 7) * (ALoader::EPT + BLoader::EPT) + 8;
    constexpr int FIRST = MFMAS / 6, PER = (SPLIT + MFMAS - FIRST - 1) / (MFMAS - FIRST);
    __builtin_amdgcn_sched_group_barrier(0x100, 3 * (TM + TN), 0);
    __builtin_amdgcn_sched_group_barrier(0x008, FIRST, 0);
#pragma unroll
    for (int i = 0; i < MFMAS - FIRST; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, PER, 0);
      __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
  };
  const bool left = LEAVES && (lost[0] | lost[1] | lost[2] | lost[3]) != 0u;  // uniform
  if (left) flag = 1u;
  const int k_sliced = left ? k_begin : k_end;
  for (int k0 = k_begin; k0 < k_sliced; k0 += 2 * BK) {
    stage(std::integral_constant<int, 0>{}, k0);
    if (k0 + BK >= k_sliced) break;
    stage(std::integral_constant<int, 1>{}, k0 + BK);
  }

  // The split does not hold for infinities and on the way over the largest number: see the head of this file.
  {
    float largest = 0.f;  // propagates NaN
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        acc[i][j] += low[i][j];
#pragma unroll
        for (int v = 0; v < 16; v += 2)
          largest = __builtin_elementwise_maximum(
              __builtin_elementwise_maximum(largest, __builtin_fabsf(acc[i][j][v])), __builtin_fabsf(acc[i][j][v + 1]));
      }
    if (!(largest < __builtin_inff())) flag = 1u;
    __syncthreads();
    if (flag != 0u) {  // uniform over the workgroup
      constexpr int PASS = BK * (LDA + LDB);  // floats of a stage: [k][m], then [k][n]
      constexpr bool TWO = LEAVES;            // stages in LDS: one is multiplied while the next one is on its way
      constexpr int UNROLL = TWO ? 4 : 1;
      static_assert(2 * (PA::BYTES + PB::BYTES) >= (TWO ? 2 : 1) * PASS * 4, "the fp32 pass reuses the planes");
      float *const planes = reinterpret_cast<float *>(lds);
      auto fetch = [&](int k0) {
        al.load(sa, k0, k_end, ra[0]);
        bl.load(sb, k0, k_end, rb[0]);
      };
      auto put = [&](int at) {
        al.each(sa, ra[0], [&](int k, int d, float v) { planes[at + k * LDA + d] = v; });
        bl.each(sb, rb[0], [&](int k, int d, float v) { planes[at + BK * LDA + k * LDB + d] = v; });
      };
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
      if (TWO) {
        fetch(k_begin);
        put(0);
      }
      int at = 0;
#pragma unroll 1
      for (int k0 = k_begin; k0 < k_end; k0 += BK) {
        fetch(TWO ? k0 + BK : k0);
        if (!TWO) {
          __syncthreads();  // the stage before has been read
          put(0);
        }
        __syncthreads();
        // else a stage is summed apart: the rounding of one long chain would exceed that of the slices
        if (!TWO) {
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
              for (int v = 0; v < 16; ++v) low[i][j][v] = 0.f;
        }
        auto &sum = TWO ? acc : low;
        const float *const fa = planes + at + lhalf * LDA + m_wave + lcol;
        const float *const fb = planes + at + BK * LDA + lhalf * LDB + n_wave + lcol;
#pragma unroll UNROLL
        for (int k = 0; k < BK; k += 2)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
              sum[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[k * LDA + 32 * i], fb[k * LDB + 32 * j], sum[i][j], 0, 0, 0);
        if (TWO) {
          at = PASS - at;
          put(at);
        } else {
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] += low[i][j];
        }
      }
      __syncthreads();
    } else {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] *= kUnscale;
    }
  }

  // the flag is free again: every wave has passed a barrier since it was read
  write_tile<BM, BN, true>(acc, ep, work, tiles, fold, m0 + m_wave, n0 + n_wave, tid, flag);
}

}  // namespace split
}  // namespace gemm
}  // namespace tf
