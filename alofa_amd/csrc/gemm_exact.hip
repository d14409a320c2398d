// Matrix products of the 32-bit path: out[m, n] = sum_k A[m, k] * W[n, k], float operands, every product and every sum in
// float64 on the matrix cores (v_mfma_f64_16x16x4_f64), rounded to float once. W is stored [out, in].
//
// Lane l of the instruction holds A[row l % 16][k l / 16], B[k l / 16][column l % 16] and D[rows 4 v + l / 16, v = 0..3][column l % 16].
// Which four k an instruction takes is free as long as both operands agree, so a lane takes four consecutive k (one 16-byte
// load) for four instructions in a row.
//
// An output is bias + c0 + c1 + ...: K is cut into chains of 128 values and more, sixteen at most, by K alone; a chain's products are summed in ascending k, four by
// an instruction, and the chains' float64 sums are added in their order. Every form below does so, whichever wave or block has a chain: a row's
// result is the same bits whatever rows are computed with it.
//
//   up to 16 rows (exact_rows_kernel): a block owns 16 weight rows (16 to 24 of gate and as many of up), its waves take a chain each, in runs of 32 k
//   straight from memory, and meet in LDS. Bound by the rate at which a compute unit takes its weights in and, within it, by the matrix
//   cores (64 cycles an instruction, 64 weights), so the chains are dealt out over blocks where blocks are few. 8 rows, us, a tile of 64 x 64
//   on the vector units (one block per 64 columns) / this: 9,728 x 896 with the gate 270 / 14.9 (12.5 dealt out evenly, launch_exact_rows), 896 x 4,864 920 / 10.2 with the second
//   launch, 896 x 896 168 / 6.5, 1,152 x 896 170 / 6.5, 151,936 x 896 658 / 113.
//
//   more rows (exact_tile_kernel): slabs of 32 k through LDS, a wave owns 32 rows x 32 weight rows (four instructions for two
//   loads of either operand), a block 64 x 64 (32 x 128 up to 32 rows). Bound by the matrix cores (69 TFLOP/s measured with
//   nothing else in the loop; 58 reached, 50 of them useful at 450 rows, whose last tile is padding) and by the widening, which the same SIMD does between the
//   products. Two slabs are on their way in registers and two lie in LDS: with one of either, a slab that came late (1.4 us from a busy memory against 0.9 us of
//   products) held up the block, 9,728 x 896 with the gate 167, 896 x 4,864 102 + 5. The chains are dealt out over blocks where the tiles are few; their float64 sums
//   go to a buffer of the caller's (not to the library's workspace, which one stream at a time may use) and a second launch adds them. Else a block adds them up in
//   registers, two blocks to a compute unit where three fit without. 450 rows, us, as above: 9,728 x 896 with the gate 377 / 154, 896 x 4,864 1,000 / 89 both launches,
//   896 x 896 185 / 30, 1,152 x 896 185 / 31. (With shares of K by the number of rows 84, 26 and 31: then a row's sums depend on the others. A block that takes several chains
//   of few, each to its own place: 89, 31, 31.)
#include "common.h"

#include <algorithm>
#include <type_traits>

namespace alofa {

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int kExactStore = 0, kExactResidual = 1;
constexpr int kExactRows = 16;       // rows that exact_rows_kernel takes at most
constexpr int kMaxChains = 16;       // chains that K is cut into at most, and exact_sum_kernel adds
constexpr int64_t kMostBytes = int64_t{64} << 20;      // of the chains' sums in memory

// four consecutive k of a row from `k` on, all of them within the row: one 16-byte load, or, where rows are not 16-byte aligned, value by value
template <bool kVec>
__device__ __forceinline__ float4 quad(const float* row, int k) {
  if constexpr (kVec) return *reinterpret_cast<const float4*>(row + k);
  else return make_float4(row[k], row[k + 1], row[k + 2], row[k + 3]);
}
// the same with zeros beyond K
template <bool kVec>
__device__ __forceinline__ float4 quad_within(const float* row, int k, int K) {
  if constexpr (kVec) return k < K ? quad<kVec>(row, k) : make_float4(0.f, 0.f, 0.f, 0.f);
  else return make_float4(k < K ? row[k] : 0.f, k + 1 < K ? row[k + 1] : 0.f, k + 2 < K ? row[k + 2] : 0.f, k + 3 < K ? row[k + 3] : 0.f);
}

__device__ __forceinline__ f64x4 fma_quad(float4 a, float4 b, f64x4 acc) {
  acc = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(a.x), static_cast<double>(b.x), acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(a.y), static_cast<double>(b.y), acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(a.z), static_cast<double>(b.z), acc, 0, 0, 0);
  return __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(a.w), static_cast<double>(b.w), acc, 0, 0, 0);
}

template <int kEpilogue>
__device__ __forceinline__ void put(float* dst, double sum) {
  const float v = static_cast<float>(sum);
  *dst = kEpilogue == kExactResidual ? *dst + v : v;
}

// both products are rounded to float first, then the activation and the product in float64
__device__ __forceinline__ float gated(double g, double u, int gelu) {
  return static_cast<float>(gate_of(static_cast<double>(static_cast<float>(g)), gelu != 0) * static_cast<double>(static_cast<float>(u)));
}

// How K is cut into chains (see the head of this file): `count` of them, `length` values each, the last one what is left. By K alone.
struct Cut {
  int length, count;
};
static Cut cut_of(int K) {
  const int length = std::max(128, ((K + kMaxChains - 1) / kMaxChains + 63) / 64 * 64);
  return {length, (K + length - 1) / length};
}

// NW waves; kMats = 2: gate and up. NT tiles of 16 weight rows a block (of each matrix). blockIdx.y: which `per` chains; parts, where those are not all: the chains' sums, [chain][M][N].
// kDealt > 0 (gate and up): a block owns `own` outputs, the rows of gate and then those of up side by side in kDealt tiles: see launch_exact_rows.
template <int NW, int NT, int kMats, int kEpilogue, bool kVec, int kDealt = 0>
__global__ void __launch_bounds__(64 * NW) exact_rows_kernel(float* __restrict__ out, int64_t ldo, const float* __restrict__ A, int64_t lda,
                                                             const float* __restrict__ W, const float* __restrict__ W2, int64_t ldw,
                                                             const float* __restrict__ bias, double* __restrict__ parts, Cut cut, int per, int M, int N, int K, int gelu, int own = 0) {
  constexpr int kTiles = kDealt ? kDealt : NT * kMats, kOut = kDealt ? (kDealt * 128 + 64 * NW - 1) / (64 * NW) : (NT * 256 + 64 * NW - 1) / (64 * NW);
  __shared__ double sums[NW][kTiles][4][64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, r = lane % 16, g = lane / 16;
  const int n0 = blockIdx.x * (kDealt ? own : 16 * NT);
  const bool row_ok = r < M;
  const float* a_row = A + static_cast<int64_t>(row_ok ? r : 0) * lda;
  const float* w_row[kTiles];
#pragma unroll
  for (int t = 0; t < kTiles; ++t) {
    if constexpr (kDealt) {
      const int q = min(t * 16 + r, 2 * own - 1), n = n0 + (q < own ? q : q - own);
      w_row[t] = (q < own ? W : W2) + static_cast<int64_t>(n < N ? n : N - 1) * ldw;
    } else {
      const int n = n0 + (t / kMats) * 16 + r;
      w_row[t] = (t % kMats ? W2 : W) + static_cast<int64_t>(n < N ? n : N - 1) * ldw;      // (rows beyond N: the last one again, not stored)
    }
  }
  // what this thread adds up: output o is place i = threadIdx.x + 64 NW o: tile, weight row 4 v + g', row of A j: (v, 16 g' + j)
  auto place = [&](int o, int& tile, int& v, int& at, int& m, int& n) __attribute__((always_inline)) {
    const int i = threadIdx.x + 64 * NW * o;
    if constexpr (kDealt) {      // (of gate's row: up's is `own` rows on)
      const int q = i / 16;
      tile = q / 16, v = q / 4 % 4, m = i % 16, at = q % 4 * 16 + m, n = n0 + q;
      return q < own && m < M && n < N;
    }
    tile = i / 256, v = i / 64 % 4, at = i % 64, m = at % 16, n = n0 + tile * 16 + 4 * v + at / 16;
    return i < NT * 256 && m < M && n < N;
  };
  double total[kOut][kMats];
#pragma unroll
  for (int o = 0; o < kOut; ++o) {
    int tile, v, at, m, n;
    const bool ok = place(o, tile, v, at, m, n);
#pragma unroll
    for (int x = 0; x < kMats; ++x) total[o][x] = ok && bias ? static_cast<double>(bias[n]) : 0.0;
  }
  const int from = blockIdx.y * per, last = min(from + per, cut.count);
  for (int first = from; first < last; first += NW) {      // the next NW chains, one a wave
    f64x4 acc[kTiles];
#pragma unroll
    for (int t = 0; t < kTiles; ++t) acc[t] = f64x4{0, 0, 0, 0};
    const int begin = (first + wave) * cut.length, end = first + wave < last ? min(begin + cut.length, K) : begin;
    // Runs of 32 k: a lane takes 4 g .. 4 g + 3 of either half (an instruction's lanes fetch 64 bytes of a row side by side). Two runs are on their
    // way or in work; each set of registers is filled again as soon as its run is multiplied, without a branch around the loads (in the last round of them a run past
    // the last is the last one again), so that the compiler waits for the oldest only.
    constexpr int kSets = 2;
    const int runs = end > begin ? (end - begin) / 32 : 0;
    float4 a[kSets][2], w[kSets][kTiles][2];
    auto fetch = [&](int s, int i) __attribute__((always_inline)) {
      const int k = begin + (i < runs ? i : runs - 1) * 32 + g * 4;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        a[s][h] = quad<kVec>(a_row, k + 16 * h);
#pragma unroll
        for (int t = 0; t < kTiles; ++t) w[s][t][h] = quad<kVec>(w_row[t], k + 16 * h);
      }
    };
    auto multiply = [&](int s) __attribute__((always_inline)) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (!row_ok) a[s][h] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int t = 0; t < kTiles; ++t) acc[t] = fma_quad(w[s][t][h], a[s][h], acc[t]);
      }
    };
    if (runs > 0) {
#pragma unroll
      for (int s = 0; s < kSets; ++s) fetch(s, s);
      int i = 0;
      for (; i + kSets < runs; i += kSets)
#pragma unroll
        for (int s = 0; s < kSets; ++s) {
          multiply(s);
          fetch(s, i + kSets + s);
        }
#pragma unroll
      for (int s = 0; s < kSets; ++s)
        if (i + s < runs) multiply(s);
    }
    for (int k = begin + runs * 32; k < end; k += 16) {      // what is left of K beyond the whole runs
      const float4 left = row_ok ? quad_within<kVec>(a_row, k + g * 4, K) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int t = 0; t < kTiles; ++t) acc[t] = fma_quad(quad_within<kVec>(w_row[t], k + g * 4, K), left, acc[t]);
    }
    if (first > from) __syncthreads();      // (the chains before have been added up)
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) sums[wave][t][v][lane] = acc[t][v];
    __syncthreads();
#pragma unroll
    for (int o = 0; o < kOut; ++o) {
      int tile, v, at, m, n;
      const bool ok = place(o, tile, v, at, m, n);
      if (!ok) continue;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        if (first + w >= last) break;      // (uniform)
#pragma unroll
        for (int x = 0; x < kMats; ++x) {
          const int up = n - n0 + own;
          const double sum = !kDealt ? sums[w][tile * kMats + x][v][at] : x == 0 ? sums[w][tile][v][at] : sums[w][up / 16][up / 4 % 4][up % 4 * 16 + m];
          if (parts) parts[(static_cast<int64_t>(first + w) * M + m) * N + n] = sum;
          else total[o][x] += sum;
        }
      }
    }
  }
  if (parts) return;
#pragma unroll
  for (int o = 0; o < kOut; ++o) {
    int tile, v, at, m, n;
    if (!place(o, tile, v, at, m, n)) continue;
    float* dst = out + static_cast<int64_t>(m) * ldo + n;
    if constexpr (kMats == 2) *dst = gated(total[o][0], total[o][1], gelu);
    else put<kEpilogue>(dst, total[o][0]);
  }
}

// A block of WM x (4 / WM) waves, each 16 RF rows x 32 weight rows; kMats = 2: the weight rows of a wave are 16 of gate and the same 16 of up.
// kFold: the block takes all chains and adds them up; else chain blockIdx.z, whose sums go to parts, [chain][M][N], and the epilogue is the second launch's.
template <int WM, int RF, int kMats, int kEpilogue, bool kVec, bool kFold>
__global__ void __launch_bounds__(256, WM == 2 && !kFold ? 3 : 2) exact_tile_kernel(float* __restrict__ out, int64_t ldo, const float* __restrict__ A, int64_t lda,
                                                         const float* __restrict__ W, const float* __restrict__ W2, int64_t ldw,
                                                         const float* __restrict__ bias, double* __restrict__ parts, Cut cut, int M, int N, int K, int gelu) {
  constexpr int WN = 4 / WM, BM = 16 * RF * WM, BW = 32 * WN, BK = 32, kPad = 4;
  constexpr int kOwn = 32 / kMats;                     // outputs of a wave along N
  __shared__ __attribute__((aligned(16))) float As[2][BM][BK + kPad], Ws[2][BW][BK + kPad];      // (as doubles, widened once as they are brought: 174 us where this took 169)
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, r = lane % 16, g = lane / 16;
  const int wm = wave / WN, wn = wave % WN;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * WN * kOwn;
  constexpr int kA = BM * BK / 4 / 256, kW = BW * BK / 4 / 256;      // quads a thread brings of either operand
  const float *a_row[kA], *w_row[kW];      // (rows past the end: the last one again, its results are not stored)
#pragma unroll
  for (int i = 0; i < kA; ++i) {
    const int m = m0 + (threadIdx.x + i * 256) / 8;
    a_row[i] = A + static_cast<int64_t>(m < M ? m : M - 1) * lda;
  }
#pragma unroll
  for (int i = 0; i < kW; ++i) {
    const int row = (threadIdx.x + i * 256) / 8, n = n0 + row / 32 * kOwn + row % kOwn;
    w_row[i] = (kMats == 2 && row % 32 >= 16 ? W2 : W) + static_cast<int64_t>(n < N ? n : N - 1) * ldw;
  }
  const int k_own = threadIdx.x % 8 * 4;      // (threadIdx.x + 256 i has the same place in its row)
  const int k_begin = kFold ? 0 : blockIdx.z * cut.length, k_end = kFold ? K : min(k_begin + cut.length, K);
  static_assert(kFold || kMats == 1, "gate and up meet in the block");
  f64x4 acc[RF][2], sum[RF][2];      // [rows of A][weight rows]: of this chain, of the chains before (kFold)
#pragma unroll
  for (int i = 0; i < RF; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = sum[i][j] = f64x4{0, 0, 0, 0};
  if constexpr (kFold && kMats == 1)
    if (bias) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int n = n0 + wn * 32 + j * 16 + r;
        const double b = n < N ? bias[n] : 0.0;
#pragma unroll
        for (int i = 0; i < RF; ++i) sum[i][j] = f64x4{b, b, b, b};
      }
    }
  auto end_chain = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < RF; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) sum[i][j] += acc[i][j], acc[i][j] = f64x4{0, 0, 0, 0};
  };
  // Two slabs in registers, on their way, while a third is worked on: a slab comes in some 1.4 us when the chip is busy, and its own products last 0.9.
  // (The loads of whole slabs are issued whatever the thread: under a condition each would be waited for by itself.)
  float4 fa[2][kA], fw[2][kW];
  auto fetch = [&](auto set, int slab) __attribute__((always_inline)) {
    constexpr int x = decltype(set)::value;
#pragma unroll
    for (int i = 0; i < kA; ++i) fa[x][i] = quad<kVec>(a_row[i], k_begin + slab * BK + k_own);
#pragma unroll
    for (int i = 0; i < kW; ++i) fw[x][i] = quad<kVec>(w_row[i], k_begin + slab * BK + k_own);
  };
  auto keep = [&](auto set) __attribute__((always_inline)) {
    constexpr int x = decltype(set)::value;
#pragma unroll
    for (int i = 0; i < kA; ++i) *reinterpret_cast<float4*>(&As[x][(threadIdx.x + i * 256) / 8][k_own]) = fa[x][i];
#pragma unroll
    for (int i = 0; i < kW; ++i) *reinterpret_cast<float4*>(&Ws[x][(threadIdx.x + i * 256) / 8][k_own]) = fw[x][i];
  };
  auto multiply = [&](auto set) __attribute__((always_inline)) {
    constexpr int x = decltype(set)::value;
#pragma unroll
    for (int q = 0; q < BK / 16; ++q) {
      float4 a[RF], w[2];
#pragma unroll
      for (int i = 0; i < RF; ++i) a[i] = *reinterpret_cast<const float4*>(&As[x][(wm * RF + i) * 16 + r][q * 16 + g * 4]);
#pragma unroll
      for (int i = 0; i < 2; ++i) w[i] = *reinterpret_cast<const float4*>(&Ws[x][wn * 32 + i * 16 + r][q * 16 + g * 4]);
#pragma unroll
      for (int i = 0; i < RF; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = fma_quad(a[i], w[j], acc[i][j]);
    }
  };
  int left = cut.length / (2 * BK);      // pairs of slabs of this chain
  auto end_pair = [&]() __attribute__((always_inline)) {
    if constexpr (kFold)
      if (--left == 0) {      // (uniform)
        end_chain();
        left = cut.length / (2 * BK);
      }
  };
  // (two slabs in LDS: a slab's place is written again two barriers after the barrier behind which it is read)
  auto step = [&](auto set, int slab, auto more) __attribute__((always_inline)) {
    keep(set);
    if constexpr (decltype(more)::value) fetch(set, slab + 2);
    __syncthreads();
    multiply(set);
  };
  constexpr std::integral_constant<int, 0> first{};
  constexpr std::integral_constant<int, 1> second{};
  constexpr std::true_type more{};
  constexpr std::false_type done{};
  const int whole = (k_end - k_begin) / BK;
  if (whole > 0) fetch(first, 0);
  if (whole > 1) fetch(second, 1);
  int slab = 0;
  for (; slab + 3 < whole; slab += 2) {
    step(first, slab, more);
    step(second, slab + 1, more);
    end_pair();
  }
  if (whole - slab == 3) {
    step(first, slab, more);
    step(second, slab + 1, done);
    end_pair();
    step(first, slab + 2, done);
  } else if (whole - slab == 2) {
    step(first, slab, done);
    step(second, slab + 1, done);
    end_pair();
  } else if (whole - slab == 1) {
    step(first, slab, done);
  }
  if (k_begin + whole * BK < k_end) {      // the last k, fewer than a slab
#pragma unroll
    for (int i = 0; i < kA; ++i) fa[0][i] = quad_within<kVec>(a_row[i], k_begin + whole * BK + k_own, k_end);
#pragma unroll
    for (int i = 0; i < kW; ++i) fw[0][i] = quad_within<kVec>(w_row[i], k_begin + whole * BK + k_own, k_end);
    __syncthreads();
    keep(first);
    __syncthreads();
    multiply(first);
  }
  end_chain();      // (the last one; zeros where its end was a pair's)
  // D: rows of A 4 v + g, weight row r
#pragma unroll
  for (int i = 0; i < RF; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int m = m0 + (wm * RF + i) * 16 + 4 * v + g;
      if (m >= M) continue;
      if constexpr (kMats == 2) {
        const int n = n0 + wn * 16 + r;
        if (n < N) out[static_cast<int64_t>(m) * ldo + n] = gated(sum[i][0][v], sum[i][1][v], gelu);
      } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int n = n0 + wn * 32 + j * 16 + r;
          if (n >= N) continue;
          if constexpr (kFold) put<kEpilogue>(out + static_cast<int64_t>(m) * ldo + n, sum[i][j][v]);
          else parts[(static_cast<int64_t>(blockIdx.z) * M + m) * N + n] = sum[i][j][v];
        }
      }
    }
}

// The chains' sums in their order, then the epilogue.
template <int kEpilogue>
__global__ void __launch_bounds__(256) exact_sum_kernel(float* __restrict__ out, int64_t ldo, const double* __restrict__ parts, const float* __restrict__ bias,
                                                        int M, int N, int chains) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x, all = static_cast<int64_t>(M) * N;
  if (i >= all) return;
  const int n = i % N;
  double s = bias ? static_cast<double>(bias[n]) : 0.0;
  double p[kMaxChains];
#pragma unroll
  for (int x = 0; x < kMaxChains; ++x) p[x] = parts[(x < chains ? x : 0) * all + i];
#pragma unroll
  for (int x = 0; x < kMaxChains; ++x)
    if (x < chains) s += p[x];
  put<kEpilogue>(out + i / N * ldo + n, s);
}

// The same behind a product that adds to the residual stream, and the RMSNorm that follows: a block per row adds its chains up, writes the stream's new row and leaves it normed (w, eps, float64) in
// `normed` [M, N] rows, the bits that exact_sum_kernel and rmsnorm_kernel leave one behind the other (the squares in that kernel's order). K4: groups of four columns a thread, N at most 1,024 K4.
// A launch less; us in captured runs, launch by launch / this: 896 x 4,864 against one row 9.8 / 9.1, eight 10.9 / 10.0, 64 22.5 / 20.7, 450 91 / 89; 896 x 896 against 8 rows 7.6 / 7.5
// (which is cut over blocks for it), 64 13.2 / 11.9, 450 32.2 / 30.3.
template <int K4>
__global__ void __launch_bounds__(256) exact_sum_norm_kernel(float* __restrict__ out, int64_t ldo, const double* __restrict__ parts, const float* __restrict__ w, float eps,
                                                             float* __restrict__ normed, int64_t rows_out, int M, int N, int chains) {
  __shared__ double scratch[4];
  const int m = blockIdx.x, groups = N / 4;
  const int64_t all = static_cast<int64_t>(M) * N;
  float* row = out + static_cast<int64_t>(m) * ldo;
  float4 xs[K4], ws[K4];
  double ss = 0;
#pragma unroll
  for (int i = 0; i < K4; ++i) {
    const int g = threadIdx.x + 256 * i, at = 4 * (g < groups ? g : 0);      // (every thread loads; what lies beyond the row is cleared)
    const double2* p = reinterpret_cast<const double2*>(parts + static_cast<int64_t>(m) * N + at);
    const float4 old = *reinterpret_cast<const float4*>(row + at);
    ws[i] = *reinterpret_cast<const float4*>(w + at);
    double2 lo[kMaxChains], hi[kMaxChains];
#pragma unroll
    for (int x = 0; x < kMaxChains; ++x) lo[x] = p[(x < chains ? x : 0) * (all / 2)], hi[x] = p[(x < chains ? x : 0) * (all / 2) + 1];
    double a = 0, b = 0, c = 0, d = 0;
#pragma unroll
    for (int x = 0; x < kMaxChains; ++x)
      if (x < chains) a += lo[x].x, b += lo[x].y, c += hi[x].x, d += hi[x].y;
    xs[i] = g < groups ? make_float4(old.x + static_cast<float>(a), old.y + static_cast<float>(b), old.z + static_cast<float>(c), old.w + static_cast<float>(d)) : make_float4(0.f, 0.f, 0.f, 0.f);
    if (g < groups) *reinterpret_cast<float4*>(row + at) = xs[i];
  }
#pragma unroll
  for (int i = 0; i < K4; ++i) {
    const double a = xs[i].x, b = xs[i].y, c = xs[i].z, d = xs[i].w;
    ss += a * a;
    ss += b * b;
    ss += c * c;
    ss += d * d;
  }
  ss = block_sum<double, 256>(ss, scratch);
  const double scale = 1.0 / sqrt(ss / static_cast<double>(N) + static_cast<double>(eps));
  float* dst = normed + static_cast<int64_t>(m) * rows_out;
#pragma unroll
  for (int i = 0; i < K4; ++i) {
    const int g = threadIdx.x + 256 * i;
    if (g < groups)
      *reinterpret_cast<float4*>(dst + 4 * g) = make_float4(static_cast<float>(static_cast<double>(xs[i].x) * scale * static_cast<double>(ws[i].x)), static_cast<float>(static_cast<double>(xs[i].y) * scale * static_cast<double>(ws[i].y)),
                                                            static_cast<float>(static_cast<double>(xs[i].z) * scale * static_cast<double>(ws[i].z)), static_cast<float>(static_cast<double>(xs[i].w) * scale * static_cast<double>(ws[i].w)));
  }
}

// Up to 16 rows: chains a block takes. Four where the blocks of 16 weight rows are fewer than half the compute units and the chains more than a block's eight
// waves, else all of them.
// With a norm behind the sum there is a second launch either way: blocks of four chains from five chains on.
static int chains_per_block(int N, const Cut& cut, bool norm) { return cut.count > (norm ? 4 : 8) && (N + 15) / 16 * 2 < compute_units() ? 4 : cut.count; }

// The norm behind a product (null weights: none).
struct ExactNorm {
  const float* w;
  float eps;
  float* rows;
  int64_t ld;
};

// More rows: whether the chains are dealt out over blocks, for the least time of the compute unit that has the most blocks: 35.5 ns a k of a block (30 of them its SIMDs'
// matrix cores) and some 0.5 us a block, a twentieth more with one block to a compute unit, and for the second launch 4 us and 0.7 us a million sums.
// Not where the sums of 64 rows are more than kMostBytes.
static bool chains_apart(int M, int N, int K, const Cut& cut) {
  if (static_cast<int64_t>(cut.count) * N * std::min(M, 64) * 8 > kMostBytes) return false;
  const int BM = M <= 32 ? 32 : 64, BW = M <= 32 ? 128 : 64, cus = compute_units();
  const int64_t tiles = static_cast<int64_t>((M + BM - 1) / BM) * ((N + BW - 1) / BW);
  auto us = [&](int64_t blocks, int k) { const int64_t rounds = (blocks + cus - 1) / cus; return rounds * (0.0355 * k + 0.5) * (rounds == 1 ? 1.05 : 1.0); };
  return cut.count > 1 && us(tiles * cut.count, cut.length) + 4.0 + 0.7e-6 * cut.count * M * N < us(tiles, K);
}

// Rows that one launch takes where the chains' sums go to memory, in whole tiles.
static int rows_at_once(int M, int N, const Cut& cut) {
  const int64_t most = kMostBytes / (static_cast<int64_t>(cut.count) * N * 8);
  return M <= most ? M : static_cast<int>(most / 64 * 64);
}

template <int kEpilogue>
static void launch_exact_sum(float* out, int64_t ldo, const double* parts, const float* bias, int M, int N, int chains, const ExactNorm& norm, hipStream_t stream) {
  const int64_t all = static_cast<int64_t>(M) * N;
  if (norm.w) {      // (N a multiple of four, aligned rows: alofa_gemm_exact_norm sees to it)
    if (N <= 1024) exact_sum_norm_kernel<1><<<M, 256, 0, stream>>>(out, ldo, parts, norm.w, norm.eps, norm.rows, norm.ld, M, N, chains);
    else if (N <= 2048) exact_sum_norm_kernel<2><<<M, 256, 0, stream>>>(out, ldo, parts, norm.w, norm.eps, norm.rows, norm.ld, M, N, chains);
    else exact_sum_norm_kernel<4><<<M, 256, 0, stream>>>(out, ldo, parts, norm.w, norm.eps, norm.rows, norm.ld, M, N, chains);
    return;
  }
  exact_sum_kernel<kEpilogue><<<static_cast<unsigned>((all + 255) / 256), 256, 0, stream>>>(out, ldo, parts, bias, M, N, chains);
}

// Up to 16 rows: blocks of eight waves; two tiles of weight rows and four waves a block against a matrix as long as a vocabulary, so that the rows of A are read half as
// often (8 rows, 151,936 x 896: 113 us; four tiles 130, eight waves 143). Gate and up: where their tiles of 16 outputs are more than the compute units but no more than one and a half times as many, a
// compute unit with two blocks had up to twice the others' work (what it brings in, 37 bytes a nanosecond, and 64 cycles for each float64 instruction). There the outputs are dealt out evenly, 17 to 24 a block, in three tiles
// that hold gate's rows and then up's (a fourth would be the two blocks' work again). us, blocks of sixteen / dealt out, 1, 8, 16 rows: 4,864 x 896 15.1, 15.4, 16.0 / 12.6, 12.5, 13.0; 5,632 x 2,048
// 28.4, 30.2, 31.7 / 25.0, 25.4, 26.7; 4,352 x 1,024 15.9, 16.2, 17.0 / 13.1, 13.2, 14.0; 6,144 x 1,024 16.3, 16.6, 17.5 / 15.1, 15.2, 15.6. The bits do not change: a sum's chains are cut by K alone.
template <int kMats, int kEpilogue, bool kVec>
static int launch_exact_rows(float* out, int64_t ldo, const float* A, int64_t lda, const float* W, const float* W2, int64_t ldw, const float* bias,
                             double* parts, int M, int N, int K, int gelu, const ExactNorm& norm, hipStream_t stream) {
  const Cut cut = cut_of(K);
  const int tiles = (N + 15) / 16;
  if (kMats == 1 && chains_per_block(N, cut, norm.w != nullptr) < cut.count) {
    exact_rows_kernel<4, 1, 1, kEpilogue, kVec><<<dim3(tiles, (cut.count + 3) / 4), 256, 0, stream>>>(out, ldo, A, lda, W, W2, ldw, bias, parts, cut, 4, M, N, K, gelu);
    launch_exact_sum<kEpilogue>(out, ldo, parts, bias, M, N, cut.count, norm, stream);
  } else if (kMats == 1 && tiles >= 16 * compute_units()) {
    exact_rows_kernel<4, 2, 1, kEpilogue, kVec><<<(tiles + 2 - 1) / 2, 64 * 4, 0, stream>>>(out, ldo, A, lda, W, W2, ldw, bias, nullptr, cut, cut.count, M, N, K, gelu);
  } else if (const int units = compute_units(); kMats == 2 && tiles > units && 2 * tiles <= 3 * units) {
    const int own = (N + units - 1) / units;      // (17 to 24)
    exact_rows_kernel<8, 1, kMats, kEpilogue, kVec, kMats == 2 ? 3 : 0><<<(N + own - 1) / own, 512, 0, stream>>>(out, ldo, A, lda, W, W2, ldw, bias, nullptr, cut, cut.count, M, N, K, gelu, own);
  } else {
    exact_rows_kernel<8, 1, kMats, kEpilogue, kVec><<<tiles, 512, 0, stream>>>(out, ldo, A, lda, W, W2, ldw, bias, nullptr, cut, cut.count, M, N, K, gelu);
  }
  return check_launch("gemm_exact_rows");
}

template <int WM, int RF, int kMats, int kEpilogue, bool kVec>
static int launch_exact_tile(float* out, int64_t ldo, const float* A, int64_t lda, const float* W, const float* W2, int64_t ldw, const float* bias,
                             double* parts, int M, int N, int K, int gelu, const ExactNorm& norm, hipStream_t stream) {
  constexpr int BM = 16 * RF * WM, kOut = 32 * (4 / WM) / kMats;
  const Cut cut = cut_of(K);
  if constexpr (kMats == 1) {
    if (chains_apart(M, N, K, cut)) {
      const int at_once = rows_at_once(M, N, cut);
      for (int m = 0; m < M; m += at_once) {
        const int rows = std::min(at_once, M - m);
        float* dst = out + static_cast<int64_t>(m) * ldo;
        exact_tile_kernel<WM, RF, 1, kEpilogue, kVec, false><<<dim3((N + kOut - 1) / kOut, (rows + BM - 1) / BM, cut.count), 256, 0, stream>>>(
            nullptr, 0, A + static_cast<int64_t>(m) * lda, lda, W, W2, ldw, bias, parts, cut, rows, N, K, gelu);
        launch_exact_sum<kEpilogue>(dst, ldo, parts, bias, rows, N, cut.count, norm.w ? ExactNorm{norm.w, norm.eps, norm.rows + static_cast<int64_t>(m) * norm.ld, norm.ld} : norm, stream);
      }
      return check_launch("gemm_exact_tile");
    }
  }
  exact_tile_kernel<WM, RF, kMats, kEpilogue, kVec, true><<<dim3((N + kOut - 1) / kOut, (M + BM - 1) / BM), 256, 0, stream>>>(out, ldo, A, lda, W, W2, ldw, bias, nullptr, cut, M, N, K, gelu);
  return check_launch("gemm_exact_tile");
}

// Gate and up of more than 64 rows: whether tiles of 96 rows come out sooner than those of 64. A compute unit takes a round's time for each of its blocks, whether they lie side by side or not, so it is
// the whole rounds that count, and a block of 96 rows (56 of whose registers are kept in memory) takes 1.55 times what one of 64 takes (31.5 us against K of 896). us, 64 / 96 rows a block, by their rounds:
// 2 and 1, 66 rows of 4,864 x 896 64.9 / 51; 5 and 3, 96 of 18,944 x 1,536 1.10 times as fast; 11 and 7, 480 of 11,008 x 1,536 1.03; 3 and 2 of 64: 65 of 8,960 x 128 19.6 / 20.9, 96 of 8,960 x 896
// 97.7 / 100.6, 240 of 4,864 x 3,584 357 / 371 (K from 128 to 5,120, 69 sizes: at the median 0.98 times as fast); 6 and 4 0.985; 3 and 3, 300 of 4,864 x 896 96 / 142.
static bool taller_tiles(int M, int N) {
  if (M <= 64) return false;
  const int64_t columns = (N + 31) / 32, cus = compute_units();
  auto rounds = [&](int rows) { return (columns * ((M + rows - 1) / rows) + cus - 1) / cus; };
  return 31 * rounds(96) < 20 * rounds(64);
}

template <int kMats, int kEpilogue>
static int launch_exact(float* out, int64_t ldo, const float* A, int64_t lda, const float* W, const float* W2, int64_t ldw, const float* bias,
                        double* parts, int M, int N, int K, int gelu, const ExactNorm& norm, hipStream_t stream) {
  auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  const bool vec = K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && aligned(A) && aligned(W) && aligned(W2);
  if (M <= kExactRows)
    return vec ? launch_exact_rows<kMats, kEpilogue, true>(out, ldo, A, lda, W, W2, ldw, bias, parts, M, N, K, gelu, norm, stream)
               : launch_exact_rows<kMats, kEpilogue, false>(out, ldo, A, lda, W, W2, ldw, bias, parts, M, N, K, gelu, norm, stream);
  if constexpr (kMats == 2) {
    if (vec && taller_tiles(M, N)) return launch_exact_tile<2, 3, kMats, kEpilogue, true>(out, ldo, A, lda, W, W2, ldw, bias, parts, M, N, K, gelu, norm, stream);
  }
  if (M <= 32)
    return vec ? launch_exact_tile<1, 2, kMats, kEpilogue, true>(out, ldo, A, lda, W, W2, ldw, bias, parts, M, N, K, gelu, norm, stream)
               : launch_exact_tile<1, 2, kMats, kEpilogue, false>(out, ldo, A, lda, W, W2, ldw, bias, parts, M, N, K, gelu, norm, stream);
  return vec ? launch_exact_tile<2, 2, kMats, kEpilogue, true>(out, ldo, A, lda, W, W2, ldw, bias, parts, M, N, K, gelu, norm, stream)
             : launch_exact_tile<2, 2, kMats, kEpilogue, false>(out, ldo, A, lda, W, W2, ldw, bias, parts, M, N, K, gelu, norm, stream);
}

}  // namespace alofa

using namespace alofa;

// Float64 sums that alofa_gemm_exact needs room for with these sizes (0: none).
static int64_t exact_parts(int M, int N, int K, bool norm) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const Cut cut = cut_of(K);
  if (M <= kExactRows ? chains_per_block(N, cut, norm) == cut.count : !chains_apart(M, N, K, cut)) return 0;
  return static_cast<int64_t>(cut.count) * (M <= kExactRows ? M : rows_at_once(M, N, cut)) * N;
}
extern "C" int64_t alofa_gemm_exact_parts(int M, int N, int K) { return exact_parts(M, N, K, false); }

// The same for alofa_gemm_exact_norm; 0: it does not take the sizes (no sums go to memory whose launch the norm could ride on, or rows that are no whole fours or too wide).
extern "C" int64_t alofa_gemm_exact_norm_parts(int M, int N, int K) { return N % 4 == 0 && N <= 4096 ? exact_parts(M, N, K, true) : 0; }

extern "C" int alofa_gemm_exact(float* out, int64_t ldo, const float* A, int64_t lda, const float* W, int64_t ldw, const float* bias, double* parts, int64_t room,
                                int M, int N, int K, int epilogue, hipStream_t stream) {
  ALOFA_REQUIRE(M > 0 && N > 0 && K > 0, "gemm: M=%d N=%d K=%d must be positive", M, N, K);
  ALOFA_REQUIRE(epilogue == kExactStore || epilogue == kExactResidual, "gemm: unknown epilogue %d", epilogue);
  ALOFA_REQUIRE(lda >= K && ldw >= K && ldo >= N, "gemm: a leading dimension is shorter than its row");
  ALOFA_REQUIRE(room >= alofa_gemm_exact_parts(M, N, K), "gemm: no room for the sums of the chains of K");
  if (epilogue == kExactStore) return launch_exact<1, kExactStore>(out, ldo, A, lda, W, W, ldw, bias, parts, M, N, K, 0, ExactNorm{}, stream);
  return launch_exact<1, kExactResidual>(out, ldo, A, lda, W, W, ldw, bias, parts, M, N, K, 0, ExactNorm{}, stream);
}

// The product added to the residual stream, and the RMSNorm of the stream's new rows in `normed` (`ld` apart).
extern "C" int alofa_gemm_exact_norm(float* out, int64_t ldo, const float* A, int64_t lda, const float* W, int64_t ldw, double* parts, int64_t room, const float* norm_w, float eps,
                                     float* normed, int64_t ld, int M, int N, int K, hipStream_t stream) {
  ALOFA_REQUIRE(M > 0 && N > 0 && K > 0 && lda >= K && ldw >= K && ldo >= N && ld >= N, "gemm: M=%d N=%d K=%d must be positive, leading dimensions no shorter than the rows", M, N, K);
  const int64_t need = alofa_gemm_exact_norm_parts(M, N, K);
  ALOFA_REQUIRE(need > 0 && room >= need && parts && norm_w && normed && eps > 0.f, "gemm: no room for the sums of the chains of K, or sizes that no norm rides on (M=%d N=%d K=%d)", M, N, K);
  auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  ALOFA_REQUIRE(aligned(out) && aligned(parts) && aligned(norm_w) && aligned(normed) && ldo % 4 == 0 && ld % 4 == 0, "gemm: the norm behind the product takes 16-byte aligned rows");
  return launch_exact<1, kExactResidual>(out, ldo, A, lda, W, W, ldw, nullptr, parts, M, N, K, 0, ExactNorm{norm_w, eps, normed, ld}, stream);
}

// Rows of a block's tile of gate and up.
extern "C" int alofa_gemm_swiglu_exact_tile(int M, int N) { return M <= kExactRows ? 16 : taller_tiles(M, N) ? 96 : M <= 32 ? 32 : 64; }

extern "C" int alofa_gemm_swiglu_exact(float* out, int64_t ldo, const float* A, int64_t lda, const float* Wg, const float* Wu, int64_t ldw, int M, int N, int K,
                                       int gelu, hipStream_t stream) {
  ALOFA_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_swiglu: M=%d N=%d K=%d must be positive", M, N, K);
  ALOFA_REQUIRE(lda >= K && ldw >= K && ldo >= N, "gemm_swiglu: a leading dimension is shorter than its row");
  return launch_exact<2, kExactStore>(out, ldo, A, lda, Wg, Wu, ldw, nullptr, nullptr, M, N, K, gelu, ExactNorm{}, stream);
}
