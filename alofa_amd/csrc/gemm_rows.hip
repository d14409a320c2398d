// Matrix products for at most eight rows (the decode steps of few requests), bfloat16, on the
// vector units: out[m, n] = sum_k A[m, k] * W[n, k] with M <= 8 (M <= 16 for plain products: bfloat16 rows,
// store or residual epilogue, K <= 6144).
//
// The work is streaming W once from memory, and the time is what a compute unit needs to pull
// its share, so the shares are made small and even: a block owns C output columns (rows of W,
// four or eight), however few columns there are, and its wavefronts cut K into runs of 512:
// lane l of wave w holds the eight values 512 w + 8 l .. + 7 of every row of A and of each of
// the block's rows of W (one 16-byte load each, a wave's loads of a row contiguous), multiplies
// them in pairs (v_dot2_f32_bf16, float sums) and keeps C * M partial sums. Nothing is waited
// for before every load of the block is on its way, and no block waits for another: where the
// matrix-core kernel for few rows needs sixteen columns per block and, for a matrix of few
// columns, a hand-over of partial sums between blocks through memory, this one needs neither.
//
// The lanes' partial sums meet by exchange: at distance 32, 16, 8, 4, 2 the lanes swap one half
// of their values and add, so that each keeps half as many, then the last pair is added; the
// waves' sums meet in LDS and are added in wave order. The order of additions is fixed and the
// same for every row whatever else is in the batch (M only selects how many rows are computed).
//
// Up to twelve runs of 512 a wave takes one run (no loop at all); a longer K (the down projection of
// a wide feed-forward) goes to a second kernel whose eight waves take every eighth run in turn, the loads
// of the next run on their way while this one is multiplied.
//
// With a norm (kNorm) the rows of A are the float residual stream: a value is x * w_norm rounded
// to bfloat16, the squares of x are summed beside the products, and the row's factor
// 1 / sqrt(mean + eps) multiplies the finished sum, as in the matrix-core kernel for few rows.
#include "common.h"

namespace alofa {

enum RowsEpilogue : int { kRwStore = 0, kRwResidual = 1, kRwSwiglu = 2, kRwGeglu = 4, kRwActivated = 5, kRwDepth = 6 };

// What kRwActivated does to an output once it is rounded to bfloat16 (as the activation's own launch reads it: the same bits), activation_of in common.h.
struct RowsActivation {
  int kind;      // -1: none
  float a, b;
};

// kRwDepth: behind the sum into the residual stream the average over depth (depth_average_kernel in pointwise.hip: the same sums in the same order): the new value goes to level n - 1 of the stack
// [levels][level_stride], and the stream receives the sum of w[j] times level j. An output's levels are read by the thread that finishes it, with the rest of its loads.
struct RowsDepth {
  float* stack;
  int64_t level_stride, ld;
  const float* w;
  int n;
};

constexpr int kRowsMaxWaves = 12;     // runs of 512 along K, one per wave
constexpr int kRowsMaxK = kRowsMaxWaves * 512;

// v of lane l ^ 4 (within a row of 16): the lanes of banks 0 and 2 (four lanes each) read four lanes up,
// those of banks 1 and 3 four lanes down
__device__ __forceinline__ float lane_xor4(float v) {
  const uint32_t x = __float_as_uint(v);
  const uint32_t up = __builtin_amdgcn_update_dpp(0u, x, 0x104, 0xf, 0x5, false);     // row_shl:4 into banks 0, 2
  return __uint_as_float(__builtin_amdgcn_update_dpp(up, x, 0x114, 0xf, 0xa, false));   // row_shr:4 into banks 1, 3
}

// The sums over all 64 lanes of n values per lane (n a power of two, at most 64), by halving: after the
// step at distance d a lane whose bit d is set holds the upper half of the values, summed with its
// partner's, the other lane the lower half; the steps go from distance 32 down, and where one value is
// left it is added across the remaining distances. Afterwards v[0] of lane l is the total of value
// l >> (6 - log2 n). Every value goes through the same tree of lanes whatever n is.
template <int n, int d>
__device__ __forceinline__ void lanes_sum_step(float* v, int lane) {
  if constexpr (d >= 1) {
    if constexpr (n > 1) {
      constexpr int h = n / 2;
      const bool upper = (lane & d) != 0;
#pragma unroll
      for (int i = 0; i < h; ++i) {
        if constexpr (d == 32) {
          const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[i]), __float_as_uint(v[i + h]), false, false);
          v[i] = __uint_as_float(s[0]) + __uint_as_float(s[1]);
        } else if constexpr (d == 16) {
          const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[i + h]), false, false);
          v[i] = __uint_as_float(s[0]) + __uint_as_float(s[1]);
        } else {
          const float send = upper ? v[i] : v[i + h];
          const float keep = upper ? v[i + h] : v[i];
          const float got = d == 8 ? lane_xor8(send) : d == 4 ? lane_xor4(send) : d == 2 ? lane_xor2(send) : lane_xor1(send);
          v[i] = keep + got;
        }
      }
      lanes_sum_step<h, d / 2>(v, lane);
    } else {
      if constexpr (d == 32) {
        const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[0]), __float_as_uint(v[0]), false, false);
        v[0] = __uint_as_float(s[0]) + __uint_as_float(s[1]);
      } else if constexpr (d == 16) {
        const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[0]), __float_as_uint(v[0]), false, false);
        v[0] = __uint_as_float(s[0]) + __uint_as_float(s[1]);
      } else {
        v[0] += d == 8 ? lane_xor8(v[0]) : d == 4 ? lane_xor4(v[0]) : d == 2 ? lane_xor2(v[0]) : lane_xor1(v[0]);
      }
      lanes_sum_step<1, d / 2>(v, lane);
    }
  }
}
template <int n>
__device__ __forceinline__ void lanes_sum(float (&v)[n], int lane) {
  static_assert(n >= 1 && n <= 64 && (n & (n - 1)) == 0, "a power of two of values, at most one per lane");
  lanes_sum_step<n, 32>(v, lane);
}
constexpr int log2_of(int n) { return n <= 1 ? 0 : 1 + log2_of(n / 2); }

// The levels of an output's average over depth (kOn: kRwDepth): asked for with the thread's other loads, eight of them (a stack of fewer: its last one again), and the weights with them;
// more are read at the end.
template <bool kOn>
struct DepthOf {
  static constexpr int kHeld = 8;
  float held[kOn ? kHeld : 1], weight[kOn ? kHeld + 1 : 1];
  __device__ __forceinline__ void ask(const RowsDepth& d, int m, int n) {
    if constexpr (kOn) {
      const float* at = d.stack + static_cast<int64_t>(m) * d.ld + n;
#pragma unroll
      for (int j = 0; j < kHeld; ++j) held[j] = at[max(min(j, d.n - 2), 0) * d.level_stride];
#pragma unroll
      for (int j = 0; j < kHeld; ++j) weight[j] = d.w[min(j, d.n - 1)];
      weight[kHeld] = d.w[d.n - 1];
    }
  }
  __device__ __forceinline__ float average(const RowsDepth& d, int m, int n, float mine) const {
    float* at = d.stack + static_cast<int64_t>(m) * d.ld + n;
    at[(d.n - 1) * d.level_stride] = mine;
    float acc = 0.f;
#pragma unroll
    for (int j = 0; j < kHeld; ++j)
      if (j < d.n - 1) acc += weight[j] * held[j];
    for (int j = kHeld; j < d.n - 1; ++j) acc += d.w[j] * at[j * d.level_stride];
    return acc + weight[kHeld] * mine;
  }
};

// The squares of four values added up. Written out, as left to itself the compiler starts with x or with y as the code around it happens to be: one unit in the last place of a row's factor, and with it now and
// then an output's rounding. One row alone starts with x, several with y.
template <bool kFirstX>
__device__ __forceinline__ float squares_of(float4 v) {
  const float two = kFirstX ? __builtin_fmaf(v.y, v.y, v.x * v.x) : __builtin_fmaf(v.x, v.x, v.y * v.y);
  return __builtin_fmaf(v.w, v.w, __builtin_fmaf(v.z, v.z, two));
}

// MR: rows computed (1, 2, 4, 8, or 16 for plain products; rows beyond M are not stored); C: columns per block; kRwSwiglu: W is the gate
// matrix and W2 the up matrix, same columns; TO: float or bf16_t; kMaxWaves: bound of the block's waves.
template <int MR, int C, int kEpilogue, typename TO, bool kNorm, int kMaxWaves>
__device__ __forceinline__ void rows_block(
    TO* __restrict__ out, int64_t ldo, const void* __restrict__ A, int64_t lda, const bf16_t* __restrict__ W,
    const bf16_t* __restrict__ W2, int64_t ldw, const float* __restrict__ bias, int M, int N, int K,
    const float* __restrict__ norm_w, float eps, int block, const RowsActivation& act, const RowsDepth& depth) {
  constexpr int kMats = is_gated(kEpilogue) ? 2 : 1;
  constexpr int V = C * MR;                                // partial sums per lane and matrix
  __shared__ float red[kMaxWaves][kMats][V];
  __shared__ float ssq[kNorm ? kMaxWaves : 1][MR];
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, n_waves = blockDim.x / 64;
  const int n0 = block * C;
  const int k0 = (wave * 64 + lane) * 8;
  const bool k_ok = k0 < K;

  // Every load of this lane sets out, the weights (from memory) first, then the rows (which every block reads:
  // from L2). No load is conditional: a lane past the end of K reads where lane 0 does, rows beyond M and columns
  // beyond N read the last row and column (what they give is cleared below, or never stored), so that the loads are
  // one straight run of instructions with nothing to wait for between them.
  const int k_at = k_ok ? k0 : 0;
  uint4 wv[kMats][C];
#pragma unroll
  for (int mat = 0; mat < kMats; ++mat)
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const bf16_t* base = mat == 0 ? W : W2;
      const int n = n0 + c < N ? n0 + c : N - 1;
      wv[mat][c] = *reinterpret_cast<const uint4*>(base + static_cast<int64_t>(n) * ldw + k_at);
    }
  uint4 av[MR];               // the rows' values as pairs of bfloat16
  float4 xlo[kNorm ? MR : 1], xhi[kNorm ? MR : 1], nlo, nhi;
  if constexpr (kNorm) {
    nlo = *reinterpret_cast<const float4*>(norm_w + k_at);
    nhi = *reinterpret_cast<const float4*>(norm_w + k_at + 4);
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      const float* row = static_cast<const float*>(A) + static_cast<int64_t>(m < M ? m : M - 1) * lda + k_at;
      xlo[m] = *reinterpret_cast<const float4*>(row);
      xhi[m] = *reinterpret_cast<const float4*>(row + 4);
    }
  } else {
#pragma unroll
    for (int m = 0; m < MR; ++m)
      av[m] = *reinterpret_cast<const uint4*>(static_cast<const bf16_t*>(A) + static_cast<int64_t>(m < M ? m : M - 1) * lda + k_at);
  }
  // what the epilogue adds sets out too: thread c * MR + m finishes out[m, n0 + c]
  const int my_c = threadIdx.x / MR, my_m = threadIdx.x % MR;
  const bool finisher = threadIdx.x < V && my_m < M && n0 + my_c < N;
  float add = 0.f;
  DepthOf<kEpilogue == kRwDepth> levels;
  if (finisher) {
    if ((kEpilogue == kRwStore || kEpilogue == kRwActivated) && bias) add = bias[n0 + my_c];
    if (kEpilogue == kRwResidual || kEpilogue == kRwDepth) add = load_f32(out + static_cast<int64_t>(my_m) * ldo + n0 + my_c);
    levels.ask(depth, my_m, n0 + my_c);
  }
  // a lane past the end of K adds nothing: its weights and its rows' values are cleared
  if (!k_ok) {
#pragma unroll
    for (int mat = 0; mat < kMats; ++mat)
#pragma unroll
      for (int c = 0; c < C; ++c) wv[mat][c] = make_uint4(0, 0, 0, 0);
    if constexpr (kNorm) {
#pragma unroll
      for (int m = 0; m < MR; ++m) xlo[m] = xhi[m] = make_float4(0.f, 0.f, 0.f, 0.f);
    } else {
#pragma unroll
      for (int m = 0; m < MR; ++m) av[m] = make_uint4(0, 0, 0, 0);
    }
  }

  float ss[MR];
  if constexpr (kNorm) {
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      const float4 a = xlo[m], b = xhi[m];
      ss[m] = squares_of<MR == 1>(a) + squares_of<MR == 1>(b);
      av[m] = make_uint4(pack_bf16x2(a.x * nlo.x, a.y * nlo.y), pack_bf16x2(a.z * nlo.z, a.w * nlo.w),
                         pack_bf16x2(b.x * nhi.x, b.y * nhi.y), pack_bf16x2(b.z * nhi.z, b.w * nhi.w));
    }
  }

  float acc[kMats][V];
#pragma unroll
  for (int mat = 0; mat < kMats; ++mat)
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int m = 0; m < MR; ++m) {
        float s = dot2(av[m].x, wv[mat][c].x, 0.f);
        s = dot2(av[m].y, wv[mat][c].y, s);
        s = dot2(av[m].z, wv[mat][c].z, s);
        acc[mat][c * MR + m] = dot2(av[m].w, wv[mat][c].w, s);
      }

  // the lanes' sums meet; lane l then holds value l >> kShift
  constexpr int kShift = 6 - log2_of(V);
#pragma unroll
  for (int mat = 0; mat < kMats; ++mat) {
    lanes_sum<V>(acc[mat], lane);
    if ((lane & ((1 << kShift) - 1)) == 0) red[wave][mat][lane >> kShift] = acc[mat][0];
  }
  if constexpr (kNorm) {
    lanes_sum<MR>(ss, lane);
    constexpr int kRowShift = 6 - log2_of(MR);
    if ((lane & ((1 << kRowShift) - 1)) == 0) ssq[wave][lane >> kRowShift] = ss[0];
  }
  __syncthreads();

  if (!finisher) return;
  float sum = red[0][0][threadIdx.x], up = 0.f;
  for (int w = 1; w < n_waves; ++w) sum += red[w][0][threadIdx.x];
  if constexpr (is_gated(kEpilogue)) {
    up = red[0][1][threadIdx.x];
    for (int w = 1; w < n_waves; ++w) up += red[w][1][threadIdx.x];
  }
  if constexpr (kNorm) {
    float total = ssq[0][my_m];
    for (int w = 1; w < n_waves; ++w) total += ssq[w][my_m];
    // (the hardware's reciprocal square root, good to one unit in the last place, as in the matrix-core kernel)
    const float factor = __builtin_amdgcn_rsqf(total / static_cast<float>(K) + eps);
    sum *= factor;
    up *= factor;
  }
  TO* dst = out + static_cast<int64_t>(my_m) * ldo + n0 + my_c;
  if constexpr (kEpilogue == kRwStore) {
    store_f32(dst, sum + add);
  } else if constexpr (kEpilogue == kRwResidual) {
    store_f32(dst, add + sum);
  } else if constexpr (kEpilogue == kRwDepth) {
    store_f32(dst, levels.average(depth, my_m, n0 + my_c, add + sum));
  } else if constexpr (kEpilogue == kRwActivated) {
    store_f32(dst, act.kind < 0 ? sum + add : activation_of(round_bf16(sum + add), act.kind, act.a, act.b));
  } else {
    store_f32(dst, gate_of<kEpilogue == kRwGeglu>(sum) * up);
  }
}

template <int MR, int C, int kEpilogue, typename TO, bool kNorm, int kMaxWaves>
__global__ void __launch_bounds__(64 * kMaxWaves) gemm_rows_kernel(
    TO* __restrict__ out, int64_t ldo, const void* __restrict__ A, int64_t lda, const bf16_t* __restrict__ W,
    const bf16_t* __restrict__ W2, int64_t ldw, const float* __restrict__ bias, int M, int N, int K,
    const float* __restrict__ norm_w, float eps, RowsDepth depth) {
  rows_block<MR, C, kEpilogue, TO, kNorm, kMaxWaves>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, norm_w, eps, blockIdx.x, RowsActivation{}, depth);
}

// Up to kRowsMany products of the same count of rows and K side by side, each with its own rows, weights, columns and activation, a range of the grid's blocks each: bfloat16 rows and results.
// Such a launch is mostly the launch: the five of a time-mixing layer and an activation (1,024 x 1,024 four times, 64 x 1,024; in a captured run, us, one by one / this): one row 11.5 / 3.0, four 13.0 / 3.6,
// eight 14.7 / 4.5; of width 2,048 four rows 16.8 / 5.8. An activation behind 4,096 x 1,024 against four rows 5.0 / 3.4, eight 5.7 / 4.0; the average over nine levels behind 1,024 x 4,096 5.8 / 3.7 and
// 6.5 / 4.4 (kRwDepth).
constexpr int kRowsMany = 5;
struct RowsProducts {
  bf16_t* out[kRowsMany];
  const bf16_t *a[kRowsMany], *w[kRowsMany];
  int64_t ldo[kRowsMany], lda[kRowsMany], ldw[kRowsMany];
  int columns[kRowsMany], blocks_upto[kRowsMany];      // blocks of the products up to this one
  RowsActivation act[kRowsMany];
  const float* bias;                                    // of a product that stands alone
};
template <int MR, int kMaxWaves>
__global__ void __launch_bounds__(64 * kMaxWaves) gemm_rows_many_kernel(RowsProducts p, int M, int K) {
  int i = 0;
#pragma unroll
  for (int j = 0; j < kRowsMany - 1; ++j) i += static_cast<int>(blockIdx.x) >= p.blocks_upto[j] ? 1 : 0;
  i = __builtin_amdgcn_readfirstlane(i);
  rows_block<MR, 4, kRwActivated, bf16_t, false, kMaxWaves>(p.out[i], p.ldo[i], p.a[i], p.lda[i], p.w[i], nullptr, p.ldw[i], p.bias, M, p.columns[i], K, nullptr, 0.f,
                                                            static_cast<int>(blockIdx.x) - (i > 0 ? p.blocks_upto[i - 1] : 0), p.act[i], RowsDepth{});
}

// K beyond kRowsMaxK: the block's eight waves (eight rows' operands leave no registers for more, and the number
// must not depend on the rows: it sets the order of the additions) take the runs wave, wave + 8, ... in turn, two
// sets of operands
// in flight (each is loaded again as soon as it has been multiplied: no copies between sets, a copy would wait
// for its load). Store and residual epilogues, bfloat16 rows.
constexpr int rows_long_waves(int) { return 8; }

template <int MR, int C, int kEpilogue, typename TO>
__global__ void __launch_bounds__(64 * rows_long_waves(MR)) gemm_rows_long_kernel(
    TO* __restrict__ out, int64_t ldo, const bf16_t* __restrict__ A, int64_t lda, const bf16_t* __restrict__ W, int64_t ldw,
    const float* __restrict__ bias, int M, int N, int K, RowsDepth depth) {
  static_assert(kEpilogue == kRwStore || kEpilogue == kRwResidual || kEpilogue == kRwDepth, "plain products, and an average over depth behind one");
  constexpr int V = C * MR, kWaves = rows_long_waves(MR);
  __shared__ float red[kWaves][V];
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int n0 = blockIdx.x * C;
  const bf16_t* w_row[C];
  const bf16_t* a_row[MR];
#pragma unroll
  for (int c = 0; c < C; ++c) w_row[c] = W + static_cast<int64_t>(n0 + c < N ? n0 + c : N - 1) * ldw;
#pragma unroll
  for (int m = 0; m < MR; ++m) a_row[m] = A + static_cast<int64_t>(m < M ? m : M - 1) * lda;
  struct Set {
    uint4 w[C], a[MR];
  };
  // run `run` of K sets out (a lane past the end of K reads where lane 0 of the first run does; cleared at use)
  auto fetch = [&](Set& s, int run) __attribute__((always_inline)) {
    const int k0 = (run * 64 + lane) * 8;
    const int k_at = k0 < K ? k0 : 0;
#pragma unroll
    for (int c = 0; c < C; ++c) s.w[c] = *reinterpret_cast<const uint4*>(w_row[c] + k_at);
#pragma unroll
    for (int m = 0; m < MR; ++m) s.a[m] = *reinterpret_cast<const uint4*>(a_row[m] + k_at);
  };
  float acc[V];
#pragma unroll
  for (int i = 0; i < V; ++i) acc[i] = 0.f;
  auto multiply = [&](const Set& s, int run) __attribute__((always_inline)) {
    const bool k_ok = (run * 64 + lane) * 8 < K;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const uint4 w = k_ok ? s.w[c] : make_uint4(0, 0, 0, 0);
#pragma unroll
      for (int m = 0; m < MR; ++m) {
        float t = dot2(s.a[m].x, w.x, acc[c * MR + m]);
        t = dot2(s.a[m].y, w.y, t);
        t = dot2(s.a[m].z, w.z, t);
        acc[c * MR + m] = dot2(s.a[m].w, w.w, t);
      }
    }
  };
  const int my_c = threadIdx.x / MR, my_m = threadIdx.x % MR;
  const bool finisher = threadIdx.x < V && my_m < M && n0 + my_c < N;
  float add = 0.f;
  DepthOf<kEpilogue == kRwDepth> levels;
  if (finisher) {
    if (kEpilogue == kRwStore && bias) add = bias[n0 + my_c];
    if (kEpilogue == kRwResidual || kEpilogue == kRwDepth) add = load_f32(out + static_cast<int64_t>(my_m) * ldo + n0 + my_c);
    levels.ask(depth, my_m, n0 + my_c);
  }
  const int runs = (K + 511) / 512;
  Set s0, s1;
  int run = wave;
  fetch(s0, run);
  fetch(s1, run + kWaves);
  // (whole rounds: every fetch is issued, a run past the end reads run 0's place and adds nothing)
  for (; run < runs; run += 2 * kWaves) {
    multiply(s0, run);
    fetch(s0, run + 2 * kWaves);
    multiply(s1, run + kWaves);
    fetch(s1, run + 3 * kWaves);
  }
  constexpr int kShift = 6 - log2_of(V);
  lanes_sum<V>(acc, lane);
  if ((lane & ((1 << kShift) - 1)) == 0) red[wave][lane >> kShift] = acc[0];
  __syncthreads();
  if (!finisher) return;
  float sum = red[0][threadIdx.x];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) sum += red[w][threadIdx.x];
  TO* dst = out + static_cast<int64_t>(my_m) * ldo + n0 + my_c;
  if constexpr (kEpilogue == kRwDepth) store_f32(dst, levels.average(depth, my_m, n0 + my_c, add + sum));
  else store_f32(dst, kEpilogue == kRwStore ? sum + add : add + sum);
}

template <int MR, int C, int kEpilogue, typename TO, bool kNorm>
static int launch_rows(void* out, int64_t ldo, const void* A, int64_t lda, const void* W, const void* W2, int64_t ldw,
                       const float* bias, int M, int N, int K, const float* norm_w, float eps, const RowsDepth& depth, hipStream_t stream) {
  const int waves = (K + 511) / 512;
  const dim3 grid((N + C - 1) / C);
  if (waves > kRowsMaxWaves) {
    if constexpr (!kNorm && !is_gated(kEpilogue) && MR <= 8) {
      gemm_rows_long_kernel<MR, C, kEpilogue, TO><<<grid, 64 * rows_long_waves(MR), 0, stream>>>(
          static_cast<TO*>(out), ldo, static_cast<const bf16_t*>(A), lda, static_cast<const bf16_t*>(W), ldw, bias, M, N, K, depth);
      return check_launch("gemm_rows (long K)");
    }
    ALOFA_REQUIRE(false, "gemm_rows: K=%d beyond %d goes with the store and residual epilogues of bfloat16 rows only", K, kRowsMaxK);
    return 1;
  }
#define ALOFA_ROWS(MAXW)                                                                                               \
  gemm_rows_kernel<MR, C, kEpilogue, TO, kNorm, MAXW><<<grid, 64 * waves, 0, stream>>>(                                \
      static_cast<TO*>(out), ldo, A, lda, static_cast<const bf16_t*>(W), static_cast<const bf16_t*>(W2), ldw, bias, M, \
      N, K, norm_w, eps, depth)
  if (waves <= 4) {
    ALOFA_ROWS(4);
  } else {
    ALOFA_ROWS(kRowsMaxWaves);
  }
#undef ALOFA_ROWS
  return check_launch("gemm_rows");
}

template <int kEpilogue, typename TO, bool kNorm>
static int dispatch_rows(void* out, int64_t ldo, const void* A, int64_t lda, const void* W, const void* W2, int64_t ldw,
                         const float* bias, int M, int N, int K, const float* norm_w, float eps, hipStream_t stream, const RowsDepth& depth = RowsDepth{}) {
  // (gate and up: eight columns of either, so that the rows, which every block reads and, with a norm, converts,
  // are read half as often where the blocks are many)
  constexpr int C = is_gated(kEpilogue) ? 8 : 4;
  if (M <= 1) return launch_rows<1, C, kEpilogue, TO, kNorm>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, norm_w, eps, depth, stream);
  if (M <= 2) return launch_rows<2, C, kEpilogue, TO, kNorm>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, norm_w, eps, depth, stream);
  if (M <= 4) return launch_rows<4, C, kEpilogue, TO, kNorm>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, norm_w, eps, depth, stream);
  if constexpr (!kNorm && !is_gated(kEpilogue) && kEpilogue != kRwDepth) {
    if (M > 8) return launch_rows<16, C, kEpilogue, TO, kNorm>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, norm_w, eps, depth, stream);
  }
  return launch_rows<8, C, kEpilogue, TO, kNorm>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, norm_w, eps, depth, stream);
}

}  // namespace alofa

using namespace alofa;

// Whether alofa_gemm_rows takes these sizes.
// (K beyond 6,144, or nine to sixteen rows: the store and residual epilogues of bfloat16 rows only, `plain` then says
// that this is such a product)
extern "C" int alofa_gemm_rows_fits(int M, int N, int K, int plain) {
  return M >= 1 && (M <= 8 || (plain && M <= 16 && K <= kRowsMaxK)) && N >= 1 && K >= 8 && K % 8 == 0 && (K <= kRowsMaxK || plain);
}

// The same operands and epilogues as alofa_gemm_skinny (bfloat16 A [M, K] and W [N, K]; W2 for the swiglu epilogue;
// 0 store (+ bias) as o_dtype, 1 add to the float residual, 2 swiglu; norm_w not null: A is float [M, K] and takes
// an RMSNorm with these weights and eps on its way, bfloat16 store and swiglu epilogues), for M <= 8; K beyond 6,144
// with the store and residual epilogues of bfloat16 rows only.
extern "C" int alofa_gemm_rows(void* out, int o_dtype, int64_t ldo, const void* A, int64_t lda, const void* W,
                               const void* W2, int64_t ldw, const float* bias, int M, int N, int K, int epilogue,
                               const float* norm_w, float eps, hipStream_t stream) {
  ALOFA_REQUIRE(alofa_gemm_rows_fits(M, N, K, norm_w == nullptr && !is_gated(epilogue)),
                "gemm_rows: M=%d (1..8; to 16 for plain products of K up to 6,144) N=%d K=%d (a multiple of 8; beyond %d with the store and residual epilogues of bfloat16 rows only)", M, N, K, kRowsMaxK);
  ALOFA_REQUIRE(ldw % 8 == 0 && reinterpret_cast<uintptr_t>(W) % 16 == 0 && (W2 == nullptr || reinterpret_cast<uintptr_t>(W2) % 16 == 0),
                "gemm_rows: rows of W must be 16-byte aligned");
  ALOFA_REQUIRE(reinterpret_cast<uintptr_t>(A) % 16 == 0 && lda % (norm_w ? 4 : 8) == 0, "gemm_rows: rows of A must be 16-byte aligned");
  ALOFA_REQUIRE(lda >= K && ldw >= K && ldo >= N, "gemm_rows: strides shorter than the rows");
  ALOFA_REQUIRE(norm_w == nullptr || (reinterpret_cast<uintptr_t>(norm_w) % 16 == 0 && eps > 0.f), "gemm_rows: the norm's weights must be 16-byte aligned, eps positive");
  if (norm_w != nullptr) {
    if (epilogue == kRwStore && o_dtype == kBF16) return dispatch_rows<kRwStore, bf16_t, true>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, norm_w, eps, stream);
    if (epilogue == kRwSwiglu && o_dtype == kBF16 && W2) return dispatch_rows<kRwSwiglu, bf16_t, true>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, norm_w, eps, stream);
    if (epilogue == kRwGeglu && o_dtype == kBF16 && W2) return dispatch_rows<kRwGeglu, bf16_t, true>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, norm_w, eps, stream);
    ALOFA_REQUIRE(false, "gemm_rows: the norm goes with the bfloat16 store and swiglu epilogues only");
    return 1;
  }
  if (epilogue == kRwStore && o_dtype == kBF16) return dispatch_rows<kRwStore, bf16_t, false>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, nullptr, 0.f, stream);
  if (epilogue == kRwStore && o_dtype == kF32) return dispatch_rows<kRwStore, float, false>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, nullptr, 0.f, stream);
  if (epilogue == kRwResidual && o_dtype == kF32) return dispatch_rows<kRwResidual, float, false>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, nullptr, 0.f, stream);
  if (epilogue == kRwSwiglu && o_dtype == kBF16 && W2) return dispatch_rows<kRwSwiglu, bf16_t, false>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, nullptr, 0.f, stream);
  if (epilogue == kRwGeglu && o_dtype == kBF16 && W2) return dispatch_rows<kRwGeglu, bf16_t, false>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, nullptr, 0.f, stream);
  ALOFA_REQUIRE(false, "gemm_rows: no kernel for epilogue %d with output type %d", epilogue, o_dtype);
  return 1;
}

// Products of up to eight rows side by side, out_i [M, columns_i] = act_i(a_i [M, K] w_i^T), bfloat16 throughout, in one launch (count 1 to 5; what comes behind is not read). kind: -1 as it is, else an
// activation of pointwise.hip with its numbers act_a, act_b (the same for all of them). bias: of a product that stands alone.
extern "C" int alofa_gemm_rows_many(int count, int M, int K, const float* bias, float act_a, float act_b,
                                    void* o0, int64_t ldo0, const void* a0, int64_t lda0, const void* w0, int64_t ldw0, int n0, int kind0,
                                    void* o1, int64_t ldo1, const void* a1, int64_t lda1, const void* w1, int64_t ldw1, int n1, int kind1,
                                    void* o2, int64_t ldo2, const void* a2, int64_t lda2, const void* w2, int64_t ldw2, int n2, int kind2,
                                    void* o3, int64_t ldo3, const void* a3, int64_t lda3, const void* w3, int64_t ldw3, int n3, int kind3,
                                    void* o4, int64_t ldo4, const void* a4, int64_t lda4, const void* w4, int64_t ldw4, int n4, int kind4, hipStream_t stream) {
  ALOFA_REQUIRE(count >= 1 && count <= kRowsMany && M >= 1 && M <= 8 && K >= 8 && K % 8 == 0 && K <= kRowsMaxK && (!bias || count == 1),
                "gemm_rows_many: %d products (1..%d; a bias with one only), M=%d (1..8), K=%d (a multiple of 8, at most %d)", count, kRowsMany, M, K, kRowsMaxK);
  void* const os[] = {o0, o1, o2, o3, o4};
  const void *const as[] = {a0, a1, a2, a3, a4}, *const ws[] = {w0, w1, w2, w3, w4};
  const int64_t ldos[] = {ldo0, ldo1, ldo2, ldo3, ldo4}, ldas[] = {lda0, lda1, lda2, lda3, lda4}, ldws[] = {ldw0, ldw1, ldw2, ldw3, ldw4};
  const int ns[] = {n0, n1, n2, n3, n4}, kinds[] = {kind0, kind1, kind2, kind3, kind4};
  RowsProducts p{};
  p.bias = bias;
  int blocks = 0;
  for (int i = 0; i < kRowsMany; ++i) {
    if (i < count) {
      ALOFA_REQUIRE(ns[i] >= 1 && ldas[i] >= K && ldws[i] >= K && ldos[i] >= ns[i] && ldas[i] % 8 == 0 && ldws[i] % 8 == 0 && reinterpret_cast<uintptr_t>(as[i]) % 16 == 0 &&
                        reinterpret_cast<uintptr_t>(ws[i]) % 16 == 0, "gemm_rows_many: product %d: columns %d, rows of A and W must be 16-byte aligned, strides no shorter than the rows", i, ns[i]);
      ALOFA_REQUIRE(kinds[i] >= -1 && kinds[i] <= 3, "gemm_rows_many: no such activation (%d)", kinds[i]);
      p.out[i] = static_cast<bf16_t*>(os[i]), p.a[i] = static_cast<const bf16_t*>(as[i]), p.w[i] = static_cast<const bf16_t*>(ws[i]);
      p.ldo[i] = ldos[i], p.lda[i] = ldas[i], p.ldw[i] = ldws[i], p.columns[i] = ns[i], p.act[i] = RowsActivation{kinds[i], act_a, act_b};
      blocks += (ns[i] + 3) / 4;
    }
    p.blocks_upto[i] = i < count ? blocks : 0x7fffffff;
  }
  const int waves = (K + 511) / 512;
#define ALOFA_MANY(MR)                                                                                         \
  if (waves <= 4) gemm_rows_many_kernel<MR, 4><<<blocks, 64 * waves, 0, stream>>>(p, M, K);                    \
  else gemm_rows_many_kernel<MR, kRowsMaxWaves><<<blocks, 64 * waves, 0, stream>>>(p, M, K)
  if (M <= 1) { ALOFA_MANY(1); }
  else if (M <= 2) { ALOFA_MANY(2); }
  else if (M <= 4) { ALOFA_MANY(4); }
  else { ALOFA_MANY(8); }
#undef ALOFA_MANY
  return check_launch("gemm_rows_many");
}

// alofa_gemm_rows with the residual epilogue, and behind it the average over depth (see RowsDepth): stack [levels][level_stride], rows of it `ld` apart, w [n].
extern "C" int alofa_gemm_rows_depth(float* out, int64_t ldo, const void* A, int64_t lda, const void* W, int64_t ldw, int M, int N, int K, float* stack, int64_t level_stride, int64_t ld,
                                     const float* w, int n, hipStream_t stream) {
  ALOFA_REQUIRE(M <= 8 && alofa_gemm_rows_fits(M, N, K, 1), "gemm_rows_depth: M=%d (1..8) N=%d K=%d (a multiple of 8)", M, N, K);
  ALOFA_REQUIRE(lda % 8 == 0 && ldw % 8 == 0 && reinterpret_cast<uintptr_t>(A) % 16 == 0 && reinterpret_cast<uintptr_t>(W) % 16 == 0, "gemm_rows_depth: rows of A and W must be 16-byte aligned");
  ALOFA_REQUIRE(lda >= K && ldw >= K && ldo >= N && ld >= N && n >= 1 && w && stack, "gemm_rows_depth: strides shorter than the rows, or no levels (%d)", n);
  return dispatch_rows<kRwDepth, float, false>(out, ldo, A, lda, W, nullptr, ldw, nullptr, M, N, K, nullptr, 0.f, stream, RowsDepth{stack, level_stride, ld, w, n});
}
