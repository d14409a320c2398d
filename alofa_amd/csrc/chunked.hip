// The linear recurrence with one constant decay g per head, for steps of many rows: S_t = g S_(t-1) + k_t v_t^T, o_t = S_t^T q_t, taken
// in chunks of up to 64 rows of one request instead of row by row. With t, s counting a chunk's rows from 0 and n its rows:
//   what the chunk adds      U = sum_s g^(n-1-s) k_s v_s^T                                    (chunk_add: every chunk by itself)
//   the state in front of it S' = g^n S + U                                                   (chunk_states: a request's chunks in order)
//   its read-outs            o_t = g^(t+1) S^T q_t + sum_(s <= t) g^(t-s) (q_t . k_s) v_s     (chunk_read: every chunk by itself)
// All products run in float on the matrix cores (v_mfma_f32_16x16x4_f32: lane l holds A row and B column l % 16 at reduction index l / 16,
// and D column l % 16, rows 4 (l / 16) .. + 3), on operands that are bfloat16 numbers times a power of g, so nothing but float rounding
// separates the result from the recurrence row by row. q, k, v come as bfloat16 rows; the powers g^0 .. g^64 from a table; q is
// scaled by q_scale and k by k_scale.
//
// Chunks: int32 [n_chunks, 4]: request, first row, rows (<= 64), 0; a request's chunks lie together, in its rows' order, and
// of_request [requests, 2] holds the first one's number and their count. added [n_chunks, heads, dk, dv] float: U, then, in its place, the
// state in front of the chunk.
#include "common.h"

namespace alofa {

typedef float chunk_f32x4 __attribute__((ext_vector_type(4)));
constexpr int kChunkRows = 64, kPowers = kChunkRows + 1;

// A block of four wavefronts per (chunk, head, 64 x 64 piece of the state); wavefront w the piece's key channels 16 w .. + 15.
__global__ void __launch_bounds__(256) chunk_add_kernel(float* __restrict__ added, const bf16_t* __restrict__ k, int64_t k_stride, const bf16_t* __restrict__ v, int64_t v_stride,
                                                        const int32_t* __restrict__ chunks, const float* __restrict__ powers, int heads, int dk, int dv, float k_scale, int key_tiles) {
  constexpr int kRow = 80;      // floats of a staged row: rows one apart start 16 banks apart
  __shared__ float ks[kChunkRows][kRow], vs[kChunkRows][kRow];
  const int chunk = blockIdx.x, head = blockIdx.y, c0 = (blockIdx.z % key_tiles) * 64, j0 = (blockIdx.z / key_tiles) * 64;
  const int row0 = chunks[4 * chunk + 1], n = chunks[4 * chunk + 2];
  const float* pow_g = powers + head * kPowers;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
#pragma unroll
  for (int e = 0; e < 16; ++e) {      // (a wavefront brings in one row after the other, a lane a channel; rows past the chunk's end and channels past the head's are zeros)
    const int s = e * 4 + wave;
    const bool in = s < n;
    const int64_t r = row0 + (in ? s : 0);
    const float f = in ? pow_g[n - 1 - s] * k_scale : 0.f;
    ks[s][lane] = (in && c0 + lane < dk) ? bf16_to_f32(k[r * k_stride + static_cast<int64_t>(head) * dk + c0 + lane]) * f : 0.f;
    vs[s][lane] = (in && j0 + lane < dv) ? bf16_to_f32(v[r * v_stride + static_cast<int64_t>(head) * dv + j0 + lane]) : 0.f;
  }
  __syncthreads();
  const int c16 = lane % 16, g = lane / 16;
  chunk_f32x4 acc[4];
#pragma unroll
  for (int jt = 0; jt < 4; ++jt) acc[jt] = chunk_f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = (n + 3) / 4;
#pragma unroll 4
  for (int st = 0; st < steps; ++st) {
    const float a = ks[4 * st + g][16 * wave + c16];
#pragma unroll
    for (int jt = 0; jt < 4; ++jt) acc[jt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, vs[4 * st + g][16 * jt + c16], acc[jt], 0, 0, 0);
  }
  float* dst = added + (static_cast<int64_t>(chunk) * heads + head) * dk * dv;
#pragma unroll
  for (int jt = 0; jt < 4; ++jt) {
    const int j = j0 + 16 * jt + c16;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = c0 + 16 * wave + 4 * g + i;
      if (c < dk && j < dv) dst[static_cast<int64_t>(c) * dv + j] = acc[jt][i];
    }
  }
}

// A thread per value of a request's state: the chunks in order, eight of them on their way together. kRows: decays per row and key channel, `powers` then holds their products
// over a chunk, [chunk][heads][dk].
template <bool kRows>
__global__ void __launch_bounds__(256) chunk_states_kernel(float* __restrict__ added, float* __restrict__ state, const int32_t* __restrict__ chunks, const int32_t* __restrict__ of_request,
                                                           const int32_t* __restrict__ req_slot, const float* __restrict__ powers, int heads, int per_head, int dv) {
  constexpr int kAhead = 8;
  const int r = blockIdx.y;
  const int64_t width = static_cast<int64_t>(heads) * per_head, e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (e >= width) return;
  const float* pow_g = kRows ? powers + e / dv : powers + static_cast<int>(e / per_head) * kPowers;      // (kRows: a head's key channels lie side by side: e / dv = head * dk + channel)
  const int64_t channels = width / dv;
  float* mine = state + static_cast<int64_t>(req_slot[r]) * width + e;
  const int first = of_request[2 * r], count = of_request[2 * r + 1];
  float S = *mine;
  for (int c0 = 0; c0 < count; c0 += kAhead) {
    float u[kAhead], f[kAhead];
#pragma unroll
    for (int a = 0; a < kAhead; ++a) {
      const int c = first + (c0 + a < count ? c0 + a : count - 1);
      u[a] = added[static_cast<int64_t>(c) * width + e];
      f[a] = kRows ? pow_g[static_cast<int64_t>(c) * channels] : pow_g[chunks[4 * c + 2]];
    }
#pragma unroll
    for (int a = 0; a < kAhead; ++a) {
      if (c0 + a < count) {
        added[static_cast<int64_t>(first + c0 + a) * width + e] = S;
        S = f[a] * S + u[a];
      }
    }
  }
  *mine = S;
}

// A block of four wavefronts per (chunk, head, 64 value channels); wavefront w the chunk's rows 16 w .. + 15.
__global__ void __launch_bounds__(256) chunk_read_kernel(float* __restrict__ out, int64_t out_stride, const bf16_t* __restrict__ q, int64_t q_stride, const bf16_t* __restrict__ k,
                                                         int64_t k_stride, const bf16_t* __restrict__ v, int64_t v_stride, const float* __restrict__ before,
                                                         const int32_t* __restrict__ chunks, const float* __restrict__ powers, int heads, int dk, int dv, float q_scale, float k_scale) {
  // floats of a staged row: values are read in rows four apart, the state's in rows eight apart, by the four rows of lanes: 16 banks apart both ways
  constexpr int kVRow = 68, kSRow = 66;
  __shared__ float vs[kChunkRows][kVRow], ss[64][kSRow];
  const int chunk = blockIdx.x, head = blockIdx.y, j0 = blockIdx.z * 64;
  const int row0 = chunks[4 * chunk + 1], n = chunks[4 * chunk + 2];
  const float* pow_g = powers + head * kPowers;
  const float* S = before + (static_cast<int64_t>(chunk) * heads + head) * dk * dv;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, c16 = lane % 16, g = lane / 16;
  const int t = 16 * wave + c16;            // this lane's query row
  const bool active = 16 * wave < n, t_ok = t < n;
  const bf16_t* q_row = q + static_cast<int64_t>(row0 + (t_ok ? t : 0)) * q_stride + static_cast<int64_t>(head) * dk;
  const float q_front = t_ok ? pow_g[t + 1] * q_scale : 0.f;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const int s = e * 4 + wave;
    vs[s][lane] = (s < n && j0 + lane < dv) ? bf16_to_f32(v[static_cast<int64_t>(row0 + s) * v_stride + static_cast<int64_t>(head) * dv + j0 + lane]) : 0.f;
  }
  chunk_f32x4 acc[4];
#pragma unroll
  for (int jt = 0; jt < 4; ++jt) acc[jt] = chunk_f32x4{0.f, 0.f, 0.f, 0.f};
  // eight channels of a row, from channel c on (a head's size is a multiple of eight: all of them or none)
  auto eight = [&](const bf16_t* row, int c, bool ok, float (&x)[8]) {
    uint4 w = make_uint4(0, 0, 0, 0);
    if (ok && c < dk) w = *reinterpret_cast<const uint4*>(row + c);
    const uint32_t p[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) x[2 * i] = __uint_as_float(p[i] << 16), x[2 * i + 1] = __uint_as_float(p[i] & 0xffff0000u);
  };
  // ---- the state in front of the chunk, 64 key channels at a time
  for (int c0 = 0; c0 < dk; c0 += 64) {
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int c = e * 4 + wave;
      ss[c][lane] = (c0 + c < dk && j0 + lane < dv) ? S[static_cast<int64_t>(c0 + c) * dv + j0 + lane] : 0.f;
    }
    __syncthreads();
    if (!active) continue;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      if (c0 + 32 * half >= dk) break;      // (uniform)
      float x[8];
      eight(q_row, c0 + 32 * half + 8 * g, t_ok, x);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float a = x[i] * q_front;
#pragma unroll
        for (int jt = 0; jt < 4; ++jt) acc[jt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, ss[32 * half + 8 * g + i][16 * jt + c16], acc[jt], 0, 0, 0);
      }
    }
  }
  if (!active) return;
  // ---- the chunk's own rows up to the query: sixteen keys at a time. The products are formed transposed (key rows, query columns): what a lane then holds,
  // query t and keys 4 g + i, is its operand of the products with the values.
  for (int st = 0; st <= wave; ++st) {
    const int s_row = 16 * st + c16;
    const bf16_t* k_row = k + static_cast<int64_t>(row0 + (s_row < n ? s_row : 0)) * k_stride + static_cast<int64_t>(head) * dk;
    chunk_f32x4 p{0.f, 0.f, 0.f, 0.f};
    for (int c0 = 0; c0 < dk; c0 += 32) {
      float x[8], y[8];
      eight(k_row, c0 + 8 * g, s_row < n, x);
      eight(q_row, c0 + 8 * g, t_ok, y);
#pragma unroll
      for (int i = 0; i < 8; ++i) p = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i], y[i], p, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int s = 16 * st + 4 * g + i;
      const float a = (s <= t && t_ok) ? p[i] * (pow_g[t - s] * (q_scale * k_scale)) : 0.f;
#pragma unroll
      for (int jt = 0; jt < 4; ++jt) acc[jt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, vs[s][16 * jt + c16], acc[jt], 0, 0, 0);
    }
  }
#pragma unroll
  for (int jt = 0; jt < 4; ++jt) {
    const int j = j0 + 16 * jt + c16;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 16 * wave + 4 * g + i;
      if (row < n && j < dv) out[static_cast<int64_t>(row0 + row) * out_stride + static_cast<int64_t>(head) * dv + j] = acc[jt][i];
    }
  }
}

// ---- decays per row and key channel (gated linear attention, time mixing): S_t = diag(w_t) S_(t-1) + k_t v_t^T, 0 <= w <= 1 ------------------------------------
// The same three launches, with products of decays in place of powers. Every factor below is a product of decays, never a quotient of two, so none exceeds one and nothing overflows however
// small the decays are. A chunk's rows fall into four runs of sixteen (one a wavefront of the read-outs); with E_t the product of its run's decays up to row t (to the row before, where the
// read-out comes before the update), F_s that of the rows behind s in its run and D the runs' own:
//   the state in front       q_t E_t D(runs between) . S
//   keys of earlier runs     (q_t E_t D(runs between)) . (k_s F_s)
//   keys of the same run     the pairs whose rows first part at 8, 4, 2 or 1 (the highest bit in which their numbers differ), each kind a product of its own: the decays from the middle up to
//                            t on the query's side, those behind s up to the middle on the key's
// and last the row's own key (times the bonus, where the read-out comes before the update). Bound by the chains of float products and, where launches are small, by the launches; 4 prompts of
// 96 to 500 rows, 16 heads of 64, us: row after row (with the decays' own launch) 125 / this 44 (12 + 5 + 27), one of 2,048 471 / 53. Distance of the read-outs from 64 bits, in units of their norm: row after
// row 0.8 to 1.3e-7, this 1.1 to 2.2e-7 (heads of 64 to 256), of which bfloat16 rows behind the norm and gate keep 2e-3.
enum ChunkDecay : int { kChunkSigmoidRoot = 1, kChunkExpNegExp = 2, kChunkGiven = 3 };

__device__ __forceinline__ float chunk_decay_of(float z, int kind, float inv_tau) {
  if (kind == kChunkSigmoidRoot) return expf(-(fmaxf(-z, 0.f) + log1pf(expf(-fabsf(z)))) * inv_tau);
  return kind == kChunkExpNegExp ? expf(-expf(z)) : z;
}

// A block of eight wavefronts per (chunk, head, 64 x 64 piece of the state). Wavefront w makes the decays of rows 8 w .. + 7, a lane a channel; the blocks of the first 64 value channels leave
// the decays for the read-outs ([rows][heads dk]) and their products over the chunk.
__global__ void __launch_bounds__(512) chunk_add_decays_kernel(float* __restrict__ added, float* __restrict__ made, float* __restrict__ totals, const bf16_t* __restrict__ k, int64_t k_stride,
                                                               const bf16_t* __restrict__ v, int64_t v_stride, const float* __restrict__ z, int64_t z_stride,
                                                               const int32_t* __restrict__ chunks, int heads, int dk, int dv, int kind, float inv_tau, float k_scale, int key_tiles) {
  constexpr int kRow = 80;      // (chunk_add_kernel)
  __shared__ float ks[kChunkRows][kRow], vs[kChunkRows][kRow], runs[8][64];
  const int chunk = blockIdx.x, head = blockIdx.y, c0 = (blockIdx.z % key_tiles) * 64, j0 = (blockIdx.z / key_tiles) * 64;
  const int row0 = chunks[4 * chunk + 1], n = chunks[4 * chunk + 2];
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const bool key = c0 + lane < dk;
  const int64_t ch = static_cast<int64_t>(head) * dk + (key ? c0 + lane : 0);
  float w[8];
  bf16_t kk[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {      // (every lane loads, from the chunk's first row where its own is past the end)
    const int s = 8 * wave + i;
    const int64_t r = row0 + (s < n ? s : 0);
    w[i] = z[r * z_stride + ch];
    kk[i] = k[r * k_stride + ch];
    vs[s][lane] = (s < n && j0 + lane < dv) ? bf16_to_f32(v[r * v_stride + static_cast<int64_t>(head) * dv + j0 + lane]) : 0.f;
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int s = 8 * wave + i;
    w[i] = s < n ? chunk_decay_of(w[i], kind, inv_tau) : 1.f;
    if (j0 == 0 && key && s < n) made[static_cast<int64_t>(row0 + s) * heads * dk + ch] = w[i];
  }
  float behind = 1.f;
#pragma unroll
  for (int i = 7; i >= 0; --i) {
    const float mine = behind;
    behind *= w[i];
    w[i] = mine;      // the product of the run's decays behind row i
  }
  runs[wave][lane] = behind;
  __syncthreads();
  float later = k_scale;
#pragma unroll
  for (int x = 7; x > 0; --x) later *= x > wave ? runs[x][lane] : 1.f;
  if (wave == 0 && j0 == 0 && key) {
    float all = behind;
#pragma unroll
    for (int x = 1; x < 8; ++x) all *= runs[x][lane];
    totals[static_cast<int64_t>(chunk) * heads * dk + ch] = all;
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) ks[8 * wave + i][lane] = (key && 8 * wave + i < n) ? bf16_to_f32(kk[i]) * (w[i] * later) : 0.f;
  __syncthreads();
  const int c16 = lane % 16, g = lane / 16;
  const int tile = wave % 4, side = wave / 4 * 2;      // this wavefront's 16 key channels, and the first of its two tiles of value channels
  chunk_f32x4 acc[2];
#pragma unroll
  for (int jt = 0; jt < 2; ++jt) acc[jt] = chunk_f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = (n + 3) / 4;
#pragma unroll 4
  for (int st = 0; st < steps; ++st) {
    const float a = ks[4 * st + g][16 * tile + c16];
#pragma unroll
    for (int jt = 0; jt < 2; ++jt) acc[jt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, vs[4 * st + g][16 * (side + jt) + c16], acc[jt], 0, 0, 0);
  }
  float* dst = added + (static_cast<int64_t>(chunk) * heads + head) * dk * dv;
#pragma unroll
  for (int jt = 0; jt < 2; ++jt) {
    const int j = j0 + 16 * (side + jt) + c16;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = c0 + 16 * tile + 4 * g + i;
      if (c < dk && j < dv) dst[static_cast<int64_t>(c) * dv + j] = acc[jt][i];
    }
  }
}

// A block of eight wavefronts per (chunk, head, 64 value channels), two for every run of sixteen rows: of 64 key channels at a time either takes 32, from the products with the state and the
// keys to those with the values, and their outputs are added at the end (four wavefronts that take all channels each: 20 us where a lone chunk takes 18). kBefore: read-outs before the update, the row's own key times the bonus.
template <bool kBefore>
__global__ void __launch_bounds__(512, 4) chunk_read_decays_kernel(float* __restrict__ out, int64_t out_stride, const bf16_t* __restrict__ q, int64_t q_stride, const bf16_t* __restrict__ k,
                                                                int64_t k_stride, const bf16_t* __restrict__ v, int64_t v_stride, const float* __restrict__ w, const float* __restrict__ bonus,
                                                                const float* __restrict__ before, const int32_t* __restrict__ chunks, int heads, int dk, int dv, float q_scale, float k_scale) {
  // floats of a staged row: what is read by sixteen bytes 68; the state's and, in its place, the values' as in chunk_read_kernel
  constexpr int kRow = 68, kSRow = 66, kVRow = 68;
  __shared__ __attribute__((aligned(16))) float ws[kChunkRows][kRow], qe[kChunkRows][kRow], kf[kChunkRows][kRow], runs[4][64], ss[64 * kVRow];
  const int chunk = blockIdx.x, head = blockIdx.y, j0 = blockIdx.z * 64;
  const int row0 = chunks[4 * chunk + 1], n = chunks[4 * chunk + 2];
  const float* S = before + (static_cast<int64_t>(chunk) * heads + head) * dk * dv;
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), c16 = lane % 16, g = lane / 16;
  const int run = wave % 4, part = wave / 4, first = 16 * run;
  const int t = first + c16;            // this lane's query row, and its key row among the run's own
  const bool active = first < n, t_ok = t < n;
  chunk_f32x4 acc[4], near[5], far[3];      // outputs; products with the run's own keys by where the rows part (0: the row itself), with earlier runs' keys
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = chunk_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 5; ++i) near[i] = chunk_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 3; ++i) far[i] = chunk_f32x4{0.f, 0.f, 0.f, 0.f};
  const bf16_t* q_row = q + static_cast<int64_t>(row0 + (t_ok ? t : 0)) * q_stride + static_cast<int64_t>(head) * dk;
  const bf16_t* k_row = k + static_cast<int64_t>(row0 + (t_ok ? t : 0)) * k_stride + static_cast<int64_t>(head) * dk;
  const int c = 32 * part + 8 * g;      // this lane's first of eight key channels
  for (int c0 = 0; c0 < dk; c0 += 64) {
    // ---- 64 key channels of the chunk, a lane one of them: of a run's rows the first wavefront makes the queries' side, the second the keys'
    const bool key = c0 + lane < dk, mine = t_ok && c0 + c < dk;
    const int64_t ch = static_cast<int64_t>(head) * dk + (key ? c0 + lane : 0);
    const bf16_t* side = part ? k : q;
    int64_t side_stride = part ? k_stride : q_stride;
    int own_row = c16, own_c = c;
    asm volatile("" : "+s"(side_stride), "+v"(own_row), "+v"(own_c));      // (sizes and places formed anew for every 64 channels: kept over all of them they fill the registers)
    float dw[16], sv[8], u[8];
    bf16_t xx[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {      // (every lane loads, from the chunk's first row where its own is past the end)
      const int64_t r = row0 + (first + i < n ? first + i : 0);
      dw[i] = w[r * heads * dk + ch], xx[i] = side[r * side_stride + ch];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) sv[e] = (c0 + e * 8 + wave < dk && j0 + lane < dv) ? S[static_cast<int64_t>(c0 + e * 8 + wave) * dv + j0 + lane] : 0.f;
    uint4 qw = make_uint4(0, 0, 0, 0), kw = make_uint4(0, 0, 0, 0);
    if (mine) qw = *reinterpret_cast<const uint4*>(q_row + c0 + c), kw = *reinterpret_cast<const uint4*>(k_row + c0 + c);
#pragma unroll
    for (int i = 0; i < 8; ++i) u[i] = kBefore && c0 + c < dk ? bonus[static_cast<int64_t>(head) * dk + c0 + c + i] : 1.f;
    if (c0 > 0) __syncthreads();      // (the channels before have been read)
#pragma unroll
    for (int e = 0; e < 8; ++e) ss[(e * 8 + wave) * kSRow + lane] = sv[e];
    if (part == 0) {
      float upto = q_scale, all = 1.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const bool in = key && first + i < n;
        const float d = in ? dw[i] : 1.f;
        if (!kBefore) upto *= d;
        ws[first + i][lane] = d;
        qe[first + i][lane] = in ? bf16_to_f32(xx[i]) * upto : 0.f;
        if (kBefore) upto *= d;
        all *= d;
      }
      runs[run][lane] = all;
    } else {
      float behind = 1.f;
#pragma unroll
      for (int i = 15; i >= 0; --i) {
        const bool in = key && first + i < n;
        kf[first + i][lane] = in ? bf16_to_f32(xx[i]) * behind : 0.f;
        behind *= in ? dw[i] : 1.f;
      }
    }
    __syncthreads();
    if (!active || c0 + 32 * part >= dk) continue;      // (uniform over the wavefront; every wavefront meets all barriers)
    float y[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = qe[first + own_row][own_c + i];
#pragma unroll
    for (int st = 2; st >= 0; --st) {
      if (st < run) {      // (uniform over the wavefront)
#pragma unroll
        for (int i = 0; i < 8; ++i) far[st] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[16 * st + own_row][own_c + i], y[i], far[st], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] *= runs[st][own_c + i];
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int jt = 0; jt < 4; ++jt) acc[jt] = __builtin_amdgcn_mfma_f32_16x16x4f32(y[i], ss[(own_c + i) * kSRow + 16 * jt + own_row], acc[jt], 0, 0, 0);
    // the run's own keys
    float x[8], own[8];
    {
      const uint32_t a[4] = {qw.x, qw.y, qw.z, qw.w}, b[4] = {kw.x, kw.y, kw.z, kw.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[2 * i] = __uint_as_float(a[i] << 16) * q_scale, x[2 * i + 1] = __uint_as_float(a[i] & 0xffff0000u) * q_scale;
        own[2 * i] = __uint_as_float(b[i] << 16), own[2 * i + 1] = __uint_as_float(b[i] & 0xffff0000u);
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) near[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(own[i] * u[i], x[i], near[0], 0, 0, 0);
#pragma unroll
    for (int level = 1; level <= 4; ++level) {
      const int size = 1 << (level - 1), mid = (own_row & ~(2 * size - 1)) + size;      // rows of the run: the upper half of 2 size rows begins at mid
      const bool upper = own_row >= mid;
      float f[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) f[i] = upper ? x[i] : own[i];
#pragma unroll
      for (int j = 0; j < size; ++j) {
        if (j % 4 == 0) __builtin_amdgcn_sched_barrier(0);      // (four rows' decays asked for at once: more do not fit the registers)
        // (upper: rows mid .. c16, or .. c16 - 1; lower: rows c16 + 1 .. mid - 1)
        const int row = upper ? mid + j : mid - 1 - j;
        const bool counts = upper ? (kBefore ? row < own_row : row <= own_row) : row > own_row;
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] *= counts ? ws[first + row][own_c + i] : 1.f;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) near[level] = __builtin_amdgcn_mfma_f32_16x16x4f32(upper ? 0.f : f[i], upper ? f[i] : 0.f, near[level], 0, 0, 0);
    }
  }
  // ---- the values, in the place of the state
  {
    float sv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int s = e * 8 + wave;
      sv[e] = (s < n && j0 + lane < dv) ? bf16_to_f32(v[static_cast<int64_t>(row0 + s) * v_stride + static_cast<int64_t>(head) * dv + j0 + lane]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 8; ++e) ss[(e * 8 + wave) * kVRow + lane] = sv[e];
  }
  __syncthreads();
  if (active) {
    // (a lane holds, for query t, the products with keys 4 g + i of a run: its operand of the products with the values)
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      if (st > run) break;      // (uniform over the wavefront)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int s = 4 * g + i, parts_at = s ^ c16;      // (of the same run)
        float a = 0.f;
        if (st < run) {
          a = far[st < 3 ? st : 0][i];
        } else if (s <= c16) {
          a = parts_at >= 8 ? near[4][i] : parts_at >= 4 ? near[3][i] : parts_at >= 2 ? near[2][i] : parts_at == 1 ? near[1][i] : near[0][i];
        }
        a = t_ok ? a * k_scale : 0.f;
#pragma unroll
        for (int jt = 0; jt < 4; ++jt) acc[jt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, ss[(16 * st + s) * kVRow + 16 * jt + c16], acc[jt], 0, 0, 0);
      }
    }
  }
  // ---- the second wavefront's outputs by way of LDS (the decays have been read)
  float* shared = &ws[0][0] + run * 1024 + lane;
  if (part == 1) {
#pragma unroll
    for (int jt = 0; jt < 4; ++jt)
#pragma unroll
      for (int i = 0; i < 4; ++i) shared[(4 * jt + i) * 64] = acc[jt][i];
  }
  __syncthreads();
  if (part == 1 || !active) return;
#pragma unroll
  for (int jt = 0; jt < 4; ++jt) {
    const int j = j0 + 16 * jt + c16;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = first + 4 * g + i;
      if (row < n && j < dv) out[static_cast<int64_t>(row0 + row) * out_stride + static_cast<int64_t>(head) * dv + j] = acc[jt][i] + shared[(4 * jt + i) * 64];
    }
  }
}

}  // namespace alofa

using namespace alofa;

extern "C" int alofa_chunk_rows() { return kChunkRows; }

extern "C" int alofa_chunked_recurrence(float* out, int64_t out_stride, const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v, int64_t v_stride, float* state,
                                        const int32_t* req_slot, const int32_t* chunks, int n_chunks, const int32_t* of_request, int requests, const float* powers, float* added,
                                        int heads, int dk, int dv, float q_scale, float k_scale, hipStream_t stream) {
  ALOFA_REQUIRE(n_chunks >= 0 && requests >= 0 && n_chunks >= requests && heads > 0 && dk > 0 && dk % 8 == 0 && dv > 0, "chunked_recurrence: bad sizes (chunks=%d requests=%d heads=%d dk=%d dv=%d; dk a multiple of 8)", n_chunks, requests, heads, dk, dv);
  ALOFA_REQUIRE(q_stride % 8 == 0 && k_stride % 8 == 0 && reinterpret_cast<uintptr_t>(q) % 16 == 0 && reinterpret_cast<uintptr_t>(k) % 16 == 0, "chunked_recurrence: rows of q and k must be 16-byte aligned");
  ALOFA_REQUIRE(heads <= 65535 && requests <= 65535, "chunked_recurrence: %d heads, %d requests", heads, requests);
  if (n_chunks == 0) return 0;
  const int key_tiles = (dk + 63) / 64, value_tiles = (dv + 63) / 64;
  const bf16_t *qb = static_cast<const bf16_t*>(q), *kb = static_cast<const bf16_t*>(k), *vb = static_cast<const bf16_t*>(v);
  chunk_add_kernel<<<dim3(n_chunks, heads, key_tiles * value_tiles), 256, 0, stream>>>(added, kb, k_stride, vb, v_stride, chunks, powers, heads, dk, dv, k_scale, key_tiles);
  if (check_launch("chunked_recurrence (add)")) return 1;
  const int64_t width = static_cast<int64_t>(heads) * dk * dv;
  chunk_states_kernel<false><<<dim3(static_cast<unsigned>((width + 255) / 256), requests), 256, 0, stream>>>(added, state, chunks, of_request, req_slot, powers, heads, dk * dv, dv);
  if (check_launch("chunked_recurrence (states)")) return 1;
  chunk_read_kernel<<<dim3(n_chunks, heads, value_tiles), 256, 0, stream>>>(out, out_stride, qb, q_stride, kb, k_stride, vb, v_stride, added, chunks, powers, heads, dk, dv, q_scale, k_scale);
  return check_launch("chunked_recurrence (read)");
}

// z [rows, heads dk]: what the decays are made of (kind 1: sigmoid(z)^(1 / tau), 2: exp(-exp(z)), 3: the decays, none above one). made [rows, heads dk] and totals [n_chunks, heads, dk]: room.
extern "C" int alofa_chunked_recurrence_decays(float* out, int64_t out_stride, const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v, int64_t v_stride,
                                               const float* z, int64_t z_stride, const float* bonus, float* state, const int32_t* req_slot, const int32_t* chunks, int n_chunks,
                                               const int32_t* of_request, int requests, float* made, float* totals, float* added, int heads, int dk, int dv, int kind, float tau,
                                               float q_scale, float k_scale, int before_update, hipStream_t stream) {
  ALOFA_REQUIRE(n_chunks >= 0 && requests >= 0 && n_chunks >= requests && heads > 0 && dk > 0 && dk % 8 == 0 && dv > 0, "chunked_recurrence: bad sizes (chunks=%d requests=%d heads=%d dk=%d dv=%d; dk a multiple of 8)", n_chunks, requests, heads, dk, dv);
  ALOFA_REQUIRE(q_stride % 8 == 0 && k_stride % 8 == 0 && reinterpret_cast<uintptr_t>(q) % 16 == 0 && reinterpret_cast<uintptr_t>(k) % 16 == 0, "chunked_recurrence: rows of q and k must be 16-byte aligned");
  ALOFA_REQUIRE(heads <= 65535 && requests <= 65535, "chunked_recurrence: %d heads, %d requests", heads, requests);
  ALOFA_REQUIRE(kind >= kChunkSigmoidRoot && kind <= kChunkGiven && (kind != kChunkSigmoidRoot || tau > 0.f), "chunked_recurrence: decay kind %d, tau %g", kind, static_cast<double>(tau));
  ALOFA_REQUIRE(!before_update || bonus, "chunked_recurrence: a read-out before the update needs the bonus");
  if (n_chunks == 0) return 0;
  const int key_tiles = (dk + 63) / 64, value_tiles = (dv + 63) / 64;
  const bf16_t *qb = static_cast<const bf16_t*>(q), *kb = static_cast<const bf16_t*>(k), *vb = static_cast<const bf16_t*>(v);
  chunk_add_decays_kernel<<<dim3(n_chunks, heads, key_tiles * value_tiles), 512, 0, stream>>>(added, made, totals, kb, k_stride, vb, v_stride, z, z_stride, chunks, heads, dk, dv, kind,
                                                                                              kind == kChunkSigmoidRoot ? 1.f / tau : 0.f, k_scale, key_tiles);
  if (check_launch("chunked_recurrence (add, decays)")) return 1;
  const int64_t width = static_cast<int64_t>(heads) * dk * dv;
  chunk_states_kernel<true><<<dim3(static_cast<unsigned>((width + 255) / 256), requests), 256, 0, stream>>>(added, state, chunks, of_request, req_slot, totals, heads, dk * dv, dv);
  if (check_launch("chunked_recurrence (states)")) return 1;
  const dim3 grid(n_chunks, heads, value_tiles);
  if (before_update) chunk_read_decays_kernel<true><<<grid, 512, 0, stream>>>(out, out_stride, qb, q_stride, kb, k_stride, vb, v_stride, made, bonus, added, chunks, heads, dk, dv, q_scale, k_scale);
  else chunk_read_decays_kernel<false><<<grid, 512, 0, stream>>>(out, out_stride, qb, q_stride, kb, k_stride, vb, v_stride, made, bonus, added, chunks, heads, dk, dv, q_scale, k_scale);
  return check_launch("chunked_recurrence (read, decays)");
}
