// Paged causal grouped-query attention of the 32-bit path on the matrix cores: float queries, keys and values, every product
// and sum in float64 (v_mfma_f64_16x16x4_f64). Token t of request r stands at position p = positions[t] and sees the keys
// lo..p of r's pages, lo = 0 or p - window + 1.
//
// A block serves one token and up to 16 query heads of one key head: the heads are the columns of the tiles, so keys and values
// are read once for all of them. Its waves take tiles of 16 keys in turn. Lane l of the instruction holds A[row l % 16][k l / 16],
// B[k l / 16][column l % 16], D[rows 4 v + l / 16, v = 0..3][column l % 16]:
//   S[key, head] = K Q^T      row i of A is key 4 (i % 4) + i / 4 of the tile, so that lane l's four results are the keys 4 (l / 16) + v;
//   O^T[c, head] += V^T P^T   instruction v takes the keys 4 g + v, g = l / 16: the weights are the results where they lie, the values
//                             four consecutive keys of a channel, one 16-byte load.
// A score is rounded to float and multiplied by the float scale, the weight is expf of its difference to the running maximum; the
// sums of weights and of weighted values are float64, and where the maximum moves they take a float64 factor. The waves meet in
// LDS in their order, and how many they are follows from the head size: a row's result depends on its own keys only, to the bit.
//
// Bound by the chain table -> keys -> scores -> weights -> values of few tiles in decode steps and by the matrix cores in prompts
// (half of the columns idle with seven heads to a key head). us before (a wave a (token, head), one key a lane, every score twice)
// and now, 14/2 heads of 64: 8 tokens at 130 to 260 keys 85 and 11; prompts of 64, 128 and 256 tokens 145 and 27 (23 with four waves a block
// where blocks are many, and then a row depends on how many there are).
// Cache layout: keys [block, kv_head, slot_in_block, d], values transposed [block, kv_head, d, slot_in_block].
#include "common.h"

#include <float.h>

namespace alofa {

typedef double f64x4 __attribute__((ext_vector_type(4)));

// What the kernel needs to take a decode step's projections as they come out of the product (kRope; one token a request): q then points to rows [queries | keys | values] not yet turned, one token
// a request. Queries and the new key are turned here as rope_kv_write_kernel turns them (elementwise.hip: the same bits), the new key and value take their place among the cache's from registers, and
// the wave that has their tile writes them to the token's slot. Needs d a multiple of 32: a channel and its partner, d / 2 on, lie in the same lane. us in captured runs, a launch for it / here, 14/2 heads of 64: one token of 128 keys 10.5 / 8.6,
// eight of 60 7.9 / 6.5, of 250 12.4 / 11.1, three of 2,000 54.8 / 52.9.
constexpr int kTurnedTiles = 6;      // heads of up to 96: beyond, the registers of a wave do not hold the new token beside the rest
struct ExactRope {
  const float *cos_t, *sin_t;      // [position, d / 2]
  const int64_t* slots;
  float *k_cache, *v_cache;
};

__device__ __forceinline__ void turn_quads(float4& lo, float4& hi, float4 c, float4 s) {
#pragma clang fp contract(off)
  const float4 a = lo, b = hi;
  lo = make_float4(a.x * c.x - b.x * s.x, a.y * c.y - b.y * s.y, a.z * c.z - b.z * s.z, a.w * c.w - b.w * s.w);
  hi = make_float4(b.x * c.x + a.x * s.x, b.y * c.y + a.y * s.y, b.z * c.z + a.z * s.z, b.w * c.w + a.w * s.w);
}

// NT = d / 16, NW waves; blockIdx.y = key head * chunks + chunk of up to 16 heads of its group
template <int NT, int NW, bool kRope>
__global__ void __launch_bounds__(64 * NW) attention_exact_kernel(
    float* __restrict__ out, int64_t out_stride, const float* __restrict__ q, int64_t q_stride, const float* __restrict__ k_cache,
    const float* __restrict__ v_cache, const int32_t* __restrict__ block_table, int max_blocks, const int32_t* __restrict__ req_of_token,
    const int32_t* __restrict__ positions, int heads, int kv_heads, int block_size, int window, float scale, ExactRope rope) {
  static_assert(!kRope || NT % 2 == 0, "a channel and its partner in the same lane");
  constexpr int d = NT * 16;
  __shared__ double sums[NW][16][d + 1];      // per wave and head: the channels' sums, then the weights'
  __shared__ float maxima[NW][16];
  const int group = heads / kv_heads, chunks = (group + 15) / 16;
  const int t = blockIdx.x, hk = blockIdx.y / chunks, h0 = (blockIdx.y % chunks) * 16;
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, r = lane % 16, g = lane / 16;
  const int served = group - h0 < 16 ? group - h0 : 16;
  const int p = positions[t];
  const int lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;
  const int32_t* table = block_table + static_cast<int64_t>(req_of_token[t]) * max_blocks;
  const bool head_ok = r < served;
  float4 qf[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
    qf[i] = head_ok ? *reinterpret_cast<const float4*>(q + static_cast<int64_t>(t) * q_stride + static_cast<int64_t>(hk * group + h0 + r) * d + i * 16 + g * 4)
                    : make_float4(0.f, 0.f, 0.f, 0.f);
  float4 new_k[kRope ? NT : 1];      // the new token's key (this lane's channels, as of a query) and value (channels 16 i + r)
  float new_v[kRope ? NT : 1];
  if constexpr (kRope) {
    const float* k_row = q + static_cast<int64_t>(t) * q_stride + static_cast<int64_t>(heads + hk) * d;
    const float* v_row = k_row + static_cast<int64_t>(kv_heads) * d;
#pragma unroll
    for (int i = 0; i < NT; ++i) new_k[i] = *reinterpret_cast<const float4*>(k_row + i * 16 + g * 4), new_v[i] = v_row[i * 16 + r];
#pragma unroll
    for (int i = 0; i < NT / 2; ++i) {
      const int64_t at = static_cast<int64_t>(p) * (d / 2) + i * 16 + g * 4;
      const float4 c = *reinterpret_cast<const float4*>(rope.cos_t + at), sn = *reinterpret_cast<const float4*>(rope.sin_t + at);
      turn_quads(qf[i], qf[i + NT / 2], c, sn);
      turn_quads(new_k[i], new_k[i + NT / 2], c, sn);
    }
    // (first of all, so that the step behind this one does not wait for it; no wave reads the slot)
    if (h0 == 0 && wave == ((p >> 4) - (lo >> 4)) % NW) {
      const int64_t page = rope.slots[t] / block_size, off = rope.slots[t] % block_size;
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        if (r == 0) *reinterpret_cast<float4*>(rope.k_cache + ((page * kv_heads + hk) * block_size + off) * d + i * 16 + g * 4) = new_k[i];
        if (g == 0) rope.v_cache[((page * kv_heads + hk) * d + i * 16 + r) * block_size + off] = new_v[i];
      }
    }
  }
  f64x4 o[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) o[i] = f64x4{0, 0, 0, 0};
  double l = 0;
  float m = -FLT_MAX;
  const int mine = 4 * (r % 4) + r / 4;      // the key of a tile whose row this lane brings
  for (int tile = (lo >> 4) + wave; tile <= p >> 4; tile += NW) {
    const int at = tile << 4;
    // (keys and values of places that are not seen come from the nearest that is: their scores are masked, their values cleared)
    int key = at + mine, key4 = at + 4 * g;
    key = key < lo ? lo : key > p ? p : key;
    key4 = key4 < (lo & ~3) ? (lo & ~3) : key4 > (p & ~3) ? (p & ~3) : key4;
    const float* kr = k_cache + ((static_cast<int64_t>(table[key / block_size]) * kv_heads + hk) * block_size + key % block_size) * d + g * 4;
    const float* vr = v_cache + ((static_cast<int64_t>(table[key4 / block_size]) * kv_heads + hk) * d + r) * block_size + key4 % block_size;
    float4 kf[NT], vf[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) kf[i] = *reinterpret_cast<const float4*>(kr + i * 16);
#pragma unroll
    for (int i = 0; i < NT; ++i) vf[i] = *reinterpret_cast<const float4*>(vr + static_cast<int64_t>(i) * 16 * block_size);
    if constexpr (kRope) {      // (what the cache holds at the new token's place is not looked at)
      if (tile == p >> 4) {     // (uniform over the wave)
#pragma unroll
        for (int i = 0; i < NT; ++i) {
          if (key == p) kf[i] = new_k[i];
          if (key4 == (p & ~3)) {
            const int at4 = p & 3;
            vf[i].x = at4 == 0 ? new_v[i] : vf[i].x;
            vf[i].y = at4 == 1 ? new_v[i] : vf[i].y;
            vf[i].z = at4 == 2 ? new_v[i] : vf[i].z;
            vf[i].w = at4 == 3 ? new_v[i] : vf[i].w;
          }
        }
      }
    }
    f64x4 s = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      s = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(kf[i].x), static_cast<double>(qf[i].x), s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(kf[i].y), static_cast<double>(qf[i].y), s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(kf[i].z), static_cast<double>(qf[i].z), s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(kf[i].w), static_cast<double>(qf[i].w), s, 0, 0, 0);
    }
    float sc[4], top = -FLT_MAX;
    bool seen[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int place = at + 4 * g + v;
      seen[v] = place >= lo && place <= p;
      sc[v] = static_cast<float>(s[v]) * scale;
      if (seen[v]) top = fmaxf(top, sc[v]);
    }
    top = fmaxf(rows_max(top), m);
    if (__any(top > m)) {      // (uniform over the wave)
      const double f = exp(static_cast<double>(m) - static_cast<double>(top));
      l *= f;
#pragma unroll
      for (int i = 0; i < NT; ++i) o[i] *= f;
      m = top;
    }
    double e[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      e[v] = seen[v] ? static_cast<double>(expf(sc[v] - m)) : 0.0;
      l += e[v];
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      o[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(seen[0] ? static_cast<double>(vf[i].x) : 0.0, e[0], o[i], 0, 0, 0);
      o[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(seen[1] ? static_cast<double>(vf[i].y) : 0.0, e[1], o[i], 0, 0, 0);
      o[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(seen[2] ? static_cast<double>(vf[i].z) : 0.0, e[2], o[i], 0, 0, 0);
      o[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(seen[3] ? static_cast<double>(vf[i].w) : 0.0, e[3], o[i], 0, 0, 0);
    }
  }
  // the four lanes of a head add up their shares of the weights' sum
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  if (g == 0) maxima[wave][r] = m;
  __syncthreads();
  float most = maxima[0][r];
#pragma unroll
  for (int w = 1; w < NW; ++w) most = fmaxf(most, maxima[w][r]);
  const double f = exp(static_cast<double>(m) - static_cast<double>(most));      // (0 for a wave that saw no key)
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) sums[wave][r][i * 16 + 4 * v + g] = o[i][v] * f;
  if (g == 0) sums[wave][r][d] = l * f;
  __syncthreads();
  for (int i = threadIdx.x; i < served * d; i += 64 * NW) {
    double value = 0, weight = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) value += sums[w][i / d][i % d], weight += sums[w][i / d][d];
    out[static_cast<int64_t>(t) * out_stride + static_cast<int64_t>(hk * group + h0 + i / d) * d + i % d] = static_cast<float>(value / weight);
  }
}

template <int NT>
static void launch_attention_exact(float* out, int64_t out_stride, const float* q, int64_t q_stride, const float* k_cache, const float* v_cache,
                                   const int32_t* block_table, int max_blocks, const int32_t* req_of_token, const int32_t* positions, int tokens, int heads,
                                   int kv_heads, int block_size, int window, float scale, const ExactRope& rope, hipStream_t stream) {
  // (the number of waves, which decides whose running maximum a key's weight is taken against, follows from the head size alone: as many as the registers and LDS allow)
  constexpr int kWaves = NT <= 8 ? 8 : 4;
  dim3 grid(tokens, kv_heads * ((heads / kv_heads + 15) / 16));
  if constexpr (NT % 2 == 0 && NT <= kTurnedTiles) {
    if (rope.cos_t) {
      attention_exact_kernel<NT, kWaves, true><<<grid, 64 * kWaves, 0, stream>>>(out, out_stride, q, q_stride, k_cache, v_cache, block_table, max_blocks, req_of_token, positions, heads, kv_heads,
                                                                                 block_size, window, scale, rope);
      return;
    }
  }
  attention_exact_kernel<NT, kWaves, false><<<grid, 64 * kWaves, 0, stream>>>(out, out_stride, q, q_stride, k_cache, v_cache, block_table, max_blocks, req_of_token, positions, heads, kv_heads,
                                                                              block_size, window, scale, rope);
}

}  // namespace alofa

using namespace alofa;

// Whether alofa_attention_exact takes these sizes: heads in whole tiles, pages that hold four consecutive keys of a channel side by side, 16-byte aligned
// rows. Everything else stays with the kernel for any size (attention_simple.hip).
extern "C" int alofa_attention_exact_takes(const void* q, int64_t q_stride, const void* k_cache, const void* v_cache, int d, int block_size) {
  auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  return d > 0 && d <= 256 && d % 16 == 0 && block_size > 0 && block_size % 4 == 0 && q_stride % 4 == 0 && aligned(q) && aligned(k_cache) && aligned(v_cache);
}

// cos_t, sin_t, slots: null for queries that are turned and a cache that is written already; else see ExactRope.
extern "C" int alofa_attention_exact(float* out, int64_t out_stride, const float* q, int64_t q_stride, const float* k_cache, const float* v_cache,
                                     const int32_t* block_table, int max_blocks, const int32_t* req_of_token, const int32_t* positions, int tokens, int heads,
                                     int kv_heads, int d, int block_size, int window, float scale, const float* cos_t, const float* sin_t, const int64_t* slots, hipStream_t stream) {
  ALOFA_REQUIRE(tokens > 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0,
                "attention: tokens=%d heads=%d kv_heads=%d (kv_heads must divide heads)", tokens, heads, kv_heads);
  ALOFA_REQUIRE(alofa_attention_exact_takes(q, q_stride, k_cache, v_cache, d, block_size), "attention: head size %d, pages of %d or the operands' places do not fit", d, block_size);
  ALOFA_REQUIRE(max_blocks > 0 && window >= 0, "attention: max_blocks=%d window=%d", max_blocks, window);
  ALOFA_REQUIRE(!cos_t || (sin_t && slots && d % 32 == 0 && d <= 16 * kTurnedTiles && q_stride >= static_cast<int64_t>(heads + 2 * kv_heads) * d && reinterpret_cast<uintptr_t>(cos_t) % 16 == 0 && reinterpret_cast<uintptr_t>(sin_t) % 16 == 0),
                "attention: the form that turns the new token takes sin, slots, rows of queries, keys and values, a head size in steps of 32 up to 96 (%d), aligned tables", d);
  const ExactRope rope{cos_t, sin_t, slots, const_cast<float*>(k_cache), const_cast<float*>(v_cache)};
  switch (d / 16) {
#define ALOFA_EXACT_HEAD(NT)                                                                                                                                      \
  case NT:                                                                                                                                                        \
    launch_attention_exact<NT>(out, out_stride, q, q_stride, k_cache, v_cache, block_table, max_blocks, req_of_token, positions, tokens, heads, kv_heads,        \
                               block_size, window, scale, rope, stream);                                                                                               \
    break;
    ALOFA_EXACT_HEAD(1) ALOFA_EXACT_HEAD(2) ALOFA_EXACT_HEAD(3) ALOFA_EXACT_HEAD(4) ALOFA_EXACT_HEAD(5) ALOFA_EXACT_HEAD(6) ALOFA_EXACT_HEAD(7) ALOFA_EXACT_HEAD(8)
    ALOFA_EXACT_HEAD(9) ALOFA_EXACT_HEAD(10) ALOFA_EXACT_HEAD(11) ALOFA_EXACT_HEAD(12) ALOFA_EXACT_HEAD(13) ALOFA_EXACT_HEAD(14) ALOFA_EXACT_HEAD(15) ALOFA_EXACT_HEAD(16)
#undef ALOFA_EXACT_HEAD
  }
  return check_launch("attention_exact");
}
