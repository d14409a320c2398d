// Paged causal grouped-query attention for many query rows of heads of 128, bfloat16 on MFMA with a running softmax: the form of
// attention_prefill.hip's product for launches with rows enough to give most compute units a block of 256 of them (eight waves of 32
// rows, one query head), so that a tile of keys and values is brought once for all of them.
//
// What bounded the smaller blocks was bringing and staging tiles: with 64 rows a block every tile of 32 KB was fetched, held in registers
// and written to LDS for 64 rows' arithmetic. Here the tiles of 64 keys come straight from memory into a ring of S in LDS
// (global_load_lds_dwordx4), in the order the pages have them: 16 keys [key, d] (the 16-byte chunks of a key's row permuted by the key's
// number, so that sixteen keys read together fall on distinct banks) and 16 keys' values [channel, 16 keys] (a fragment is 1 KB in one
// piece as it is). Nothing passes through registers, one barrier a tile. What is left is the softmax on the vector unit (some 1,000
// cycles a wave and tile) beside 1,024 cycles of products; the two waves of a SIMD fill one another's gaps.
//
// 40/8 heads, 2 x 2,048 rows on 6,144 and 10,240 keys 1,315 -> 766 us (1.01 PFLOP/s); 28/4 heads, 2,048 rows on 8,192 keys 538 -> 282. Measured
// and not kept (beside 725 and 268 us, with one state a row): the two waves of a SIMD half a tile apart by barriers, one with the products while the other has the weights (788 and 301 us: their
// slots come out unequal, and the slower of eight waves ends each); the fetches behind the first product (774 and 285); a higher wave priority for the
// products (no difference); head size 64, 256 or 128 rows (14/2 heads, 8,192 rows 241 and 292 us against 212: half the products for the same softmax).
//
// Both products are taken transposed (v_mfma_f32_32x32x16_bf16; lane l: A row and B column l % 32, reduction slots 8 (l / 32) .. + 7, D column
// l % 32 and rows 8 j + 4 (l / 32) + r): S^T = K Q^T, O^T += V^T P^T. Row i = 16 y + 8 jj + 4 h + r of a 32-key half is key 16 y + 8 h + 4 jj + r, so that the
// weights a lane holds for one instruction of the second product are eight consecutive keys: its values are one 16-byte read.
//
// Scores, maximum, weights and their sum are float, the weights are rounded to bfloat16 as operands only. A row's maximum is followed in every tile
// that raises it, so that the weight that counts most is one, which no rounding touches; a tile that raises no row's maximum leaves the outputs alone. A row has
// two running states, of the even and of the odd tiles, which meet at the end: the highest weight of either is exact, as it is with the two teams of the blocks of
// 64 rows, and the results are as far from 64 bits as theirs (40/8 heads, 1,024 rows on 3,072 keys, scores times 1, 2, 4 and 8: 0.002246, 0.001869,
// 0.001708 and 0.001655 here and there; with one state 0.002270, 0.001916, 0.001736 and 0.001672; with one state that follows the maximum only where a tile passes it by
// more than 2^8 0.002342, 0.002306, 0.002142 and 0.001976). The times of the three: 766, 759 and 722 us, 282, 276 and 265.
//
// Blocks of one key head go to one die where there are eight of them (the dies take blocks in turn): its keys and values then stay in that
// die's L2 for all the rows and heads that read them.
// Cache layout: keys [block, kv_head, slot_in_block, d], values transposed [block, kv_head, d, slot_in_block]; pages of 16 tokens or more, a power of two.
#include "common.h"

#include <float.h>

#include <type_traits>

namespace alofa {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float two_halves_max(float v) {
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float two_halves_sum(float v) {
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// runs: int32 [n_runs, 4]: request index, first row in the packed batch, rows (1 .. 256), position of the first row; longest first
template <int S>
__global__ void __launch_bounds__(512) attention_tall_kernel(bf16_t* __restrict__ out, int64_t out_stride, const bf16_t* __restrict__ q, int64_t q_stride,
                                                                 const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
                                                                 const int32_t* __restrict__ block_table, int max_blocks, const int32_t* __restrict__ runs, int n_runs,
                                                                 int heads, int kv_heads, int bs_shift, int window, float scale) {
  constexpr int DT = 8, NW = 8, d = DT * 16, KT = 64, OT = d / 32;
  constexpr int kKeyBytes = KT * d * 2, kStage = 2 * kKeyBytes;
  constexpr int kLoads = d / 8 / NW;                 // fetch instructions (1 KB each) of a wave for a tile's keys, and as many for its values
  static_assert(kLoads * NW * 8 == d && S >= 2 && S * kStage <= 160 * 1024, "the waves share a tile's fetches evenly");
  __shared__ __attribute__((aligned(1024))) char ring[S * kStage];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  const int r32 = lane % 32, h = lane / 32;
  const int group = heads / kv_heads;
  // die b % 8 takes one contiguous stretch of the blocks in the order key head, run, head of the group; where that cuts a key head's blocks over several dies, each of them takes every
  // so-manieth run, else one had all the longest
  const int total = gridDim.x, die = blockIdx.x % 8, at = die * (total / 8) + min(die, total % 8) + blockIdx.x / 8;
  const int hk = at / (n_runs * group), place = at % (n_runs * group) / group, head = hk * group + at % group;
  const int dies = 8 % kv_heads == 0 ? 8 / kv_heads : 1, each = n_runs / dies, larger = n_runs % dies * (each + 1);      // (the first dies of a key head may have a run more)
  const int run = place < larger ? place % (each + 1) * dies + place / (each + 1) : (place - larger) % each * dies + n_runs % dies + (place - larger) / each;
  const int req = runs[4 * run], row0 = runs[4 * run + 1], n_rows = runs[4 * run + 2], pos0 = runs[4 * run + 3];
  const int32_t* table = block_table + static_cast<int64_t>(req) * max_blocks;
  const int my_row = wave * 32 + r32;
  const bool row_ok = my_row < n_rows;
  const int my_pos = pos0 + my_row;
  const int last_pos = pos0 + n_rows - 1, first_key = (window > 0 && pos0 - window + 1 > 0) ? pos0 - window + 1 : 0;
  const int t_begin = first_key / KT, t_end = last_pos / KT;
  const int first_page = first_key >> bs_shift, last_page = last_pos >> bs_shift, page_mask = (1 << bs_shift) - 1;

  bf16x8 qf[DT];
#pragma unroll
  for (int ds = 0; ds < DT; ++ds)
    qf[ds] = __builtin_bit_cast(bf16x8, row_ok ? *reinterpret_cast<const uint4*>(q + static_cast<int64_t>(row0 + my_row) * q_stride + static_cast<int64_t>(head) * d + ds * 16 + h * 8)
                                               : make_uint4(0, 0, 0, 0));

  // (the queries must have arrived before the loop: a wait for them within it would be a wait for the tiles on their way)
#pragma unroll
  for (int ds = 0; ds < DT; ++ds) asm volatile("" : "+v"(qf[ds]));

  // What this wave fetches of a tile lies within the 16 keys 16 x .. of it: one page. Keys: instruction j brings kLoads .. of d / 8 instructions, 512 / d keys each;
  // values: of each 16 keys d / 32 instructions of 32 channels.
  const int x16 = wave * 4 / NW;
  int k_off[kLoads], v_off[kLoads];      // within a page, of this lane's 16 bytes
  unsigned k_to[kLoads], v_to[kLoads];
  const unsigned ring_at = static_cast<unsigned>(reinterpret_cast<uintptr_t>(ring));
#pragma unroll
  for (int j = 0; j < kLoads; ++j) {
    const int ii = wave * kLoads + j;
    const int key = ii * (512 / d) + lane / (d / 8), chunk = (lane % (d / 8)) ^ (key & 15);
    k_off[j] = key % 16 * d + chunk * 8;      // (+ the page's first slot of these 16 keys)
    k_to[j] = ring_at + ii * 1024;
    const int channel = ii % (d / 32) * 32 + lane / 2;
    v_off[j] = (channel << bs_shift) + lane % 2 * 8;
    v_to[j] = ring_at + kKeyBytes + ii * 1024;
  }
  auto page_of = [&](int t) {      // (uniform; places past the visible keys come from the last page that is visible, before them from the first)
    const int p = (t * KT + 16 * x16) >> bs_shift;
    return table[p < first_page ? first_page : p > last_page ? last_page : p];
  };
  auto fetch = [&](int t, int page, unsigned stage) __attribute__((always_inline)) {
    const int slot = (t * KT + 16 * x16) & page_mask;
    const bf16_t* kb = k_cache + (((static_cast<int64_t>(page) * kv_heads + hk) << bs_shift) + slot) * d;
    const bf16_t* vb = v_cache + ((static_cast<int64_t>(page) * kv_heads + hk) * d << bs_shift) + slot;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                   :: "s"(__builtin_amdgcn_readfirstlane(k_to[j] + stage)), "v"(2u * k_off[j]), "s"(kb), "r"(ring) : "memory", "m0");
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                   :: "s"(__builtin_amdgcn_readfirstlane(v_to[j] + stage)), "v"(2u * v_off[j]), "s"(vb), "r"(ring) : "memory", "m0");
    }
  };

  f32x16 o[2][OT];      // of the even tiles and of the odd ones, counted from the block's first
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int nt = 0; nt < OT; ++nt)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[x][nt][e] = 0.f;
  float m[2] = {-FLT_MAX, -FLT_MAX}, l[2] = {0.f, 0.f};
  const float scale2 = scale * 1.44269504088896340736f;   // scores in units of log2(e)

  // fragments: keys row 32 kh + (r32's key), chunk 2 ds + h; values channel 32 nt + r32, keys 16 x + 8 h ..
  const int my_key = (r32 & 0x13) | ((r32 & 4) << 1) | ((r32 & 8) >> 1);      // 16 y + 8 jj + 4 h' + r -> 16 y + 8 h' + 4 jj + r
  const int key_row = my_key * d * 2, key_sw = my_key & 15;
  f32x16 s[2];
  bf16x8 pf[4];
  // n products with a read from LDS each: kAhead reads set out before the first product, then one with every product
  auto reads_ahead = [](auto n) __attribute__((always_inline)) {
    constexpr int kAhead = 4;
    __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);
#pragma unroll
    for (int i = 0; i < n.value - kAhead; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, kAhead, 0);
  };
  auto take_values = [&](const char* st, auto which) __attribute__((always_inline)) {
    constexpr int w = decltype(which)::value;
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int nt = 0; nt < OT; ++nt) {
        const uint4 vv = *reinterpret_cast<const uint4*>(st + kKeyBytes + ((x * d + nt * 32 + r32) * 2 + h) * 16);
        o[w][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, vv), pf[x], o[w][nt], 0, 0, 0);
      }
    reads_ahead(std::integral_constant<int, 4 * OT>{});
  };
  auto take_keys = [&](const char* st) __attribute__((always_inline)) {
#pragma unroll
    for (int kh = 0; kh < 2; ++kh)
#pragma unroll
      for (int e = 0; e < 16; ++e) s[kh][e] = 0.f;
#pragma unroll
    for (int ds = 0; ds < DT; ++ds)
#pragma unroll
      for (int kh = 0; kh < 2; ++kh) {
        const uint4 kv = *reinterpret_cast<const uint4*>(st + kh * 32 * d * 2 + key_row + ((2 * ds + h) ^ key_sw) * 16);
        s[kh] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kv), qf[ds], s[kh], 0, 0, 0);
      }
    reads_ahead(std::integral_constant<int, 2 * DT>{});
  };
  auto take_weights = [&](int t, bool whole, auto which) __attribute__((always_inline)) {
    constexpr int w = decltype(which)::value;
    if (!whole) {      // (uniform) what a row does not see: minus infinity, whose weight is zero against any maximum
#pragma unroll
      for (int i = 0; i < 32; ++i) {
        const int key = t * KT + i / 16 * 32 + i % 16 / 8 * 16 + h * 8 + i % 8;
        const bool seen = key <= my_pos && (window <= 0 || key > my_pos - window);
        s[i / 16][i % 16] = seen ? s[i / 16][i % 16] : -__builtin_inff();
      }
    }
    float top = s[0][0];
#pragma unroll
    for (int i = 1; i < 32; ++i) top = fmaxf(top, s[i / 16][i % 16]);
    top = two_halves_max(top) * scale2;
    if (__any(top > m[w])) {
      const float m_new = fmaxf(m[w], top), corr = __builtin_amdgcn_exp2f(m[w] - m_new);      // (1 where a row's maximum stays, and while it has seen nothing yet: m is -FLT_MAX)
      m[w] = m_new;
      l[w] *= corr;
#pragma unroll
      for (int nt = 0; nt < OT; ++nt) o[w][nt] *= corr;
    }
    float sum = 0.f;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      float p[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        p[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[x / 2][x % 2 * 8 + i], scale2, -m[w]));
        sum += p[i];
      }
      pf[x] = __builtin_bit_cast(bf16x8, make_uint4(pack_bf16x2(p[0], p[1]), pack_bf16x2(p[2], p[3]), pack_bf16x2(p[4], p[5]), pack_bf16x2(p[6], p[7])));
    }
    l[w] += sum;
  };
  // Values beyond the block's visible keys (in its first and last tiles) are not data: cleared, so that a weight of zero times them is zero.
  auto clear = [&](int t, char* st) {
    for (int i = threadIdx.x; i < 4 * d; i += 64 * NW) {      // 16 keys of a channel
      uint32_t* row = reinterpret_cast<uint32_t*>(st + kKeyBytes + i * 32);
      const int key = t * KT + i / d * 16;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const bool a = key + 2 * e >= first_key && key + 2 * e <= last_pos, b = key + 2 * e + 1 >= first_key && key + 2 * e + 1 <= last_pos;
        row[e] &= (a ? 0x0000ffffu : 0u) | (b ? 0xffff0000u : 0u);
      }
    }
  };

  // tile t + S - 1 takes the place of tile t - 1, which every wave has read before the barrier of tile t
  const int first_row_pos = pos0 + wave * 32, last_row_pos = min(first_row_pos + 31, last_pos);      // of this wave (none of the run's rows: last < first)
  int page_next = page_of(t_begin + S - 1);
#pragma unroll
  for (int p = 0; p < S - 1; ++p)
    if (t_begin + p <= t_end) fetch(t_begin + p, page_of(t_begin + p), p * kStage);
  unsigned stage = 0;
  auto step = [&](int t, auto which) __attribute__((always_inline)) {
    if (t + S - 2 <= t_end) asm volatile("s_waitcnt vmcnt(%0)" :: "n"(2 * kLoads * (S - 2)) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    char* st = ring + stage;
    if (t + S - 1 <= t_end) {
      fetch(t + S - 1, page_next, stage == 0 ? (S - 1) * kStage : stage - kStage);
      page_next = page_of(t + S);
    }
    stage = stage == (S - 1) * kStage ? 0 : stage + kStage;
    if (t * KT < first_key || t * KT + KT - 1 > last_pos) {      // (uniform over the block)
      clear(t, st);
      __syncthreads();
    }
    // (uniform over the wave) a wave without rows, which only brings its share of the tiles (28/4 heads, 8 portions of 64 rows on 8,192 keys 197 us when it worked too, 146 so); a tile of which no row of the wave sees a key; one that every row sees whole
    if (last_row_pos < first_row_pos || t * KT > last_row_pos || (window > 0 && t * KT + KT - 1 <= first_row_pos - window)) return;
    take_keys(st);
    take_weights(t, t * KT + KT - 1 <= first_row_pos && (window <= 0 || t * KT > last_row_pos - window), which);
    take_values(st, which);
  };
  for (int t = t_begin; t <= t_end; t += 2) {
    step(t, std::integral_constant<int, 0>{});
    if (t + 1 <= t_end) step(t + 1, std::integral_constant<int, 1>{});
  }
  const float most = fmaxf(m[0], m[1]), even = __builtin_amdgcn_exp2f(m[0] - most), odd = __builtin_amdgcn_exp2f(m[1] - most);
  const float all = two_halves_sum(l[0] * even + l[1] * odd);
#pragma unroll
  for (int nt = 0; nt < OT; ++nt) o[0][nt] = o[0][nt] * even + o[1][nt] * odd;
  if (row_ok) {
    const float inv = 1.f / all;
    bf16_t* dst = out + static_cast<int64_t>(row0 + my_row) * out_stride + static_cast<int64_t>(head) * d;
#pragma unroll
    for (int nt = 0; nt < OT; ++nt)
#pragma unroll
      for (int j = 0; j < 4; ++j)      // four consecutive channels
        *reinterpret_cast<uint2*>(dst + nt * 32 + 8 * j + 4 * h) =
            make_uint2(pack_bf16x2(o[0][nt][4 * j] * inv, o[0][nt][4 * j + 1] * inv), pack_bf16x2(o[0][nt][4 * j + 2] * inv, o[0][nt][4 * j + 3] * inv));
  }
}

}  // namespace alofa

using namespace alofa;

extern "C" int alofa_attention_tall(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* k_cache, const void* v_cache, const int32_t* block_table,
                                    int max_blocks, const int32_t* runs, int n_runs, int heads, int kv_heads, int d, int block_size, int window, float scale,
                                    hipStream_t stream) {
  ALOFA_REQUIRE(n_runs > 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0, "attention_tall: runs=%d heads=%d kv_heads=%d (kv_heads must divide heads)", n_runs, heads, kv_heads);
  ALOFA_REQUIRE(d == 128 && scale > 0.f, "attention_tall: head size %d (128 is built), scale %g (positive)", d, static_cast<double>(scale));
  ALOFA_REQUIRE(block_size >= 16 && (block_size & (block_size - 1)) == 0 && max_blocks > 0 && window >= 0,
                "attention_tall: block_size=%d must be a power of two, at least 16; max_blocks=%d window=%d", block_size, max_blocks, window);
  ALOFA_REQUIRE(q_stride % 8 == 0 && out_stride % 4 == 0 && reinterpret_cast<uintptr_t>(q) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 8 == 0 &&
                    reinterpret_cast<uintptr_t>(k_cache) % 16 == 0 && reinterpret_cast<uintptr_t>(v_cache) % 16 == 0,
                "attention_tall: q rows and the caches must be 16-byte aligned and out rows 8-byte aligned");
  int bs_shift = 0;
  while ((1 << bs_shift) < block_size) ++bs_shift;
  attention_tall_kernel<4><<<n_runs * heads, 512, 0, stream>>>(static_cast<bf16_t*>(out), out_stride, static_cast<const bf16_t*>(q), q_stride,
                                                               static_cast<const bf16_t*>(k_cache), static_cast<const bf16_t*>(v_cache), block_table, max_blocks, runs,
                                                               n_runs, heads, kv_heads, bs_shift, window, scale);
  return check_launch("attention_tall");
}
