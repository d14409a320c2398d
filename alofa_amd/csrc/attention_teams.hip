// Paged causal grouped-query attention for prompt portions of heads of 64, bfloat16 on MFMA with a running softmax: 64 query rows of one head a block (up to two runs of rows, a long one
// with a short one, as in attention_prefill.hip), four teams of two waves that take the tiles of 64 keys in turn, a wave 32 rows.
//
// What bounded the blocks of attention_prefill.hip (four teams of four waves, sixteen rows a wave) was reading the tiles: every wave reads all 16 KB of a tile from LDS for sixteen rows'
// arithmetic, 0.85 us of LDS time a round of four tiles beside 0.43 of products, and the tiles pass through registers on their way in, each by waits and writes of its own. Here a fragment
// read feeds twice the products (v_mfma_f32_32x32x16_bf16), half as many waves read, and the tiles come straight from memory into LDS (global_load_lds_dwordx4; two tiles a team, the
// next one on its way while one is worked on), one barrier a round. What is left is the softmax on the vector unit, some 460 cycles a tile of 64 x 64.
// us, attention_prefill.hip / this, 14/2 heads: one prompt of 2,048 29.7 / 22.9, of 512 10.5 / 8.5, two of 1,500 44.2 / 35.1, 2,048 rows on 8,000 keys 155 / 113, three prompts of 5 to 33
// 7.2 / 6.9; 8/8 heads, one prompt of 2,048 23.8 / 18.7. A round of the teams takes 1.4 to 1.6 us, 1.15 without the tiles' way into LDS (64 KB a round, 45 bytes a nanosecond a compute
// unit), and a run 3 us beside its rounds. Measured and not kept: the second run's pages, queries and first tile asked for before the first one's states meet (23.7 and 7.7), other
// cache policies for the tiles (streaming 26.2), a key head's blocks on one die (even).
//
// Both products are taken transposed and the keys of a tile are in the order that attention_tall.hip explains: a lane's weights for one instruction of the second product are eight consecutive
// keys. Scores, the running maximum, the weights and their sum are float, the weights are rounded to bfloat16 as operands only. A row has a running state per team, which meet in
// LDS in team order, as many states as it had: the results are as near 64 bits.
// Cache layout: keys [block, kv_head, slot_in_block, d], values transposed [block, kv_head, d, slot_in_block]; pages of 16 tokens or more, a power of two.
#include "common.h"

#include <float.h>

namespace alofa {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float pair_max(float v) {
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float pair_sum(float v) {
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// tiles: int32 [n_blocks, 2, 4], up to two runs of rows a block: (request index, first row in the packed batch, rows (<= 64; 0: none), position of the first row)
__global__ void __launch_bounds__(512) attention_teams_kernel(bf16_t* __restrict__ out, int64_t out_stride, const bf16_t* __restrict__ q, int64_t q_stride,
                                                              const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache, const int32_t* __restrict__ block_table,
                                                              int max_blocks, const int32_t* __restrict__ tiles, int heads, int kv_heads, int bs_shift, int window, float scale) {
  constexpr int d = 64, KT = 64, kTeams = 4, OT = 2, kKeyBytes = KT * d * 2, kTile = 2 * kKeyBytes, kRoom = 2 * kTile;      // kRoom: a team's two tiles
  constexpr int kWords = 16 * OT + 2;      // of a lane's running state
  static_assert(kWords * 512 * 4 <= kTeams * kRoom, "the states fit where the tiles were");
  __shared__ __attribute__((aligned(1024))) char ring[kTeams * kRoom];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, team = wave >> 1, half = wave & 1;
  const int r32 = lane % 32, h = lane / 32;
  const int head = blockIdx.y, hk = head / (heads / kv_heads), page_mask = (1 << bs_shift) - 1;
  char* room = ring + team * kRoom;
  const float scale2 = scale * 1.44269504088896340736f;   // scores in units of log2(e)

  // What this wave fetches of a tile: its two groups of sixteen keys, each within one page; two instructions of 1 KB for a group's keys (a key's 16-byte chunks permuted by the key's number, so that
  // sixteen keys read together fall on distinct banks) and two for its values (in the page's order).
  int k_off[2], v_off[2];      // within a page, of this lane's 16 bytes, in elements
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int key = 8 * j + lane / 8;
    k_off[j] = key * d + ((lane % 8) ^ (key >> 1)) * 8;
    v_off[j] = ((32 * j + lane / 2) << bs_shift) + lane % 2 * 8;
  }
  const unsigned room_at = static_cast<unsigned>(reinterpret_cast<uintptr_t>(room));
  const int my_key = (r32 & 0x13) | ((r32 & 4) << 1) | ((r32 & 8) >> 1);      // row 16 y + 8 jj + 4 h' + r of a 32-key half is key 16 y + 8 h' + 4 jj + r
  const int key_row = my_key * d * 2, key_sw = my_key >> 1 & 7;

  for (int part = 0; part < 2; ++part) {
    const int32_t* run = tiles + 8 * blockIdx.x + 4 * part;
    const int req = run[0], row0 = run[1], n_rows = run[2], pos0 = run[3];
    if (n_rows <= 0) break;      // uniform over the block
    const int32_t* table = block_table + static_cast<int64_t>(req) * max_blocks;
    const int my_row = half * 32 + r32, my_pos = pos0 + my_row;
    const bool row_ok = my_row < n_rows;
    const int last_pos = pos0 + n_rows - 1, first_key = (window > 0 && pos0 - window + 1 > 0) ? pos0 - window + 1 : 0;
    const int t_begin = first_key / KT, t_end = last_pos / KT, first_page = first_key >> bs_shift, last_page = last_pos >> bs_shift;
    const int first_row_pos = pos0 + half * 32, last_row_pos = min(first_row_pos + 31, last_pos);      // of this wave (none of the run's rows: last < first)

    bf16x8 qf[4];
#pragma unroll
    for (int ds = 0; ds < 4; ++ds)
      qf[ds] = __builtin_bit_cast(bf16x8, row_ok ? *reinterpret_cast<const uint4*>(q + static_cast<int64_t>(row0 + my_row) * q_stride + static_cast<int64_t>(head) * d + ds * 16 + h * 8)
                                                 : make_uint4(0, 0, 0, 0));
    // (the queries must have arrived before the loop: a wait for them within it would be a wait for the tiles on their way)
#pragma unroll
    for (int ds = 0; ds < 4; ++ds) asm volatile("" : "+v"(qf[ds]));

    auto page_of = [&](int t, int group) {      // (uniform; places past the visible keys come from the last page that is visible, before them from the first)
      const int p = (t * KT + 16 * group) >> bs_shift;
      return table[p < first_page ? first_page : p > last_page ? last_page : p];
    };
    auto fetch = [&](int t, int page0, int page1, unsigned stage) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int group = 2 * half + i, slot = (t * KT + 16 * group) & page_mask, page = i == 0 ? page0 : page1;
        const bf16_t* kb = k_cache + (((static_cast<int64_t>(page) * kv_heads + hk) << bs_shift) + slot) * d;
        const bf16_t* vb = v_cache + ((static_cast<int64_t>(page) * kv_heads + hk) * d << bs_shift) + slot;
        const unsigned to = room_at + stage + group * 2048;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                       :: "s"(__builtin_amdgcn_readfirstlane(to + j * 1024)), "v"(2u * k_off[j]), "s"(kb), "r"(ring) : "memory", "m0");
          asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                       :: "s"(__builtin_amdgcn_readfirstlane(to + kKeyBytes + j * 1024)), "v"(2u * v_off[j]), "s"(vb), "r"(ring) : "memory", "m0");
        }
      }
    };
    // Values beyond the run's visible keys (in its first and last tiles) are not data: cleared, so that a weight of zero times them is zero.
    auto clear = [&](int t, char* st) {
      for (int i = half * 64 + lane; i < 4 * d; i += 128) {      // 16 keys of a channel
        uint32_t* row = reinterpret_cast<uint32_t*>(st + kKeyBytes + i * 32);
        const int key = t * KT + i / d * 16;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const bool a = key + 2 * e >= first_key && key + 2 * e <= last_pos, b = key + 2 * e + 1 >= first_key && key + 2 * e + 1 <= last_pos;
          row[e] &= (a ? 0x0000ffffu : 0u) | (b ? 0xffff0000u : 0u);
        }
      }
    };

    f32x16 o[OT];
#pragma unroll
    for (int nt = 0; nt < OT; ++nt)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[nt][e] = 0.f;
    float m = -FLT_MAX, l = 0.f;

    if (part > 0) __syncthreads();      // (the first run's states have been read)
    int t = t_begin + team;
    if (t <= t_end) fetch(t, page_of(t, 2 * half), page_of(t, 2 * half + 1), 0);
    int next0 = page_of(t + kTeams, 2 * half), next1 = page_of(t + kTeams, 2 * half + 1);
    unsigned stage = 0;
    for (int t0 = t_begin; t0 <= t_end; t0 += kTeams, t += kTeams) {      // uniform over the block
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_barrier" ::: "memory");      // (every wave's pieces of this tile are there, and the tile before has been read by all)
      __builtin_amdgcn_sched_barrier(0);
      char* st = room + stage;
      stage ^= kTile;
      if (t + kTeams <= t_end) {
        fetch(t + kTeams, next0, next1, stage);
        next0 = page_of(t + 2 * kTeams, 2 * half);
        next1 = page_of(t + 2 * kTeams, 2 * half + 1);
      }
      if (t0 * KT < first_key || (t0 + kTeams) * KT - 1 > last_pos) {      // (uniform over the block: one of its tiles has keys that are none)
        if (t <= t_end && (t * KT < first_key || t * KT + KT - 1 > last_pos)) clear(t, st);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_barrier" ::: "memory");      // (not a wait for the tiles on their way)
        __builtin_amdgcn_sched_barrier(0);
      }
      // (uniform over the wave) no tile, no rows, a tile of which no row of the wave sees a key
      if (t > t_end || last_row_pos < first_row_pos || t * KT > last_row_pos || (window > 0 && t * KT + KT - 1 <= first_row_pos - window)) continue;

      f32x16 s[2];
#pragma unroll
      for (int kh = 0; kh < 2; ++kh)
#pragma unroll
        for (int e = 0; e < 16; ++e) s[kh][e] = 0.f;
#pragma unroll
      for (int ds = 0; ds < 4; ++ds)
#pragma unroll
        for (int kh = 0; kh < 2; ++kh) {
          const uint4 kv = *reinterpret_cast<const uint4*>(st + kh * 32 * d * 2 + key_row + ((2 * ds + h) ^ key_sw) * 16);
          s[kh] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kv), qf[ds], s[kh], 0, 0, 0);
        }
      if (!(t * KT + KT - 1 <= first_row_pos && (window <= 0 || t * KT > last_row_pos - window))) {      // what a row does not see: minus infinity, whose weight is zero against any maximum
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
      top = pair_max(top) * scale2;
      if (__any(top > m)) {
        const float m_new = fmaxf(m, top), corr = __builtin_amdgcn_exp2f(m - m_new);      // (1 where a row's maximum stays, and while it has seen nothing yet: m is -FLT_MAX)
        m = m_new;
        l *= corr;
#pragma unroll
        for (int nt = 0; nt < OT; ++nt) o[nt] *= corr;
      }
      bf16x8 pf[4];
      float sum = 0.f;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        float p[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          p[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[x / 2][x % 2 * 8 + i], scale2, -m));
          sum += p[i];
        }
        pf[x] = __builtin_bit_cast(bf16x8, make_uint4(pack_bf16x2(p[0], p[1]), pack_bf16x2(p[2], p[3]), pack_bf16x2(p[4], p[5]), pack_bf16x2(p[6], p[7])));
      }
      l += sum;
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int nt = 0; nt < OT; ++nt) {
          const uint4 vv = *reinterpret_cast<const uint4*>(st + kKeyBytes + ((x * d + nt * 32 + r32) * 2 + h) * 16);
          o[nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, vv), pf[x], o[nt], 0, 0, 0);
        }
    }
    l = pair_sum(l);

    // The teams' states of a row meet in LDS; wave (team, half) makes eight of its half's channels a lane.
    __syncthreads();      // (the last tiles have been read)
    float* states = reinterpret_cast<float*>(ring);
    {
      float* mine = states + wave * kWords * 64 + lane;
      mine[0] = m;
      mine[64] = l;
#pragma unroll
      for (int nt = 0; nt < OT; ++nt)
#pragma unroll
        for (int e = 0; e < 16; ++e) mine[(2 + nt * 16 + e) * 64] = o[nt][e];
    }
    __syncthreads();
    if (row_ok) {
      float ms[kTeams], big = -FLT_MAX, total = 0.f, acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < kTeams; ++w) {
        ms[w] = states[(2 * w + half) * kWords * 64 + lane];
        big = fmaxf(big, ms[w]);
      }
#pragma unroll
      for (int w = 0; w < kTeams; ++w) {
        const float* from = states + (2 * w + half) * kWords * 64 + lane;
        const float e = __builtin_amdgcn_exp2f(ms[w] - big);
        total += from[64] * e;
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] += from[(2 + team * 8 + i) * 64] * e;
      }
      const float inv = 1.f / total;
      bf16_t* dst = out + static_cast<int64_t>(row0 + my_row) * out_stride + static_cast<int64_t>(head) * d + team / 2 * 32 + team % 2 * 16 + 4 * h;
#pragma unroll
      for (int j = 0; j < 2; ++j)      // four consecutive channels
        *reinterpret_cast<uint2*>(dst + 8 * j) = make_uint2(pack_bf16x2(acc[4 * j] * inv, acc[4 * j + 1] * inv), pack_bf16x2(acc[4 * j + 2] * inv, acc[4 * j + 3] * inv));
    }
  }
}

}  // namespace alofa

using namespace alofa;

extern "C" int alofa_attention_teams(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* k_cache, const void* v_cache, const int32_t* block_table,
                                     int max_blocks, const int32_t* tiles, int n_tiles, int heads, int kv_heads, int d, int block_size, int window, float scale, hipStream_t stream) {
  ALOFA_REQUIRE(n_tiles > 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0, "attention_teams: tiles=%d heads=%d kv_heads=%d (kv_heads must divide heads)", n_tiles, heads, kv_heads);
  ALOFA_REQUIRE(d == 64 && scale > 0.f, "attention_teams: head size %d (64 is built), scale %g (positive)", d, static_cast<double>(scale));
  ALOFA_REQUIRE(block_size >= 16 && (block_size & (block_size - 1)) == 0 && max_blocks > 0 && window >= 0,
                "attention_teams: block_size=%d must be a power of two, at least 16; max_blocks=%d window=%d", block_size, max_blocks, window);
  ALOFA_REQUIRE(q_stride % 8 == 0 && out_stride % 4 == 0 && reinterpret_cast<uintptr_t>(q) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 8 == 0 &&
                    reinterpret_cast<uintptr_t>(k_cache) % 16 == 0 && reinterpret_cast<uintptr_t>(v_cache) % 16 == 0,
                "attention_teams: q rows and the caches must be 16-byte aligned and out rows 8-byte aligned");
  int bs_shift = 0;
  while ((1 << bs_shift) < block_size) ++bs_shift;
  attention_teams_kernel<<<dim3(n_tiles, heads), 512, 0, stream>>>(static_cast<bf16_t*>(out), out_stride, static_cast<const bf16_t*>(q), q_stride, static_cast<const bf16_t*>(k_cache),
                                                                   static_cast<const bf16_t*>(v_cache), block_table, max_blocks, tiles, heads, kv_heads, bs_shift, window, scale);
  return check_launch("attention_teams");
}
