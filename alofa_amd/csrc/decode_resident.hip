// All layers of a decode step in one launch: pre-norm layers of grouped-query attention (heads of 64, rotary, keys and values in pages) and a
// gated feed-forward, bfloat16 weights and a float32 residual stream, for at most 16 rows (one new token each) of a model whose layer fits the
// chip's registers.
//
// Kernel by kernel a layer of such a step is five launches of 3 to 9 us whose weights (30 MB at a width of 896) would take 6 us at the memory's
// rate: the time goes to launches (1.9 us each, empty), to the first loads of each and to the hand-overs inside them. Here 256 blocks stay for
// the whole step, each owning columns of every matrix, and what a launch boundary did is done by the values themselves:
//
//   * A value that another block needs leaves as eight bytes, the value and the layer's number in the step ("stamp"), in one store to uncached
//     memory. Whoever needs it reads its place until the stamp is the one it waits for. There is no barrier, no flag and no wait for a store's
//     acknowledgement: an exchange among all blocks costs 1.6 us for 896 values and 2.0 for 3,584 (a barrier of flags and a read of data behind
//     it: 3.5 to 3.9).
//   * The weights of the phases ahead are on their way in registers while a phase waits. Loads of a wave come back in order, so a wait for
//     values is also a wait for the weights asked for before it: every phase asks for about as much as an exchange takes to arrive.
//
// A layer is seven exchanges:
//   A  rows -> their norm -> queries, keys, values (a block: 1/256 of the columns; K over the eight waves, sums met in LDS in wave order)
//   B  (row, key head, part of its keys) per block: the new token's query and key turned, its cache slot written, attention over the part
//   C  (row, head) per block: the parts meet in part order
//   D  output projection, residual sum (the block that owns a column of the stream keeps it for the whole step)
//   E  rows -> their norm -> gate and up -> act
//   F  down, K in eight shares (a block: an eighth of K for 1/32 of the columns), float partial sums
//   G  the owner of a column adds the shares in a fixed order to the stream
// A place is written again a layer later by a block that has seen all of G's values, which every block leaves after its last read of the layer
// before: nothing is overwritten that is still waited for.
//
// All blocks have to be on the chip at once. A block takes at most half of a compute unit (eight waves of up to 128 registers, at most 80 KB of
// LDS), so that 256 of them fit beside 256 of another such launch, whatever process it belongs to; kernels that wait for nobody make room by ending.
// No wait is without end: a wave that has asked kLimit times sets `stop` and `failed`, which end every other wait, and what it waited for is NaN from then on.
//
// A step of the 0.5B sizes (24 layers of 896, 14/2 heads, 4,864; the head's 70 us among them), us, kernel by kernel / this: 1 row of 512 keys 643 / 450, 2 667 / 469,
// 4 of 512 to 768 715 / 500, 8 785 / 529, 12 of 64 to 700 890 / 599, 16 of 128 to 1,024 937 / 644, 1 of 4,000 707 / 472, 8 of 3,000 to 4,000 860 / 574. What a layer takes (16 us at
// one row, 19 at eight) is the exchanges, 1.1 to 2.2 us each with the loads that are waited for before them, and 0.5 to 1.3 us of dependent instructions in every phase. Where the
// weights are asked for was found by trying: behind a phase's products and before its barrier, before the values leave, a phase earlier or later cost 1 to 5 %, a single register
// that the compiler keeps in memory 10 (it is read back behind the weights on their way), and weights by pointers of any kind, which LDS's waits wait for too, 15.
//
// Numbers as in the kernels this replaces: the norm's weight on the row rounded to bfloat16 as an operand and the row's factor on the finished
// sum, queries and keys (once, when they have been turned), values, attention's result and act rounded to bfloat16, everything else float.
#include "resident.h"

namespace alofa {

// MB: rows computed (1, 2, 4, 8 or 16; M of them count)
template <int MB>
__global__ void __launch_bounds__(kResThreads, 4) decode_resident_kernel(ResidentArgs a) {
  constexpr int d = 64;
  constexpr int KS = kResMaxWidth / 32 / kResWaves;          // steps of 32 along K a wave takes at most (4)
  constexpr int GT = 3, DT = 2, DK = kResMaxFF / kResShares / 32 / kResWaves;      // tiles of gate and up, of down; down's steps a wave (3)
  constexpr int kRowWaves = MB >= 8 ? 1 : 8 / MB, kRounds = MB == 16 ? 2 : 1;      // waves that share a row on its way in; rows a wave takes one after the other
  constexpr bool kEarlyDown = MB <= 4;                       // (more rows on their way in leave no registers for a part of down's weights as well)
  constexpr int kLdx = kResMaxWidth + 8;                     // bfloat16 numbers from row to row of the operand in LDS (not on the same banks)
  __shared__ __attribute__((aligned(16))) bf16_t xs[MB * kLdx];
  constexpr int kRed = 20;                                   // floats from row to row of a tile's sums
  constexpr int kSums = kResWaves * GT * MB * kRed, kStates = kResWaves * kResMaxGroup * (d + 4);
  __shared__ __attribute__((aligned(16))) float red[kSums > kStates ? kSums : kStates];      // the waves' sums; in B their attention states
  __shared__ __attribute__((aligned(16))) float norms[2][kResMaxWidth];
  __shared__ float ssq[2][MB * kRowWaves];
  __shared__ __attribute__((aligned(16))) uint32_t table[kResMaxLayers * kLayerWords];
  __shared__ __attribute__((aligned(16))) float angles[2][32];
  __shared__ float hs[4 * MB];                               // the block's columns of the stream
  __shared__ __attribute__((aligned(16))) bf16_t qs[(kResMaxGroup + 2) * 72];      // B: the turned queries of the key head (rows 0..), behind them the new key and value
  static_assert(kLdsOf<decltype(xs), decltype(red), decltype(norms), decltype(ssq), decltype(table), decltype(angles), decltype(hs), decltype(qs)> <= kResMostLds,
                "two launches' blocks fit a compute unit");
  // (what follows from these is formed anew in every phase: kept from layer to layer it would take the registers of the weights, and a register that is
  // read back from memory is waited for behind the weights that are on their way)
  int b = blockIdx.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), tid = threadIdx.x, lane = tid % 64, c16 = lane % 16, g = lane / 16;
  int M = a.M, H = a.H, FF = a.FF;
  auto anew = [&]() __attribute__((always_inline)) {
    asm volatile("" : "+v"(tid), "+s"(b), "+s"(wave), "+s"(M), "+s"(H), "+s"(FF));
    lane = tid % 64, c16 = lane % 16, g = lane / 16;
  };
  const int heads = a.heads, kv_heads = a.kv_heads, group = heads / kv_heads, NQ = (heads + 2 * kv_heads) * d, KO = heads * d;

  Wait w;
  w.area = __builtin_amdgcn_make_buffer_rsrc(a.area, 0, kAreaPlaces * 8, 0x00020000);
  w.words = a.area;
  w.failed = a.failed;
  w.limit = a.limit;
  w.dead = false;
  const uint32_t base = static_cast<uint32_t>(__hip_atomic_load(a.area, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));

  // what this block owns: columns of queries, keys and values, of the stream, pairs of act, a share and columns of down
  struct Run {
    int first, n;
  };
  auto run_of = [&](int n) __attribute__((always_inline)) {
    const int first = static_cast<int>(static_cast<uint32_t>(b * n) / kResBlocks);
    return Run{first, static_cast<int>(static_cast<uint32_t>((b + 1) * n) / kResBlocks) - first};
  };
  auto qkv_columns = [&]() __attribute__((always_inline)) { return run_of(NQ); };
  auto own_columns = [&]() __attribute__((always_inline)) { return run_of(H); };
  auto act_pairs = [&]() __attribute__((always_inline)) { return run_of(FF / 2); };
  auto down_columns = [&]() __attribute__((always_inline)) { return Run{(b / kResShares) * (H / 32), H / 32}; };
  auto share_of = [&]() __attribute__((always_inline)) { return b % kResShares; };
  auto share_length = [&]() __attribute__((always_inline)) { return FF / kResShares; };
  const bool attends = b < M * kv_heads * a.parts, meets = b < M * heads;
  const int am = b / (kv_heads * a.parts), ahk = b / a.parts % kv_heads, apart = b % a.parts;      // B's row, key head and part
  const int cm = b / heads, ch = b % heads;                                                         // C's row and head

  // Fragments of weights: lane l of a tile holds eight values of row l % 16 (a row beyond the block's own reads its last one: the sums are not used) from 8 (l / 16) on
  // of a step of 32 along K. A wave's steps come in pairs (whole lines of 128 bytes), every eighth pair; a pair beyond the end reads the first one.
  auto step_of = [&](int j) { return 2 * (wave + kResWaves * (j >> 1)) + (j & 1); };
  u32x4 wq[KS], wo[KS], wg[GT][KS], wd[DT][DK];
  auto row_of = [&](int row, int ld) { return static_cast<uint32_t>(row * ld + g * 8) * 2u; };      // in bytes
  auto fetch_pairs = [&](u32x4 (&to)[KS], gbytes matrix, int64_t row, int K) __attribute__((always_inline)) {
    gbytes first = matrix + (2 * wave < K / 32 ? wave * 128 : 0);
    gbytes second = first + (2 * (wave + kResWaves) < K / 32 ? kResWaves * 128 : 0);
    static_assert(KS == 4, "two pairs");
    to[0] = load_global<u32x4>(first + row);
    to[1] = load_global<u32x4>(first + row + 64);
    to[2] = load_global<u32x4>(second + row);
    to[3] = load_global<u32x4>(second + row + 64);
  };
  auto fetch_cols = [&](u32x4 (&to)[KS], gbytes matrix, int first, int n, int K) __attribute__((always_inline)) {
    fetch_pairs(to, matrix + static_cast<int64_t>(first) * K * 2, row_of(c16 < n ? c16 : n - 1, K), K);
  };
  auto fetch_gate_up = [&](int t, const ResidentLayer& layer) __attribute__((always_inline)) {
    const auto [p0, np] = act_pairs();
    int r = t * 16 + c16;
    r = r < 4 * np ? r : 4 * np - 1;
    const int64_t apart = layer.w_up - layer.w_gate;
    const bool up = r >= 2 * np;
    fetch_pairs(wg[t], layer.w_gate + static_cast<int64_t>(2 * p0) * H * 2, row_of(up ? r - 2 * np : r, H) + (up ? apart : 0), H);
  };
  auto fetch_down = [&](int t, gbytes matrix) __attribute__((always_inline)) {
    const auto [f0, nf] = down_columns();
    const int steps = share_length() / 32;
    gbytes from = matrix + (static_cast<int64_t>(f0) * FF + share_of() * share_length()) * 2;
    const int r = t * 16 + c16;
    const uint32_t row = row_of(r < nf ? r : nf - 1, FF);
#pragma unroll
    for (int j = 0; j < DK; ++j) {
      const int s = wave + kResWaves * j;
      wd[t][j] = load_global<u32x4>(from + (s < steps ? s : 0) * 64 + row);
    }
  };
  // the operand's fragment: row c16 of the rows (beyond M: row M - 1, a column of the result that nobody reads); beyond the last step zeros
  auto operand = [&](int step, int steps) __attribute__((always_inline)) {
    u32x4 x = *reinterpret_cast<const u32x4*>(xs + (c16 < M ? c16 : M - 1) * kLdx + g * 8 + (step < steps ? step : 0) * 32);
    const uint32_t keep = step < steps ? 0xffffffffu : 0u;
    x &= u32x4{keep, keep, keep, keep};
    return __builtin_bit_cast(bf16x8, x);
  };
  auto leave_sums = [&](int tiles, int t, f32x4 acc) __attribute__((always_inline)) {
    if (c16 < M) *reinterpret_cast<f32x4*>(red + ((wave * tiles + t) * MB + c16) * kRed + 4 * g) = acc;
  };
  auto sum_of = [&](int tiles, int t, int m, int n) __attribute__((always_inline)) {
    float v[kResWaves];
#pragma unroll
    for (int i = 0; i < kResWaves; ++i) v[i] = red[((i * tiles + t) * MB + m) * kRed + n];
    float sum = v[0];
#pragma unroll
    for (int i = 1; i < kResWaves; ++i) sum += v[i];
    return sum;
  };

  // --- rows on their way in: a wave takes the runs of 64 pairs of a row (or of its share of one)
  auto in_part_of = [&]() __attribute__((always_inline)) { return kRowWaves > 1 ? wave % kRowWaves : 0; };
  auto in_row = [&](int round) { return kRowWaves > 1 ? wave / kRowWaves : wave + 8 * round; };
  constexpr int kIn = kResMaxWidth / 2 / 64 / kRowWaves;      // pairs of values a lane takes of a row
  auto in_len = [&]() __attribute__((always_inline)) { return (H / 2 + kRowWaves - 1) / kRowWaves; };      // pairs a wave takes
  auto in_at = [&](int i) __attribute__((always_inline)) { return in_part_of() * in_len() + i * 64 + lane; };
  auto in_ok = [&](int i) __attribute__((always_inline)) { return i * 64 + lane < in_len() && in_at(i) < H / 2; };
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  f32x2 nw[2];      // two weights of either norm, on their way to LDS
  float bias = 0.f;    // of the column of queries, keys and values that this thread finishes
  auto fetch_norms = [&](const ResidentLayer& layer) __attribute__((always_inline)) {
    const int at = 2 * tid < H ? 2 * tid : 0;
    nw[0] = *reinterpret_cast<ALOFA_GLOBAL const f32x2*>(layer.norm0 + at);
    nw[1] = *reinterpret_cast<ALOFA_GLOBAL const f32x2*>(layer.norm1 + at);
    const auto [q0, nq] = qkv_columns();
    if (a.has_bias) bias = layer.b_qkv[q0 + ((tid & 15) < nq ? (tid & 15) : 0)];
  };
  auto leave_norms = [&]() __attribute__((always_inline)) {
    if (2 * tid < H) {
      *reinterpret_cast<f32x2*>(norms[0] + 2 * tid) = nw[0];
      *reinterpret_cast<f32x2*>(norms[1] + 2 * tid) = nw[1];
    }
  };
  // the rows (from the area's places from `from` on; kFirst: from the stream itself) times the norm's weight into LDS, their sums of squares beside them
  auto take_rows = [&](int from, bool first, int norm) __attribute__((always_inline)) {
#pragma unroll
    for (int round = 0; round < kRounds; ++round) {
      const int m = in_row(round);
      if (m >= M) continue;
      u32x4 v[kIn];
      if (first) {
#pragma unroll
        for (int i = 0; i < kIn; ++i) {
          const float2 x = *reinterpret_cast<const float2*>(a.hidden + static_cast<int64_t>(m) * H + 2 * (in_ok(i) ? in_at(i) : 0));
          v[i] = u32x4{__float_as_uint(x.x), 0u, __float_as_uint(x.y), 0u};
        }
      } else {
        w.pairs(v, [&](int i) { return from + m * H + 2 * (in_ok(i) ? in_at(i) : in_part_of() * in_len()); });
      }
      // (every lane reads and writes, one without a pair of its own the row's padding: nothing to wait for in between)
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < kIn; ++i) {
        const float x = __uint_as_float(v[i][0]), y = __uint_as_float(v[i][2]);
        const float2 weight = *reinterpret_cast<const float2*>(norms[norm] + 2 * (in_ok(i) ? in_at(i) : 0));
        ss += in_ok(i) ? x * x + y * y : 0.f;
        *reinterpret_cast<uint32_t*>(xs + m * kLdx + (in_ok(i) ? 2 * in_at(i) : kResMaxWidth)) = pack_bf16x2(x * weight.x, y * weight.y);
      }
      ss = wave_sum(ss);
      if (lane == 0) ssq[norm][m * kRowWaves + in_part_of()] = ss;
    }
  };
  auto factor = [&](const float (&squares)[MB * kRowWaves], int m, float eps) __attribute__((always_inline)) {
    float total = squares[m * kRowWaves];
#pragma unroll
    for (int i = 1; i < kRowWaves; ++i) total += squares[m * kRowWaves + i];
    return __builtin_amdgcn_rsqf(total / static_cast<float>(H) + eps);
  };
  // rows that are bfloat16 already: pairs of places, four numbers each; `n`: pairs of places a row has (stride `stride` places)
  auto take_packed = [&](auto most, int from, int stride, int n) __attribute__((always_inline)) {
    constexpr int N = decltype(most)::value;
    const int len = (n + kRowWaves - 1) / kRowWaves, in_part = in_part_of();
#pragma unroll
    for (int round = 0; round < kRounds; ++round) {
      const int m = in_row(round);
      if (m >= M) continue;
      u32x4 v[N];
      auto at = [&](int i) { return in_part * len + i * 64 + lane; };
      auto ok = [&](int i) { return i * 64 + lane < len && at(i) < n; };
      w.pairs(v, [&](int i) { return from + m * stride + 2 * (ok(i) ? at(i) : (in_part * len < n ? in_part * len : 0)); });
#pragma unroll
      for (int i = 0; i < N; ++i) *reinterpret_cast<uint2*>(xs + m * kLdx + (ok(i) ? 4 * at(i) : kResMaxWidth)) = make_uint2(v[i][0], v[i][2]);
    }
  };

  // --- B's share of keys: tiles of 16 keys, two a step, the waves in turn; the pages of a wave's first step and the angles do not change from layer to layer
  const int pos = __builtin_amdgcn_readfirstlane(attends ? a.positions[am] : 0), last = pos >> 4, bs_mask = (1 << a.bs_shift) - 1;
  const int per_part = (last + a.parts) / a.parts;
  const int tile_begin = apart * per_part, tile_end = tile_begin + per_part < last + 1 ? tile_begin + per_part : last + 1;
  const bool writes = attends && tile_begin <= last && last < tile_end;
  const int32_t* pages = a.table + static_cast<int64_t>(am) * a.max_blocks;
  auto page_of = [&](int tile) { return __builtin_amdgcn_readfirstlane(pages[(tile < last ? tile : last) << 4 >> a.bs_shift]); };
  const int first_tile = tile_begin + 2 * wave;
  const bool has_step = attends && first_tile < tile_end;
  int page0 = 0, page1 = 0;
  if (has_step) {
    page0 = page_of(first_tile);
    page1 = page_of(first_tile + 1);
  }
  int64_t new_slot = 0;
  if (attends) {
    if (tid < 32) angles[0][tid] = a.cos_t[static_cast<int64_t>(pos) * 32 + tid], angles[1][tid] = a.sin_t[static_cast<int64_t>(pos) * 32 + tid];
    new_slot = a.slots[am];
    new_slot = static_cast<int64_t>(static_cast<u64>(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(new_slot >> 32)))) << 32 |
                                    static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(new_slot))));
  }
  struct Step {
    u32x4 k[2][2];
    u32x2 v[2][4];
  } st;
  auto fetch_step = [&](Step& s, const ResidentLayer& layer, int tile, int pg0, int pg1) __attribute__((always_inline)) {
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      int key = ((tile + kt) << 4) + c16, key4 = ((tile + kt) << 4) + 4 * g;
      key = key > pos ? pos : key;
      key4 = key4 > (pos & ~3) ? (pos & ~3) : key4;
      const int64_t head_at = (static_cast<int64_t>(kt == 0 ? pg0 : pg1) * kv_heads + ahk) * d;
#pragma unroll
      for (int ds = 0; ds < 2; ++ds)
        s.k[kt][ds] = *reinterpret_cast<ALOFA_GLOBAL const u32x4*>(layer.k_cache + ((head_at << a.bs_shift) + static_cast<int64_t>(key & bs_mask) * d) + ds * 32 + g * 8);
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
        s.v[kt][nt] = *reinterpret_cast<ALOFA_GLOBAL const u32x2*>(layer.v_cache + (((head_at + nt * 16 + c16) << a.bs_shift) + (key4 & bs_mask)));
    }
  };

  // the block's columns of the stream
  if (tid < 4 * MB) {
    const int n = tid & 3, m = tid >> 2;
    const auto [h0, nh] = own_columns();
    if (n < nh && m < M) hs[m * 4 + n] = a.hidden[static_cast<int64_t>(m) * H + h0 + n];
  }
  // the layers' addresses in LDS: a read from memory, where the weights streaming past push them out of the caches, would be waited for in every layer
  for (int i = tid; i < a.n_layers * kLayerWords; i += kResThreads) table[i] = reinterpret_cast<const uint32_t*>(a.layers)[i];
  __syncthreads();
  ResidentLayer layer;
  auto next_layer = [&](int l) __attribute__((always_inline)) {
    uint32_t words[kLayerWords];
#pragma unroll
    for (int i = 0; i < kLayerWords; ++i) words[i] = __builtin_amdgcn_readfirstlane(table[l * kLayerWords + i]);
    layer = __builtin_bit_cast(ResidentLayer, *reinterpret_cast<const LayerWords*>(words));
  };
  next_layer(0);
  fetch_cols(wq, layer.w_qkv, qkv_columns().first, qkv_columns().n, H);
  fetch_norms(layer);
  leave_norms();
  if (has_step) fetch_step(st, layer, first_tile, page0, page1);
  __syncthreads();

#pragma unroll 1
  for (int l = 0; l < a.n_layers; ++l) {
    w.stamp = base + l + 1;
    // ---- A
    anew();
    take_rows(kAtRowsB, l == 0, 0);
    anew();
    const int fn = tid & 15, fm = tid >> 4;      // the output this thread finishes: column, row
    const auto [q0, nq] = qkv_columns();
    __syncthreads();
    const float factor_a = factor(ssq[0], fm < M ? fm : 0, a.eps0);
    {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      bf16x8 x[KS];
#pragma unroll
      for (int j = 0; j < KS; ++j) x[j] = operand(step_of(j), H / 32);
#pragma unroll
      for (int j = 0; j < KS; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wq[j]), x[j], acc, 0, 0, 0);
      leave_sums(1, 0, acc);
    }
    __syncthreads();
    if (fn < nq && fm < M) {
      const float v = sum_of(1, 0, fm, fn) * factor_a + bias;
      put(a.area + kAtQkv + fm * NQ + q0 + fn, v, w.stamp);
    }

    // ---- B
    anew();
    auto fetch_ahead = [&]() __attribute__((always_inline)) {
      fetch_cols(wo, layer.w_o, own_columns().first, own_columns().n, KO);
      fetch_gate_up(0, layer);
    };
    if (!attends) fetch_ahead();
    if (attends) {
      const int item = tid / 16, chan = 2 * (tid % 16);      // head `item` (group: the key, group + 1: the value), channels chan, chan + 1 and their partners 32 on
      if (wave * 4 < group + 2) {      // (all lanes of a wave ask, those without a head of their own for the first one: a wait is a wave's)
        const int row = item < group || item > group + 1 ? ahk * group + (item < group ? item : 0) : item == group ? heads + ahk : heads + kv_heads + ahk;
        const int at = kAtQkv + am * NQ + row * d + chan;
        u32x4 v[2];
        w.pairs(v, [&](int i) { return at + 32 * i; });
        const float a0 = __uint_as_float(v[0][0]), a1 = __uint_as_float(v[0][2]), b0 = __uint_as_float(v[1][0]), b1 = __uint_as_float(v[1][2]);
        uint32_t lo = pack_bf16x2(a0, a1), hi = pack_bf16x2(b0, b1);
        if (item <= group) {
          const float2 angle_c = *reinterpret_cast<const float2*>(angles[0] + chan), angle_s = *reinterpret_cast<const float2*>(angles[1] + chan);
          lo = pack_bf16x2(a0 * angle_c.x - b0 * angle_s.x, a1 * angle_c.y - b1 * angle_s.y);
          hi = pack_bf16x2(b0 * angle_c.x + a0 * angle_s.x, b1 * angle_c.y + a1 * angle_s.y);
        }
        bf16_t* to = qs + (item < group ? item : item - group + kResMaxGroup) * 72 + chan;
        if (item < group + 2) {
          *reinterpret_cast<uint32_t*>(to) = lo;
          *reinterpret_cast<uint32_t*>(to + 32) = hi;
        }
      }
    }
    if (attends) {
      __syncthreads();
      if (writes) {      // the new token's cache slot
        const int64_t head_at = ((new_slot >> a.bs_shift) * kv_heads + ahk) * d;
        const int off = static_cast<int>(new_slot) & bs_mask;
        if (tid < 8) *reinterpret_cast<ALOFA_GLOBAL u32x4*>(layer.k_cache + (head_at << a.bs_shift) + static_cast<int64_t>(off) * d + tid * 8) = *reinterpret_cast<const u32x4*>(qs + kResMaxGroup * 72 + tid * 8);
        if (tid >= 64 && tid < 128) layer.v_cache[((head_at + lane) << a.bs_shift) + off] = qs[(kResMaxGroup + 1) * 72 + lane];
      }
      bf16x8 qf[2];
#pragma unroll
      for (int ds = 0; ds < 2; ++ds) {
        const uint4 x = *reinterpret_cast<const uint4*>(qs + (c16 < group ? c16 : 0) * 72 + ds * 32 + g * 8);
        qf[ds] = __builtin_bit_cast(bf16x8, x);
      }
      f32x4 o[4];
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) o[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
      float mx = -FLT_MAX, sum = 0.f;
      const float scale2 = a.scale * 1.44269504088896340736f;
#pragma unroll 1
      for (int tile = first_tile; tile < tile_end;) {
        const bool last_here = tile + 1 >= last;
        f32x4 s[2];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
          s[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
          const bool new_row = last_here && tile + kt == last && c16 == (pos & 15);
#pragma unroll
          for (int ds = 0; ds < 2; ++ds) {
            u32x4 kf = st.k[kt][ds];
            if (last_here) {      // (the new token's key is not in the cache yet)
              const u32x4 new_k = *reinterpret_cast<const u32x4*>(qs + kResMaxGroup * 72 + ds * 32 + g * 8);
              kf.x = new_row ? new_k.x : kf.x;
              kf.y = new_row ? new_k.y : kf.y;
              kf.z = new_row ? new_k.z : kf.z;
              kf.w = new_row ? new_k.w : kf.w;
            }
            s[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kf), qf[ds], s[kt], 0, 0, 0);
          }
        }
        float pw[8], step_max = -FLT_MAX;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int key = ((tile + i / 4) << 4) + 4 * g + i % 4;
          pw[i] = key <= pos && tile + i / 4 < tile_end ? s[i / 4][i % 4] * scale2 : -FLT_MAX;
          step_max = fmaxf(step_max, pw[i]);
        }
        step_max = rows_max(step_max);
        const float m_new = fmaxf(mx, step_max), corr = __builtin_amdgcn_exp2f(mx - m_new);
        mx = m_new;
        float add = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          pw[i] = pw[i] <= -FLT_MAX ? 0.f : __builtin_amdgcn_exp2f(pw[i] - m_new);      // (a score that is no number stays one)
          add += pw[i];
        }
        sum = sum * corr + add;
        const bf16x8 pf = __builtin_bit_cast(bf16x8, make_uint4(pack_bf16x2(pw[0], pw[1]), pack_bf16x2(pw[2], pw[3]), pack_bf16x2(pw[4], pw[5]), pack_bf16x2(pw[6], pw[7])));
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
          o[nt] *= corr;
          uint32_t vw[4] = {st.v[0][nt].x, st.v[0][nt].y, st.v[1][nt].x, st.v[1][nt].y};
          if (last_here) {      // what lies beyond the new token is cleared, the new token's value takes its place
            const uint32_t new_v = qs[(kResMaxGroup + 1) * 72 + nt * 16 + c16];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int key = ((tile + i / 2) << 4) + 4 * g + 2 * (i % 2);
              vw[i] &= (key <= pos ? 0x0000ffffu : 0u) | (key + 1 <= pos ? 0xffff0000u : 0u);
              const uint32_t ins = (pos & 1) ? ((vw[i] & 0x0000ffffu) | (new_v << 16)) : ((vw[i] & 0xffff0000u) | new_v);
              vw[i] = key == (pos & ~1) ? ins : vw[i];
            }
          }
          o[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, make_uint4(vw[0], vw[1], vw[2], vw[3])), pf, o[nt], 0, 0, 0);
        }
        tile += 2 * kResWaves;
        if (tile < tile_end) fetch_step(st, layer, tile, page_of(tile), page_of(tile + 1));
      }
      fetch_ahead();
      sum = rows_sum(sum);
      float* mine = red + (wave * kResMaxGroup + c16) * (d + 4);
      if (g == 0 && c16 < kResMaxGroup) {
        mine[0] = mx;
        mine[1] = sum;
      }
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
        if (c16 < kResMaxGroup) *reinterpret_cast<f32x4*>(mine + 4 + nt * 16 + 4 * g) = o[nt];
      __syncthreads();
      for (int x = tid; x < group * d; x += kResThreads) {
        const int i = x / d, c = x % d;
        float big = red[i * (d + 4)];
#pragma unroll
        for (int v = 1; v < kResWaves; ++v) big = fmaxf(big, red[(v * kResMaxGroup + i) * (d + 4)]);
        float total = 0.f, acc = 0.f;
#pragma unroll
        for (int v = 0; v < kResWaves; ++v) {
          const float* from = red + (v * kResMaxGroup + i) * (d + 4);
          const float e = __builtin_amdgcn_exp2f(from[0] - big);
          total += from[1] * e;
          acc += from[4 + c] * e;
        }
        u64* to = a.area + kAtParts + static_cast<int64_t>((am * heads + ahk * group + i) * a.parts + apart) * 66;
        put(to + 2 + c, acc, w.stamp);
        if (c < 2) put(to + c, c == 0 ? big : total, w.stamp);
      }
    }

    // ---- C
    anew();
    if (meets) {
      float big = -FLT_MAX, total = 0.f, acc = 0.f;
      float ms[2], ls[2], vs[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int part = wave + kResWaves * i;
        ms[i] = -FLT_MAX, ls[i] = 0.f, vs[i] = 0.f;
        if (part < a.parts) {
          const int at = kAtParts + ((cm * heads + ch) * a.parts + part) * 66;
          u32x4 v[2];
          w.pairs(v, [&](int n) { return at + (n == 0 ? 0 : 2 + (lane & ~1)); });
          ms[i] = __uint_as_float(v[0][0]), ls[i] = __uint_as_float(v[0][2]), vs[i] = __uint_as_float((lane & 1) ? v[1][2] : v[1][0]);
        }
      }
      big = fmaxf(ms[0], ms[1]);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float e = __builtin_amdgcn_exp2f(ms[i] - big);
        total += ls[i] * e;
        acc += vs[i] * e;
      }
      __syncthreads();      // (B's states have been read)
      red[wave * 68 + 4 + lane] = acc;
      if (lane == 0) {
        red[wave * 68] = big;
        red[wave * 68 + 1] = total;
      }
      __syncthreads();
      if (wave == 0) {
        big = red[0];
#pragma unroll
        for (int v = 1; v < kResWaves; ++v) big = fmaxf(big, red[v * 68]);
        total = 0.f, acc = 0.f;
#pragma unroll
        for (int v = 0; v < kResWaves; ++v) {
          const float e = __builtin_amdgcn_exp2f(red[v * 68] - big);
          total += red[v * 68 + 1] * e;
          acc += red[v * 68 + 4 + lane] * e;
        }
        const float x = acc / total, y = lane_xor1(x);
        if ((lane & 1) == 0) put(a.area + kAtAttn + cm * (KO / 2) + ch * 32 + lane / 2, pack_bf16x2(x, y), w.stamp);
      }
    }

    // ---- D
    anew();
    fetch_gate_up(1, layer);
    if (kEarlyDown) fetch_down(0, layer.w_down);
    take_packed(std::integral_constant<int, (kResMaxWidth / 4 / 64 + kRowWaves - 1) / kRowWaves>(), kAtAttn, KO / 2, KO / 4);
    __syncthreads();
    {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      bf16x8 x[KS];
#pragma unroll
      for (int j = 0; j < KS; ++j) x[j] = operand(step_of(j), KO / 32);
#pragma unroll
      for (int j = 0; j < KS; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wo[j]), x[j], acc, 0, 0, 0);
      leave_sums(1, 0, acc);
    }
    __syncthreads();
    const int on = tid & 15, om = tid >> 4;
    const auto [h0, nh] = own_columns();
    if (on < nh && om < M) {
      const float v = hs[om * 4 + on] + sum_of(1, 0, om, on);
      hs[om * 4 + on] = v;
      put(a.area + kAtRowsA + om * H + h0 + on, v, w.stamp);
    }

    // ---- E
    anew();
    fetch_gate_up(2, layer);
    take_rows(kAtRowsA, false, 1);
    anew();
    __syncthreads();
    const float factor_e = factor(ssq[1], (tid >> 5) < M ? tid >> 5 : 0, a.eps1);
    {
      f32x4 acc[GT];
      bf16x8 x[KS];
#pragma unroll
      for (int t = 0; t < GT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < KS; ++j) x[j] = operand(step_of(j), H / 32);
#pragma unroll
      for (int j = 0; j < KS; ++j)
#pragma unroll
        for (int t = 0; t < GT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wg[t][j]), x[j], acc[t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < GT; ++t) leave_sums(GT, t, acc[t]);
    }
    __syncthreads();
    {
      const int n = tid & 31, m = tid >> 5;      // column 2 p0 + n of act
      const auto [p0, np] = act_pairs();
      if (n < 2 * np && m < M) {
        const int u = 2 * np + n;
        const float f = factor_e;
        const float gate = sum_of(GT, n >> 4, m, n & 15) * f, up = sum_of(GT, u >> 4, m, u & 15) * f;
        const float x = gate_of<false>(gate) * up, y = lane_xor1(x);
        if ((n & 1) == 0) put(a.area + kAtAct + m * (FF / 2) + p0 + n / 2, pack_bf16x2(x, y), w.stamp);
      }
    }

    // ---- F
    anew();
    if (!kEarlyDown) fetch_down(0, layer.w_down);
    fetch_down(1, layer.w_down);
    take_packed(std::integral_constant<int, (kResMaxFF / kResShares / 4 / 64 + kRowWaves - 1) / kRowWaves>(), kAtAct + share_of() * (share_length() / 2), FF / 2, share_length() / 4);
    __syncthreads();
    {
      f32x4 acc[DT];
#pragma unroll
      for (int t = 0; t < DT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < DK; ++j) {
        const bf16x8 x = operand(wave + kResWaves * j, share_length() / 32);
#pragma unroll
        for (int t = 0; t < DT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wd[t][j]), x, acc[t], 0, 0, 0);
      }
#pragma unroll
      for (int t = 0; t < DT; ++t) leave_sums(DT, t, acc[t]);
    }
    __syncthreads();
    {
      const int n = tid & 31, m = tid >> 5;
      const auto [f0, nf] = down_columns();
      if (n < nf && m < M) put(a.area + kAtDown + ((f0 + n) * M + m) * kResShares + share_of(), sum_of(DT, n >> 4, m, n & 15), w.stamp);
    }

    // ---- G
    anew();
    const bool more = l + 1 < a.n_layers;
    next_layer(more ? l + 1 : l);      // (behind the last layer its own once more: a load under a condition would keep the old registers)
    fetch_cols(wq, layer.w_qkv, qkv_columns().first, qkv_columns().n, H);
    fetch_norms(layer);
    {
      const int m = tid / 16, n = tid / 4 % 4, pair = tid % 4;      // two shares a thread
      const auto [h0, nh] = own_columns();
      const int first = h0, own = nh;
      const bool mine = m < M && n < own;
      u32x4 v[1] = {u32x4{0u, 0u, 0u, 0u}};
      if (wave * 4 < M) w.pairs(v, [&](int) { return kAtDown + ((first + (n < own ? n : 0)) * M + (m < M ? m : 0)) * kResShares + 2 * pair; });
      float sum = __uint_as_float(v[0][0]) + __uint_as_float(v[0][2]);
      sum += lane_xor1(sum);
      sum += lane_xor2(sum);
      if (mine && pair == 0) {
        const float x = hs[m * 4 + n] + sum;
        hs[m * 4 + n] = x;
        if (more) put(a.area + kAtRowsB + m * H + h0 + n, x, w.stamp + 1);
        else a.hidden[static_cast<int64_t>(m) * H + h0 + n] = x;
      }
    }
    if (has_step) fetch_step(st, layer, first_tile, page0, page1);
    else st = Step{};      // (nothing of the layer before is kept)
    leave_norms();
    __syncthreads();      // (and the waves without a column wait here and not by asking for rows that cannot be there yet)
  }
  // the next step's stamps go on from here (every block has read `base` before this one could finish its last layer)
  if (b == 0 && tid == 0) __hip_atomic_store(a.area, static_cast<u64>(base + a.n_layers), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int MB>
static int launch_resident(const ResidentArgs& a, hipStream_t stream) {
  decode_resident_kernel<MB><<<kResBlocks, kResThreads, 0, stream>>>(a);
  return check_launch("decode_resident");
}

}  // namespace alofa

// Bytes of an area (uncached device memory; it is never given back to the runtime: tensors that took the place of such memory have held wrong values).
extern "C" int64_t alofa_resident_area_bytes() { return static_cast<int64_t>(alofa::kAreaPlaces) * 8 * alofa::kResGroups; }

// An area as it was when new, zeros, behind everything that the device has been given. Not to be called under graph capture.
extern "C" int alofa_resident_area_clear(void* area) {
  using namespace alofa;
  ALOFA_REQUIRE(area, "resident_area_clear: no area");
  hipError_t e = hipDeviceSynchronize();
  if (e == hipSuccess) e = hipMemset(area, 0, alofa_resident_area_bytes());
  if (e == hipSuccess) e = hipDeviceSynchronize();
  ALOFA_REQUIRE(e == hipSuccess, "resident_area_clear: %s", hipGetErrorString(e));
  return 0;
}

// A new area, zeros. Not to be called under graph capture.
extern "C" int alofa_resident_area(void** area) {
  using namespace alofa;
  *area = nullptr;
  const hipError_t e = hipExtMallocWithFlags(area, alofa_resident_area_bytes(), hipDeviceMallocUncached);
  if (e != hipSuccess) static_cast<void>(hipGetLastError());      // (the caller goes on without one: not the next launch's error)
  ALOFA_REQUIRE(e == hipSuccess, "resident_area: %s", hipGetErrorString(e));
  return alofa_resident_area_clear(*area);
}

// How many blocks share a row and key head's keys: as many as there are blocks for, at most sixteen.
extern "C" int alofa_resident_parts(int M, int kv_heads) {
  const int parts = alofa::kResBlocks / (M * kv_heads);
  return parts < alofa::kResMaxParts ? parts : alofa::kResMaxParts;
}

// Whether a model of these sizes runs in one launch: a block's columns of every matrix have to fit the registers they are fetched into.
extern "C" int alofa_resident_takes(int H, int FF, int heads, int kv_heads, int d, int page) {
  using namespace alofa;
  return d == 64 && H % 64 == 0 && H >= kResBlocks && H <= kResMaxWidth && FF % (32 * kResShares) == 0 && FF >= 2 * kResBlocks && FF <= kResMaxFF && heads > 0 && kv_heads > 0 &&
         heads % kv_heads == 0 && heads / kv_heads <= kResMaxGroup && heads * d <= kResMaxWidth && (heads + 2 * kv_heads) * d >= kResBlocks && (heads + 2 * kv_heads) * d <= 16 * kResBlocks &&
         page >= 16 && (page & (page - 1)) == 0 && compute_units() >= kResBlocks;
}

// hidden [M, H] float32, in and out; layers: n_layers x ten pointers (ResidentLayer) in device memory; positions [M], table [M, max_blocks], slots [M]: the new token's
// place per row, row i request i; cos, sin [positions, 32]; area: of alofa_resident_area, of one launch at a time; failed: an int in memory that the host reads, set if a wait is given up;
// limit: after how many asks (0: kLimit). tiled (more than sixteen rows): the layers' gate, up and down are laid out in tiles (decode_groups.hip).
extern "C" int alofa_decode_resident(float* hidden, const void* layers, const int32_t* positions, const int32_t* table, const int64_t* slots, const float* cos_t,
                                     const float* sin_t, void* area, int* failed, int n_layers, int M, int H, int FF, int heads, int kv_heads, int d, int page, int max_blocks,
                                     int has_bias, int limit, int tiled, float scale, float eps0, float eps1, hipStream_t stream) {
  using namespace alofa;
  ALOFA_REQUIRE(alofa_resident_takes(H, FF, heads, kv_heads, d, page) && M >= 1 && M <= alofa_resident_rows(H, FF, heads, kv_heads) && (M > kResMaxRows || (M * kv_heads <= kResBlocks && M * heads <= kResBlocks)) && n_layers > 0 && n_layers <= kResMaxLayers && max_blocks > 0,
                "decode_resident: sizes beyond what a block holds (M=%d H=%d FF=%d heads=%d/%d d=%d page=%d)", M, H, FF, heads, kv_heads, d, page);
  ALOFA_REQUIRE(!tiled || M > kResMaxRows, "decode_resident: up to %d rows read the matrices as they are", kResMaxRows);
  ALOFA_REQUIRE(hidden && layers && positions && table && slots && cos_t && sin_t && area && failed, "decode_resident: an operand is missing");
  int shift = 0;
  while ((1 << shift) < page) ++shift;
  const ResidentArgs a = {hidden, static_cast<const ResidentLayer*>(layers), positions, table, slots, cos_t, sin_t, static_cast<u64*>(area), failed, n_layers, M, H, FF, heads, kv_heads,
                          max_blocks, shift, alofa_resident_parts(M, kv_heads), has_bias, limit > 0 ? limit : kLimit, scale, eps0, eps1};
  if (M > kResMaxRows) return launch_groups(a, tiled != 0, stream);
  if (M == 1) return launch_resident<1>(a, stream);
  if (M == 2) return launch_resident<2>(a, stream);
  if (M <= 4) return launch_resident<4>(a, stream);
  if (M <= 8) return launch_resident<8>(a, stream);
  return launch_resident<16>(a, stream);
}
