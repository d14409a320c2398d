// All layers of a decode step in one launch, for 17 to 64 rows: the layers and the exchanges of decode_resident.hip, whose comment says how values are handed over and
// why nothing is overwritten that is still waited for, with the 256 blocks in G groups (two up to 32 rows, four beyond) that each take up to sixteen of the rows
// through all layers by themselves.
//
// What bounds it is what a compute unit takes in. All blocks reading all rows would be 64 x 896 values of eight bytes in four of a layer's exchanges. Within a group a block reads sixteen rows
// and G / 256 of the weights instead; the G blocks with the same columns lie on one die (block b on die b % 8), so that its L2 serves G - 1 of them and memory is read about once. For that the
// weights no longer fit the registers: gate, up and down go through a ring of fragments in a phase, the first of them asked for before the phase's values are waited for, as all weights are there.
// A compute unit takes a fragment of a row-major matrix (1 KB, sixteen rows' 64 bytes: sixteen lanes in a row bring sixteen lines) in 27 ns however many are on their way, 37 bytes a nanosecond, 1 KB
// in one piece in 10 to 17: gate and up's 280 fragments of a block at four groups 7.5 us, down's 140 3.8. So these matrices come laid out in tiles, fragment behind fragment as the matrix cores take them
// (kTiled; ops.in_tiles: copies, 26 MB a layer at the 0.5B sizes, made once per model when a step first needs them), and blocks take whole tiles of them; where there is no room for copies, or none that
// follow what is written to the matrices, a step reads these as they are: the same bits. Eight steps of the 0.5B sizes with logits behind
// the last, us, rows of the matrices / tiles: 64 rows of 128 to 2,048 keys 8,194 / 7,300, of 64 to 256 7,502 / 6,543, of 3,300 to 4,000 11,361 / 10,381, 48 of 128 to 1,024 7,372 / 6,485, 33 of 64 to 512
// 7,068 / 6,195, 32 of 128 to 1,024 6,055 / 5,795, 17 of 64 to 700 5,711 / 5,405. Other widths (256 to 1,024) and feed-forwards (512 to 5,120), 12 layers, rows of 100 to 290 keys: 1.00 to 1.07 times as fast
// at 17 and 32 rows, 1.06 to 1.18 at 33 and 64. Loads marked as read once (nt) lose half of it at four groups (7,806 for 7,374): the L2's other three readers; past the L1 (sc0) is even.
//
// A step of the 0.5B sizes before that (24 layers; the head's 70 us among them), us, kernel by kernel / this: 17 rows of 64 to 700 keys 1,101 / 712, 32 of 128 to 1,024 1,185 / 754, 48 of 128 to 1,024
// 1,312 / 917, 64 of 128 to 2,048 1,363 / 1,023, 64 of 3,300 to 4,000 1,676 / 1,360. Other widths from 256 (one key head) to 1,024 (four), 24 layers, 17 to 64 rows of 200 to 1,000 keys: 1.25 to 1.83 times
// as fast. Tried on the way: without the halves of a line side by side, with the waves' steps in pairs of which some are beyond the end, one number of parts for all keys
// 1,071 at 64 rows; gate's, up's and down's lines asked for into the L2 in phase B, one number a line: the phases that read them 1.4 us less, B 4 us more.
//
//   * A row leaves its owner times the next norm's weight, rounded to bfloat16, two columns a place, with the sum of the squares of the owner's columns beside it: what
//     all readers of float values would form is formed once, and a row is H / 2 + 256 / G places instead of H.
//   * The rows are dealt to the groups by length (the longest to one after the other, then back), and a group's blocks to its rows' keys in proportion to their number, so that groups and
//     blocks end at about the same time whatever the lengths.
//   * Several output tiles a wave and K over four waves instead of eight: gate's tiles are four waves', up's the other four's.
//   * Phase B is decode_resident.hip's with values by sixteen bytes: masks, the new token's place and the states' end are the same in both.
//
// The compiler keeps two registers of a lane in memory (12 bytes; three, 16, with four groups and the matrices as they are; decode_resident.hip has none, whose comment says what one costs there; here it was not
// measured apart). A block's LDS, 64,580 and 80,964 bytes, leaves room for another launch's block in the compute unit (kLdsOf).
#include "resident.h"

namespace alofa {

// row_ror:4 and row_half_mirror within rows of sixteen lanes
__device__ __forceinline__ float lane_ror4(float v) { return dpp_move<0x124, 0xf>(0.f, v); }
__device__ __forceinline__ float lane_mirror8(float v) { return dpp_move<0x141, 0xf>(0.f, v); }

constexpr int kRowPlaces = kResMaxWidth / 2 + 128;      // of a row on its way: pairs of columns, behind them the blocks' sums of squares
constexpr int kColumnPlaces = kResMaxWidth;             // of down's sums: a share and row's columns
constexpr int kQkvMost = 2048;                          // columns of queries, keys and values
static_assert(kRowPlaces <= kResMaxWidth && kQkvMost <= 4096, "the places lie where decode_resident.hip has them");

// kTiled: gate, up and down laid out in tiles
template <int G, int GS, bool kTiled>
__global__ void __launch_bounds__(kResThreads, 4) decode_groups_kernel(ResidentArgs a) {
  constexpr int d = 64, MB = kResMaxRows, NB = kResBlocks / G;      // NB: blocks of a group
  constexpr int QT = G == 4 ? 2 : 1, QK = 8 / QT, QS = 32 / QK;     // queries, keys, values: tiles, waves that share K, steps of a wave
  constexpr int GT = G == 4 ? 5 : 3;                                // gate and up: tiles of either; K over four waves, GS steps each at most
  constexpr int DT = G == 4 ? 4 : 2, DS = 5;                        // down: tiles of half of the waves, steps of a wave
  constexpr int kRing = 16, kFirst = kTiled && G == 4 ? 4 : 8, kBefore = kTiled && G == 4 ? 8 : 10;                             // fragments of a wave on their way, and of them before attention's values are there
  constexpr int kLdx = kResMaxWidth + 8;
  constexpr int kStates = kResWaves * kResMaxGroup * (d + 4), kSums = 2 * GT * 4 * 256, kQsAt = kStates;
  static_assert(kSums * 4 >= (kStates + 10 * 72 / 2) * 4, "queries lie behind the attention states");
  __shared__ __attribute__((aligned(16))) bf16_t xs[MB * kLdx];
  __shared__ __attribute__((aligned(16))) float red[kSums];      // the waves' sums, [tile][wave][row][column]; in B their attention states, behind them the turned queries
  __shared__ float ssq[2][MB];
  __shared__ __attribute__((aligned(16))) uint32_t table[kResMaxLayers * kLayerWords];
  __shared__ __attribute__((aligned(16))) float angles[2][32];
  __shared__ __attribute__((aligned(16))) float hs[MB * 16];     // the block's columns of the stream
  __shared__ int rows_of[MB], parts_of[MB], first_of[MB], order[64], n_rows;
  static_assert(kLdsOf<decltype(xs), decltype(red), decltype(ssq), decltype(table), decltype(angles), decltype(hs), decltype(rows_of), decltype(parts_of), decltype(first_of), decltype(order),
                       decltype(n_rows)> <= kResMostLds, "two launches' blocks fit a compute unit");
  bf16_t* qs = reinterpret_cast<bf16_t*>(red + kQsAt);           // B: the turned queries of the key head (rows 0..), behind them the new key and value
  const int b = blockIdx.x;
  int s = b / (8 * G) * 8 + b % 8, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), tid = threadIdx.x, lane = tid % 64, c16 = lane % 16, g = lane / 16;
  const int grp = b / 8 % G;
  int H = a.H, FF = a.FF;
  auto anew = [&]() __attribute__((always_inline)) {
    asm volatile("" : "+v"(tid), "+s"(s), "+s"(wave), "+s"(H), "+s"(FF));
    lane = tid % 64, c16 = lane % 16, g = lane / 16;
  };
  const int heads = a.heads, kv_heads = a.kv_heads, group = heads / kv_heads, NQ = (heads + 2 * kv_heads) * d, KO = heads * d;
  const int blocks_a_head = NB / kv_heads;

  u64* area = a.area + static_cast<int64_t>(grp) * kAreaPlaces;      // (the group's; the word that ends all waits is the first group's)
  Wait w;
  w.area = __builtin_amdgcn_make_buffer_rsrc(area, 0, kAreaPlaces * 8, 0x00020000);
  w.words = a.area;
  w.failed = a.failed;
  w.limit = a.limit;
  w.dead = false;
  const uint32_t base = static_cast<uint32_t>(__hip_atomic_load(area, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));

  // --- which rows are the group's, and which blocks take which of their keys: by the number of tiles of sixteen keys
  if (wave == 0) {
    const int mine = lane < a.M ? (a.positions[lane] >> 4) + 1 : 0;
    int rank = 0;
    for (int k = 0; k < a.M; ++k) {
      const int other = __builtin_amdgcn_readlane(mine, k);
      rank += other > mine || (other == mine && k < lane);
    }
    if (lane < a.M) order[rank] = lane;
    wave_lds_sync();
    const int at = lane * G + ((lane & 1) ? G - 1 - grp : grp);
    const bool has = lane < MB && at < a.M;
    const int n = __popcll(__ballot(has));
    const int row = has ? order[at] : 0, tiles = has ? (a.positions[row] >> 4) + 1 : 0;
    int all = 0;
    for (int k = 0; k < MB; ++k) all += __builtin_amdgcn_readlane(tiles, k);
    // as many parts as it takes for none to have more tiles than a quota, the least of 64 between an even share of all and one that always fits for which the blocks suffice
    const int least = (all + blocks_a_head - 1) / blocks_a_head, spare = blocks_a_head - n, most = spare > 0 ? (all + spare - 1) / spare : all;
    const int step = (most - least) / 63 + 1, tried = least + lane * step;
    int blocks = 0;
    for (int k = 0; k < MB; ++k) blocks += (__builtin_amdgcn_readlane(tiles, k) + tried - 1) / tried;
    const u64 fit = __ballot(blocks <= blocks_a_head);
    int quota = least + (fit != 0 ? __ffsll(fit) - 1 : 63) * step;
    quota = fit == 0 || quota > all ? all : quota;
    quota = quota < 2 * kResWaves ? 2 * kResWaves : quota;      // (a part with less than a step for every wave saves nothing)
    int parts = (tiles + quota - 1) / quota;
    parts = parts < kResMaxParts ? parts : kResMaxParts;      // (such a row's parts are longer than the quota, and what the phase waits for: blocks that it leaves would shorten others' parts only)
    int first = 0;
    for (int k = 0; k < MB; ++k) {
      const int p = __builtin_amdgcn_readlane(parts, k);
      first += k < lane ? p : 0;
    }
    if (lane < MB) rows_of[lane] = row, parts_of[lane] = parts, first_of[lane] = first;
    if (lane == 0) n_rows = n;
  }
  // the layers' addresses in LDS, as in decode_resident.hip
  for (int i = tid; i < a.n_layers * kLayerWords; i += kResThreads) table[i] = reinterpret_cast<const uint32_t*>(a.layers)[i];
  __syncthreads();
  const int M = __builtin_amdgcn_readfirstlane(n_rows);

  struct Run {
    int first, n;
  };
  auto run_of = [&](int n) __attribute__((always_inline)) {
    const int first = static_cast<int>(static_cast<uint32_t>(s * n) / NB);
    return Run{first, static_cast<int>(static_cast<uint32_t>((s + 1) * n) / NB) - first};
  };
  auto qkv_columns = [&]() __attribute__((always_inline)) { return run_of(NQ); };
  auto own_pairs = [&]() __attribute__((always_inline)) { return run_of(H / 2); };
  // gate, up and down in tiles are dealt out in whole ones, of sixteen rows of theirs
  auto act_tiles = [&]() __attribute__((always_inline)) { return run_of(FF / 16); };      // (none where the tiles are fewer than the blocks)
  auto act_pairs = [&]() __attribute__((always_inline)) {
    if constexpr (!kTiled) return run_of(FF / 2);
    const auto [t0, nt] = act_tiles();
    return Run{8 * t0, 8 * nt};
  };
  auto down_tiles = [&]() __attribute__((always_inline)) {
    constexpr int kParts = NB / kResShares;
    const int part = s / kResShares, first = static_cast<int>(static_cast<uint32_t>(part * (H / 16)) / kParts);
    return Run{first, static_cast<int>(static_cast<uint32_t>((part + 1) * (H / 16)) / kParts) - first};
  };
  auto down_columns = [&]() __attribute__((always_inline)) {
    if constexpr (!kTiled) return Run{(s / kResShares) * (H * kResShares / NB), H * kResShares / NB};
    const auto [t0, nt] = down_tiles();
    return Run{16 * t0, 16 * nt};
  };
  auto share_of = [&]() __attribute__((always_inline)) { return s % kResShares; };
  auto share_length = [&]() __attribute__((always_inline)) { return FF / kResShares; };

  // Fragments of weights: lane l of a tile holds eight values of row l % 16 (beyond the block's own: its last one, whose sums are not used) from 8 (l / 16) on of a step
  // of 32 along K; a wave's steps come in pairs (whole lines of 128 bytes), every so-manieth pair; a pair beyond the end reads the first one.
  auto row_at = [&](int row, int n, int ld) __attribute__((always_inline)) { return static_cast<uint32_t>((row < n ? row : n - 1) * ld + g * 8) * 2u; };
  auto fragment = [&](gbytes from, uint32_t row, int step, int steps) __attribute__((always_inline)) {
    const int pair = step & ~1;
    return load_global<u32x4>(from + (pair < steps ? pair : 0) * 64 + (step & 1) * 64 + row);
  };
  // step j of a wave whose number among the n that share K is k
  auto step_of = [](int k, int n, int j) __attribute__((always_inline)) { return 2 * (k + n * (j >> 1)) + (j & 1); };
  auto operand = [&](int step, int steps) __attribute__((always_inline)) {
    const bool in = step >= 0 && step < steps;
    u32x4 x = *reinterpret_cast<const u32x4*>(xs + (c16 < M ? c16 : M - 1) * kLdx + g * 8 + (in ? step : 0) * 32);
    const uint32_t keep = in ? 0xffffffffu : 0u;
    x &= u32x4{keep, keep, keep, keep};
    return __builtin_bit_cast(bf16x8, x);
  };
  auto leave_sums = [&](int tile, int n, int k, f32x4 acc) __attribute__((always_inline)) { *reinterpret_cast<f32x4*>(red + ((tile * n + k) * 16 + c16) * 16 + 4 * g) = acc; };
  auto sum_of = [&](int tile, auto waves, int m, int n) __attribute__((always_inline)) {
    constexpr int N = decltype(waves)::value;
    float v[N];
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = red[((tile * N + i) * 16 + m) * 16 + n];
    float sum = v[0];
#pragma unroll
    for (int i = 1; i < N; ++i) sum += v[i];
    return sum;
  };
  typedef std::integral_constant<int, 4> Four;
  typedef std::integral_constant<int, 8> Eight;
  u32x4 wq[QS], wo[4], wg[kRing], wd[kRing];
  auto fetch_qkv = [&](const ResidentLayer& layer) __attribute__((always_inline)) {
    const auto [q0, nq] = qkv_columns();
    gbytes from = layer.w_qkv + static_cast<int64_t>(q0) * H * 2;
    const uint32_t row = row_at((QT > 1 ? wave / QK : 0) * 16 + c16, nq, H);
#pragma unroll
    for (int j = 0; j < QS; ++j) wq[j] = fragment(from, row, step_of(wave % QK, QK, j), H / 32);
  };
  auto fetch_out = [&](const ResidentLayer& layer) __attribute__((always_inline)) {
    const auto [p0, np] = own_pairs();
    gbytes from = layer.w_o + static_cast<int64_t>(2 * p0) * KO * 2;
    const uint32_t row = row_at(c16, 2 * np, KO);
#pragma unroll
    for (int j = 0; j < 4; ++j) wo[j] = fragment(from, row, step_of(wave, 8, j), KO / 32);
  };
  // Gate, up and down: a run of steps a wave, K over four waves. Fragment i: i / 2 of (pair of the run's steps, tile), its first or second half, the last step's tiles by themselves: the halves of a
  // line are asked for one behind the other; when the second is asked for later, the line has been pushed out of the L1 and is fetched again.
  auto run_step = [&](int j, int steps) __attribute__((always_inline)) {
    const int each = (steps + 3) / 4, step = (wave & 3) * each + j;
    return j < each && step < steps ? step : -1;
  };
  constexpr auto step_at = [](int i, int tiles, int n) { return i / (2 * tiles) * 2 + 1 < n ? i / (2 * tiles) * 2 + i % 2 : n - 1; };
  constexpr auto tile_at = [](int i, int tiles, int n) { return i / (2 * tiles) * 2 + 1 < n ? i / 2 % tiles : i % (2 * tiles); };
  auto fetch_gate_up = [&](u32x4& to, const ResidentLayer& layer, int i) __attribute__((always_inline)) {
    const int step = run_step(step_at(i, GT, GS), H / 32), tile = tile_at(i, GT, GS);
    if constexpr (!kTiled) {
      const auto [p0, np] = act_pairs();
      gbytes from = (wave < 4 ? layer.w_gate : layer.w_up) + static_cast<int64_t>(2 * p0) * H * 2;
      to = load_global<u32x4>(from + (step >= 0 ? step : 0) * 64 + row_at(tile * 16 + c16, 2 * np, H));
      return;
    }
    const auto [t0, nt] = act_tiles();
    to = load_global<u32x4>((wave < 4 ? layer.w_gate : layer.w_up) + static_cast<uint32_t>((t0 + (tile < nt ? tile : nt > 0 ? nt - 1 : 0)) * (H / 32) + (step >= 0 ? step : 0)) * 1024u + lane * 16);
  };
  auto fetch_down = [&](u32x4& to, const ResidentLayer& layer, int i) __attribute__((always_inline)) {
    const int steps = share_length() / 32, step = run_step(step_at(i, DT, DS), steps), tile = (wave >> 2) * DT + tile_at(i, DT, DS);
    if constexpr (!kTiled) {
      const auto [f0, nf] = down_columns();
      gbytes from = layer.w_down + (static_cast<int64_t>(f0) * FF + share_of() * share_length()) * 2;
      to = load_global<u32x4>(from + (step >= 0 ? step : 0) * 64 + row_at(tile * 16 + c16, nf, FF));
      return;
    }
    const auto [t0, nt] = down_tiles();
    to = load_global<u32x4>(layer.w_down + static_cast<uint32_t>((t0 + (tile < nt ? tile : nt - 1)) * (FF / 32) + share_of() * steps + (step >= 0 ? step : 0)) * 1024u + lane * 16);
  };

  // the rows from the area's places from `from` on into LDS, their sums of squares beside them; two rows a wave, asked for together
  auto take_rows = [&](int from, float* squares) __attribute__((always_inline)) {
    constexpr int kIn = (kResMaxWidth / 2 + NB) / 2 / 64 + ((kResMaxWidth / 2 + NB) / 2 % 64 != 0);
    if (wave >= M) return;
    const int m1 = wave + 8 < M ? wave + 8 : wave, n = H / 4, all = n + NB / 2;
    u32x4 v[2 * kIn];
    w.pairs<true>(v, [&](int i) { return from + (i < kIn ? wave : m1) * kRowPlaces + 2 * (i % kIn * 64 + lane < all ? i % kIn * 64 + lane : 0); });
    float ss[2] = {0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 2 * kIn; ++i) {
      const int at = i % kIn * 64 + lane, m = i < kIn ? wave : m1;
      *reinterpret_cast<uint2*>(xs + m * kLdx + (at < n ? 4 * at : kResMaxWidth)) = make_uint2(v[i][0], v[i][2]);
      ss[i / kIn] += at >= n && at < all ? __uint_as_float(v[i][0]) + __uint_as_float(v[i][2]) : 0.f;
    }
    ss[0] = wave_sum(ss[0]);
    ss[1] = wave_sum(ss[1]);
    if (lane == 0) {
      squares[wave] = ss[0];
      squares[m1] = m1 == wave ? ss[0] : ss[1];
    }
  };
  // the same in front of the first layer, from the stream itself
  auto take_stream = [&](ALOFA_GLOBAL const float* weight, float* squares) __attribute__((always_inline)) {
    for (int m = wave; m < M; m += 8) {
      const float* from = a.hidden + static_cast<int64_t>(rows_of[m]) * H;
      float ss = 0.f;
      for (int i = lane; i < H / 2; i += 64) {
        const float2 x = *reinterpret_cast<const float2*>(from + 2 * i);
        ss += x.x * x.x + x.y * x.y;
        *reinterpret_cast<uint32_t*>(xs + m * kLdx + 2 * i) = pack_bf16x2(x.x * weight[2 * i], x.y * weight[2 * i + 1]);
      }
      ss = wave_sum(ss);
      if (lane == 0) squares[m] = ss;
    }
  };
  auto factor = [&](float squares, float eps) __attribute__((always_inline)) { return __builtin_amdgcn_rsqf(squares / static_cast<float>(H) + eps); };
  // `n` pairs of places of every row, four numbers of 16 bits each (rows `stride` places apart)
  auto take_packed = [&](auto most, int from, int stride, int n) __attribute__((always_inline)) {
    constexpr int N = decltype(most)::value;
    if (wave >= M) return;
    const int m1 = wave + 8 < M ? wave + 8 : wave;
    u32x4 v[2 * N];
    w.pairs<true>(v, [&](int i) { return from + (i < N ? wave : m1) * stride + 2 * (i % N * 64 + lane < n ? i % N * 64 + lane : 0); });
#pragma unroll
    for (int i = 0; i < 2 * N; ++i) {
      const int at = i % N * 64 + lane;
      *reinterpret_cast<uint2*>(xs + (i < N ? wave : m1) * kLdx + (at < n ? 4 * at : kResMaxWidth)) = make_uint2(v[i][0], v[i][2]);
    }
  };

  // --- B's share of keys: tiles of sixteen keys, two a step, the waves in turn
  const int ahk = s % kv_heads, slot = s / kv_heads;      // the block's key head, and its place among the head's blocks
  int am = -1, apart = 0;
  for (int i = 0; i < M; ++i)
    if (slot >= first_of[i] && slot < first_of[i] + parts_of[i]) am = i, apart = slot - first_of[i];
  am = __builtin_amdgcn_readfirstlane(am);
  apart = __builtin_amdgcn_readfirstlane(apart);
  const bool attends = am >= 0 && slot < blocks_a_head;
  const int arow = __builtin_amdgcn_readfirstlane(attends ? rows_of[am] : 0), aparts = __builtin_amdgcn_readfirstlane(attends ? parts_of[am] : 1);
  const int pos = __builtin_amdgcn_readfirstlane(attends ? a.positions[arow] : 0), last = pos >> 4, bs_mask = (1 << a.bs_shift) - 1;
  const int per_part = (last + aparts) / aparts;
  const int tile_begin = apart * per_part, tile_end = tile_begin + per_part < last + 1 ? tile_begin + per_part : last + 1;
  const bool writes = attends && tile_begin <= last && last < tile_end;
  const int32_t* pages = a.table + static_cast<int64_t>(arow) * a.max_blocks;
  auto page_of = [&](int tile) __attribute__((always_inline)) { return __builtin_amdgcn_readfirstlane(pages[(tile < last ? tile : last) << 4 >> a.bs_shift]); };
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
    new_slot = a.slots[arow];
    new_slot = static_cast<int64_t>(static_cast<u64>(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(new_slot >> 32)))) << 32 |
                                    static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(new_slot))));
  }
  // A step's operands. Row i of the first product kt is key 16 (i / 8) + 8 (i / 4 % 2) + 4 kt + i % 4 of the step's 32: of the scores a lane then has eight consecutive keys, whose values
  // are one load of sixteen bytes (loads of eight are twice as many, in pieces of 32 bytes, and it is pieces that a compute unit's loads are bound by).
  struct Step {
    u32x4 k[2][2], v[4];
  };
  auto fetch_step = [&](Step& to, const ResidentLayer& layer, int tile, int pg0, int pg1) __attribute__((always_inline)) {
    const int64_t at0 = ((static_cast<int64_t>(pg0) * kv_heads + ahk) * d << a.bs_shift) * 2, at1 = ((static_cast<int64_t>(pg1) * kv_heads + ahk) * d << a.bs_shift) * 2;
    gbytes kb = reinterpret_cast<gbytes>(layer.k_cache) + (c16 < 8 ? at0 : at1), vb = reinterpret_cast<gbytes>(layer.v_cache) + (g < 2 ? at0 : at1);
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      int key = ((tile + (c16 >> 3)) << 4) + 8 * (c16 >> 2 & 1) + 4 * kt + (c16 & 3);
      key = key > pos ? pos : key;
#pragma unroll
      for (int ds = 0; ds < 2; ++ds) to.k[kt][ds] = load_global<u32x4>(kb + static_cast<uint32_t>((key & bs_mask) * d + ds * 32 + g * 8) * 2u);
    }
    int key8 = ((tile + (g >> 1)) << 4) + 8 * (g & 1);
    key8 = key8 > (pos & ~7) ? (pos & ~7) : key8;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) to.v[nt] = load_global<u32x4>(vb + static_cast<uint32_t>(((nt * 16 + c16) << a.bs_shift) + (key8 & bs_mask)) * 2u);
  };

  // the block's columns of the stream
  if (tid < 256) {
    const auto [p0, np] = own_pairs();
    const int m = tid >> 4, n = tid & 15;
    hs[tid] = n < 2 * np && m < M ? a.hidden[static_cast<int64_t>(rows_of[m]) * H + 2 * p0 + n] : 0.f;
  }
  ResidentLayer layer;
  auto next_layer = [&](int l) __attribute__((always_inline)) {
    uint32_t words[kLayerWords];
#pragma unroll
    for (int i = 0; i < kLayerWords; ++i) words[i] = __builtin_amdgcn_readfirstlane(table[l * kLayerWords + i]);
    layer = __builtin_bit_cast(ResidentLayer, *reinterpret_cast<const LayerWords*>(words));
  };
  next_layer(0);
  fetch_qkv(layer);
  __syncthreads();

#pragma unroll 1
  for (int l = 0; l < a.n_layers; ++l) {
    w.stamp = base + l + 1;
    // ---- A
    anew();
    float bias = 0.f;      // of the column of queries, keys and values that this thread finishes
    {
      const auto [q0, nq] = qkv_columns();
      if (a.has_bias) bias = layer.b_qkv[q0 + ((tid & 31) < nq ? (tid & 31) : 0)];
    }
    if (l == 0) take_stream(layer.norm0, ssq[0]);
    else take_rows(kAtRowsB, ssq[0]);
    Step st0 = {};
    if (has_step) fetch_step(st0, layer, first_tile, page0, page1);
    __syncthreads();
    {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < QS; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wq[j]), operand(step_of(wave % QK, QK, j), H / 32), acc, 0, 0, 0);
      leave_sums(QT > 1 ? wave / QK : 0, QK, wave % QK, acc);
    }
    __syncthreads();
    {
      const auto [q0, nq] = qkv_columns();
      const int n = tid & 31, m = tid >> 5;
      if (n < nq && m < M) put(area + kAtQkv + m * NQ + q0 + n, sum_of(n >> 4, std::integral_constant<int, QK>{}, m, n & 15) * factor(ssq[0][m], a.eps0) + bias, w.stamp);
    }

    // ---- B
    anew();
    if (attends) {
      Step st1 = {};
      int next0 = 0, next1 = 0;      // pages of the step behind the one asked for last
      if (has_step) {
        fetch_step(st1, layer, first_tile + 2 * kResWaves, page_of(first_tile + 2 * kResWaves), page_of(first_tile + 2 * kResWaves + 1));
        next0 = page_of(first_tile + 4 * kResWaves);
        next1 = page_of(first_tile + 4 * kResWaves + 1);
      }
      const int item = tid / 16, chan = 2 * (tid % 16);      // head `item` (group: the key, group + 1: the value), channels chan, chan + 1 and their partners 32 on
      if (wave * 4 < group + 2) {      // (all lanes of a wave ask, those without a head of their own for the first one: a wait is a wave's)
        const int row = item < group || item > group + 1 ? ahk * group + (item < group ? item : 0) : item == group ? heads + ahk : heads + kv_heads + ahk;
        const int at = kAtQkv + am * NQ + row * d + chan;
        u32x4 v[2];
        w.pairs<true>(v, [&](int i) { return at + 32 * i; });
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
      auto take_step = [&](Step& in, int tile) __attribute__((always_inline)) {
        const bool last_here = tile + 1 >= last;
        f32x4 sc[2];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
          sc[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
          const bool new_row = last_here && ((tile + (c16 >> 3)) << 4) + 8 * (c16 >> 2 & 1) + 4 * kt + (c16 & 3) == pos;
#pragma unroll
          for (int ds = 0; ds < 2; ++ds) {
            u32x4 kf = in.k[kt][ds];
            if (last_here) {      // (the new token's key is not in the cache yet)
              const u32x4 new_k = *reinterpret_cast<const u32x4*>(qs + kResMaxGroup * 72 + ds * 32 + g * 8);
              kf.x = new_row ? new_k.x : kf.x;
              kf.y = new_row ? new_k.y : kf.y;
              kf.z = new_row ? new_k.z : kf.z;
              kf.w = new_row ? new_k.w : kf.w;
            }
            sc[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kf), qf[ds], sc[kt], 0, 0, 0);
          }
        }
        const int first_key = ((tile + (g >> 1)) << 4) + 8 * (g & 1);
        const bool mine = tile + (g >> 1) < tile_end;
        float pw[8], step_max = -FLT_MAX;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          pw[i] = first_key + i <= pos && mine ? sc[i / 4][i % 4] * scale2 : -FLT_MAX;
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
          uint32_t vw[4] = {in.v[nt].x, in.v[nt].y, in.v[nt].z, in.v[nt].w};
          if (last_here) {      // what lies beyond the new token is cleared, the new token's value takes its place
            const uint32_t new_v = qs[(kResMaxGroup + 1) * 72 + nt * 16 + c16];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int key = first_key + 2 * i;
              vw[i] &= (key <= pos ? 0x0000ffffu : 0u) | (key + 1 <= pos ? 0xffff0000u : 0u);
              const uint32_t ins = (pos & 1) ? ((vw[i] & 0x0000ffffu) | (new_v << 16)) : ((vw[i] & 0xffff0000u) | new_v);
              vw[i] = key == (pos & ~1) ? ins : vw[i];
            }
          }
          o[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, make_uint4(vw[0], vw[1], vw[2], vw[3])), pf, o[nt], 0, 0, 0);
        }
      };
      // (two steps on their way; a step beyond the last key brings that key's page once more and is not taken)
#pragma unroll 1
      for (int tile = first_tile; tile < tile_end; tile += 4 * kResWaves) {
        anew();
        take_step(st0, tile);
        fetch_step(st0, layer, tile + 4 * kResWaves, next0, next1);
        next0 = page_of(tile + 6 * kResWaves);
        next1 = page_of(tile + 6 * kResWaves + 1);
        if (tile + 2 * kResWaves >= tile_end) break;
        take_step(st1, tile + 2 * kResWaves);
        fetch_step(st1, layer, tile + 6 * kResWaves, next0, next1);
        next0 = page_of(tile + 8 * kResWaves);
        next1 = page_of(tile + 8 * kResWaves + 1);
      }
      sum = rows_sum(sum);
      float* mine = red + (wave * kResMaxGroup + c16) * (d + 4);
      if (g == 0 && c16 < kResMaxGroup) {
        mine[0] = mx;
        mine[1] = sum;
      }
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
        if (c16 < kResMaxGroup) *reinterpret_cast<f32x4*>(mine + 4 + nt * 16 + 4 * g) = o[nt];
      fetch_out(layer);
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
        u64* to = area + kAtParts + static_cast<int64_t>(s * kResMaxGroup + i) * 66;
        put(to + 2 + c, acc, w.stamp);
        if (c < 2) put(to + c, c == 0 ? big : total, w.stamp);
      }
    } else {
      fetch_out(layer);
    }

    // ---- C: (row, head) per wave, the parts in turn
    anew();
    {
      const int item = wave * NB + s;
      if (item < M * heads) {
        const int m = item / heads, ch = item % heads, n_parts = __builtin_amdgcn_readfirstlane(parts_of[m]), f0 = __builtin_amdgcn_readfirstlane(first_of[m]);
        const int hk = ch / group, i = ch % group;
        float big = -FLT_MAX, total = 0.f, acc = 0.f;
        for (int p0 = 0; p0 < n_parts; p0 += 4) {
          u32x4 v[8];
          w.pairs<true>(v, [&](int n) {
            const int part = p0 + n / 2 < n_parts ? p0 + n / 2 : p0;
            return kAtParts + (((f0 + part) * kv_heads + hk) * kResMaxGroup + i) * 66 + (n % 2 == 0 ? 0 : 2 + (lane & ~1));
          });
          float ms[4], most = big;
#pragma unroll
          for (int n = 0; n < 4; ++n) {
            ms[n] = p0 + n < n_parts ? __uint_as_float(v[2 * n][0]) : -FLT_MAX;
            most = fmaxf(most, ms[n]);
          }
          const float before = __builtin_amdgcn_exp2f(big - most);
          total *= before;
          acc *= before;
#pragma unroll
          for (int n = 0; n < 4; ++n) {
            const float e = p0 + n < n_parts ? __builtin_amdgcn_exp2f(ms[n] - most) : 0.f;
            total += __uint_as_float(v[2 * n][2]) * e;
            acc += __uint_as_float((lane & 1) ? v[2 * n + 1][2] : v[2 * n + 1][0]) * e;
          }
          big = most;
        }
        const float x = acc / total, y = lane_xor1(x);
        if ((lane & 1) == 0) put(area + kAtAttn + m * (KO / 2) + ch * 32 + lane / 2, pack_bf16x2(x, y), w.stamp);
      }
    }

    // ---- D
    anew();
#pragma unroll
    for (int i = 0; i < kFirst && i < GS * GT; ++i) fetch_gate_up(wg[i], layer, i);
    float weight1;      // of the second norm, for the column that this thread finishes
    {
      const auto [p0, np] = own_pairs();
      weight1 = layer.norm1[2 * p0 + ((tid & 15) < 2 * np ? (tid & 15) : 0)];
    }
    take_packed(std::integral_constant<int, kResMaxWidth / 4 / 64>{}, kAtAttn, KO / 2, KO / 4);
    __syncthreads();
    {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wo[j]), operand(step_of(wave, 8, j), KO / 32), acc, 0, 0, 0);
      leave_sums(0, 8, wave, acc);
    }
    __syncthreads();
    if (wave < 4) {
      const auto [p0, np] = own_pairs();
      const int n = tid & 15, m = tid >> 4;
      const bool ok = n < 2 * np && m < M;
      const float v = hs[tid] + sum_of(0, Eight{}, m, n);
      hs[tid] = v;
      const float x = v * weight1, y = lane_xor1(x);
      float ss = ok ? v * v : 0.f;
      ss += lane_xor1(ss);
      ss += lane_xor2(ss);
      ss += lane_ror4(ss);
      ss += lane_xor8(ss);
      u64* row = area + kAtRowsA + m * kRowPlaces;
      if (ok && (n & 1) == 0) put(row + p0 + n / 2, pack_bf16x2(x, y), w.stamp);
      if (n == 0 && m < M) put(row + H / 2 + s, ss, w.stamp);
    }

    // ---- E
    anew();
#pragma unroll
    for (int i = kFirst; i < kBefore && i < GS * GT; ++i) fetch_gate_up(wg[i], layer, i);
    take_rows(kAtRowsA, ssq[1]);
#pragma unroll
    for (int i = kBefore; i < kRing && i < GS * GT; ++i) fetch_gate_up(wg[i], layer, i);
    __syncthreads();
    {
      f32x4 acc[GT];
#pragma unroll
      for (int t = 0; t < GT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < GS; j += 2) {
        const bf16x8 x[2] = {operand(run_step(j, H / 32), H / 32), operand(j + 1 < GS ? run_step(j + 1, H / 32) : -1, H / 32)};
#pragma unroll
        for (int i = j * GT; i < (j + 2 < GS ? j + 2 : GS) * GT; ++i) {
          acc[tile_at(i, GT, GS)] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wg[i % kRing]), x[step_at(i, GT, GS) - j], acc[tile_at(i, GT, GS)], 0, 0, 0);
          if (i + kRing < GS * GT) fetch_gate_up(wg[i % kRing], layer, i + kRing);
        }
      }
#pragma unroll
      for (int t = 0; t < GT; ++t) leave_sums((wave >> 2) * GT + t, 4, wave & 3, acc[t]);
    }
    __syncthreads();
    {
      const auto [p0, np] = act_pairs();
      const int m = tid >> 5;
      const float f = factor(ssq[1][m < M ? m : 0], a.eps1);
#pragma unroll
      for (int i = 0; i < (GT + 1) / 2; ++i) {
        const int n = (tid & 31) + 32 * i;      // column 2 p0 + n of act
        const bool ok = n < 2 * np && m < M;
        const int at = n < 16 * GT ? n : 0;
        const float gate = sum_of(at >> 4, Four{}, m, at & 15) * f, up = sum_of(GT + (at >> 4), Four{}, m, at & 15) * f;
        const float x = gate_of<false>(gate) * up, y = lane_xor1(x);
        if (ok && (n & 1) == 0) put(area + kAtAct + m * (FF / 2) + p0 + n / 2, pack_bf16x2(x, y), w.stamp);
      }
    }

    // ---- F
    anew();
    constexpr int kDown = DS * DT, kDownRing = kDown < kRing ? kDown : kRing;
#pragma unroll
    for (int i = 0; i < kDownRing; ++i) fetch_down(wd[i], layer, i);
    take_packed(std::integral_constant<int, kResMaxFF / kResShares / 4 / 64>{}, kAtAct + share_of() * (share_length() / 2), FF / 2, share_length() / 4);
    __syncthreads();
    {
      f32x4 acc[DT];
#pragma unroll
      for (int t = 0; t < DT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < DS; j += 2) {
        const int steps = share_length() / 32;
        const bf16x8 x[2] = {operand(run_step(j, steps), steps), operand(j + 1 < DS ? run_step(j + 1, steps) : -1, steps)};
#pragma unroll
        for (int i = j * DT; i < (j + 2 < DS ? j + 2 : DS) * DT; ++i) {
          acc[tile_at(i, DT, DS)] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wd[i % kDownRing]), x[step_at(i, DT, DS) - j], acc[tile_at(i, DT, DS)], 0, 0, 0);
          if (i + kDownRing < kDown) fetch_down(wd[i % kDownRing], layer, i + kDownRing);
        }
      }
#pragma unroll
      for (int t = 0; t < DT; ++t) leave_sums((wave >> 2) * DT + t, 4, wave & 3, acc[t]);
    }
    __syncthreads();
    {
      const auto [f0, nf] = down_columns();
      const int m = tid >> 5;
#pragma unroll
      for (int i = 0; i < DT; ++i) {
        const int n = (tid & 31) + 32 * i;
        if (n < nf && m < M) put(area + kAtDown + (share_of() * MB + m) * kColumnPlaces + f0 + n, sum_of(n >> 4, Four{}, m, n & 15), w.stamp);
      }
    }

    // ---- G
    anew();
    const bool more = l + 1 < a.n_layers;
    next_layer(more ? l + 1 : l);      // (behind the last layer its own once more: a load under a condition would keep the old registers)
    fetch_qkv(layer);
    {
      const auto [p0, np] = own_pairs();
      const int pair = lane & 7, share = lane >> 3, mine = pair < np ? pair : 0;      // two columns and a share a lane, two rows a wave
      const float weight0 = layer.norm0[2 * (p0 + mine)], weight1 = layer.norm0[2 * (p0 + mine) + 1];
      u32x4 v[2] = {u32x4{0u, 0u, 0u, 0u}, u32x4{0u, 0u, 0u, 0u}};
      if (wave < M) w.pairs<true>(v, [&](int i) { return kAtDown + (share * MB + (wave + 8 * i < M ? wave + 8 * i : wave)) * kColumnPlaces + 2 * (p0 + mine); });
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int m = wave + 8 * i;
        float x = __uint_as_float(v[i][0]), y = __uint_as_float(v[i][2]);
        x += lane_xor8(x);
        y += lane_xor8(y);
        x = rows_sum(x);
        y = rows_sum(y);
        float2* to = reinterpret_cast<float2*>(hs + m * 16) + mine;
        x += to->x;
        y += to->y;
        float ss = pair < np ? x * x + y * y : 0.f;
        ss += lane_xor1(ss);
        ss += lane_xor2(ss);
        ss += lane_mirror8(ss);
        if (m < M && lane < np) {
          *to = make_float2(x, y);
          if (more) put(area + kAtRowsB + m * kRowPlaces + p0 + lane, pack_bf16x2(x * weight0, y * weight1), w.stamp + 1);
          else *reinterpret_cast<float2*>(a.hidden + static_cast<int64_t>(rows_of[m]) * H + 2 * (p0 + lane)) = make_float2(x, y);
        }
        if (more && m < M && lane == 0) put(area + kAtRowsB + m * kRowPlaces + H / 2 + s, ss, w.stamp + 1);
      }
    }
  }
  // the group's next step's stamps go on from here (every block of the group has read `base` before this one could finish its last layer)
  if (s == 0 && tid == 0) __hip_atomic_store(area, static_cast<u64>(base + a.n_layers), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int G, bool kTiled>
static void launch_steps(const ResidentArgs& a, hipStream_t stream) {      // (by the steps of a wave's run of a row: 512, 896 and 1,024 columns)
  if (a.H <= 512) decode_groups_kernel<G, 4, kTiled><<<kResBlocks, kResThreads, 0, stream>>>(a);
  else if (a.H <= 896) decode_groups_kernel<G, 7, kTiled><<<kResBlocks, kResThreads, 0, stream>>>(a);
  else decode_groups_kernel<G, 8, kTiled><<<kResBlocks, kResThreads, 0, stream>>>(a);
}

int launch_groups(const ResidentArgs& a, bool tiled, hipStream_t stream) {
  if (a.M <= 32) tiled ? launch_steps<2, true>(a, stream) : launch_steps<2, false>(a, stream);
  else tiled ? launch_steps<4, true>(a, stream) : launch_steps<4, false>(a, stream);
  return check_launch("decode_groups");
}

}  // namespace alofa

// The most rows of a step of a model that alofa_resident_takes: sixteen, or as many as the groups hold of it, with the matrices as they are and in tiles alike.
extern "C" int alofa_resident_rows(int H, int FF, int heads, int kv_heads) {
  using namespace alofa;
  auto fits = [&](int groups) {
    const int blocks = kResBlocks / groups, gate_tiles = groups == 4 ? 5 : 3, down_tiles = groups == 4 ? 4 : 2, qkv_tiles = groups == 4 ? 2 : 1;
    auto most = [&](int n) { return (n + blocks - 1) / blocks; };
    return H / 2 >= blocks && 2 * most(H / 2) <= 16 && (heads + 2 * kv_heads) * 64 <= kQkvMost && most((heads + 2 * kv_heads) * 64) <= 16 * qkv_tiles && FF % 16 == 0 && 2 * most(FF / 2) <= 16 * gate_tiles &&
           most(FF / 16) <= gate_tiles && FF / kResShares <= 20 * 32 && H % 16 == 0 && H * kResShares / blocks <= 32 * down_tiles && (H / 16 * kResShares + blocks - 1) / blocks <= 2 * down_tiles &&
           kv_heads * kResMaxRows <= blocks && kResMaxRows * heads <= kResWaves * blocks;
  };
  return !fits(2) ? kResMaxRows : !fits(4) ? 2 * kResMaxRows : 4 * kResMaxRows;
}
