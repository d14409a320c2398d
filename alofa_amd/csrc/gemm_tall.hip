// The tiled product for many rows: tiles of up to 256 x 320 outputs by eight waves in two groups that take turns at the matrix
// cores. out[m, n] = sum_k A[m, k] * W[n, k], bfloat16, float sums: one accumulator an output, products in ascending k (the same
// bits as the forms of gemm_mfma.hip without shares of K).
//
// What bounds such a product is the way from the L2s into LDS and the order of things in a compute unit. Measured here with the
// products left out: a compute unit brings 47 bytes a nanosecond with 64 KB on their way and 68 with 96 KB (a fetch takes 1.4 us whatever
// is asked), and only where a fetch asks for whole lines of 128 bytes: with slabs of 32 along K (64 bytes a row) it stays at 45
// whatever is on its way. Without the fetches the products reach 1.53 PFLOP/s, with neither fetches nor reads from LDS 1.64 (the
// clock drops to 1.9 GHz under them). Hence:
//
//   * Slabs of 64 along K, straight from memory into a ring of S slabs in LDS (global_load_lds_dwordx4). A slab comes in P units: A's rows
//     with the first of a wave's groups of 32 columns, then the other column groups. A step through a slab has P phases, one a unit, so that a
//     unit's place is free again, and its successor S slabs on sets out, as soon as its phase is over: all of the ring but one unit is on its way or in use.
//   * Waves 0..3 and waves 4..7 (one of each on every SIMD) run half a phase apart: while one group reads its fragments of a phase from LDS,
//     the other multiplies; a barrier ends every such slot. The fetches are issued between the products, where the wave has nothing else to issue.
//
// 4,096 x 27,648 x 5,120 with the gate 2,132 us (tiles of 256 x 256, eight waves, slabs of 32, all waves in step) -> 2,029 (the groups half a
// phase apart) -> 1,880 (slabs of 64 in two units) -> 1,765 (fetches between the products): 1.31 PFLOP/s.
//
// A tile's way out counts as much as its way in where K is short. bfloat16 outputs are written as whole lines of rows by way of LDS (rows_epilogue), the gate's division takes what its range needs
// (common.h), and gate and up share a group of 32 rows of W eight and eight, so that any tile does for them: 4,864 x 896 with the gate against 2,048 rows 47.6 us (tiles of 128 x 64 of gemm_mfma.hip; 53.1
// with 256 x 128 here) -> 40.3 (256 x 160, one round of the chip) -> 37.2 (the division; with the general one's bits for every gate 0.4 to 0.7 % more); 8,960 x 1,536 against 2,048 133 -> 102, 18,944 x 3,584 against 1,970 460 -> 441, 27,648 x 5,120
// against 4,096 1,797 -> 1,756; stored as bfloat16 7,168 x 5,120 against 4,096 266 -> 243, 4,608 x 3,584 against 1,970 72.0 -> 65.7.
//
// Tiles (Tall<rows, columns, waves along rows, along columns, slabs in the ring, column groups of the phases>): the wider, the less a
// product fetches; which one comes out best is a matter of how full its last round of the chip is: see pick_tall.
//
// Which slots may touch which place: group 0 reads phase x (phases counted through all slabs) in slot 2 x and multiplies in slot 2 x + 1,
// group 1 one slot later. Unit x is read in slots 2 x and 2 x + 1; its successor, unit x + S P, is fetched among the products of phase x + 1,
// in slot 2 x + 3 or 2 x + 4. A wave waits for its own fetches of unit x + 1 before the barrier that ends slot 2 x + 1, behind which group 0 reads it.
// `allowed` counts the fetches issued behind that unit, which stay on their way.
#include "gemm_tiles.h"

#include <cstdlib>
#include <type_traits>

namespace alofa {

template <int kTM, int kTN, int kWM, int kWN, int kS, int J0, int J1, int J2 = 0>
struct Tall {
  static constexpr int TM = kTM, TN = kTN, WM = kWM, WN = kWN, S = kS, P = J2 > 0 ? 3 : 2;
  static constexpr int TI = TM / 32 / WM, TJ = TN / 32 / WN, kStage = (TM + TN) * 128;                // 32 x 32 tiles a wave; bytes a slab
  static constexpr int J(int p) { return p == 0 ? J0 : p == 1 ? J1 : J2; }
  static constexpr int before(int p) { return p == 0 ? 0 : p == 1 ? J0 : J0 + J1; }                   // column groups of a wave in earlier phases
  static constexpr int first_row(int p) { return p == 0 ? 0 : TM + WN * 32 * before(p); }             // a unit's rows within the slab in LDS
  static constexpr int rows(int p) { return WN * J(p) * 32 + (p == 0 ? TM : 0); }
  static constexpr int loads(int p) { return (rows(p) + 63) / 64; }                                   // fetch instructions (eight rows each) a wave
  static constexpr int most_loads() { int m = 0; for (int p = 0; p < P; ++p) m = loads(p) > m ? loads(p) : m; return m; }
  static constexpr int most_j() { int m = 0; for (int p = 0; p < P; ++p) m = J(p) > m ? J(p) : m; return m; }
  // fetches of a wave behind those of the next phase's unit; R: slabs after this one (S for S and more); late: group 1, which waits before its products
  static constexpr int allowed(int p, int R, bool late) {
    int n = 0;
    for (int o = p + 2; o <= p + S * P - 1 - late && o < (R + 1) * P; ++o) n += loads(o % P);
    return n;
  }
  static_assert(WM * WN == 8 && TM % (32 * WM) == 0 && TN % (32 * WN) == 0 && J0 + J1 + J2 == TJ && S * kStage <= 160 * 1024, "eight waves share the tile, the phases its columns");
};

// bfloat16 outputs leave by way of LDS, 32 rows of a wave at a time: the products are taken with W's rows first, so that a lane holds four
// consecutive columns of one row (element e of a group: row lane % 32, column 8 (e / 4) + 4 (lane / 32) + e % 4); it writes them as eight bytes, and
// the wave reads whole rows back, sixteen bytes a lane.
template <int kEpilogue, int TJ>
constexpr int kRowsStride = TJ * (is_gated(kEpilogue) ? 32 : 64) + 16;      // bytes of a wave's row in LDS
template <int kEpilogue, int TJ>
constexpr int kRowsBytes = 32 * kRowsStride<kEpilogue, TJ>;
template <int kEpilogue, int TI, int TJ>
__device__ __forceinline__ void rows_epilogue(f32x16 (&acc)[TI][TJ], char* mine, bf16_t* __restrict__ out, int64_t ldo, const float* __restrict__ bias, int M, int N, int m0,
                                              int n0, int lane) {
  constexpr bool kGated = is_gated(kEpilogue);
  constexpr int kStride = kRowsStride<kEpilogue, TJ>, kChunks = TJ * (kGated ? 2 : 4);      // sixteen-byte chunks a row
  const bool whole = ldo % 8 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
  char* to = mine + (lane % 32) * kStride + (lane / 32) * 8;
#pragma unroll
  for (int i = 0; i < TI; ++i) {
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
#pragma unroll
      for (int e = 0; e < 16; e += kGated ? 8 : 4) {
        float v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          if constexpr (kGated) {
            v[c] = gate_of<kEpilogue == kMfGeglu>(acc[i][j][e + c]) * acc[i][j][e + 4 + c];
          } else {
            v[c] = acc[i][j][e + c];
            if (bias) v[c] += bias[min(n0 + j * 32 + e * 2 + (lane / 32) * 4 + c, N - 1)];
          }
        }
        *reinterpret_cast<uint2*>(to + j * (kGated ? 32 : 64) + e * (kGated ? 2 : 4)) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
      }
    }
    wave_lds_sync();
#pragma unroll
    for (int x = 0; x < kChunks / 2; ++x) {
      const int at = x * 64 + lane, r = at / kChunks, c = at % kChunks, m = m0 + i * 32 + r, n = n0 + c * 8;
      const uint4 v = *reinterpret_cast<const uint4*>(mine + r * kStride + c * 16);
      bf16_t* dst = out + static_cast<int64_t>(m) * ldo + n;
      if (m < M) {
        if (whole && n + 8 <= N) {
          *reinterpret_cast<uint4*>(dst) = v;
        } else {
          const uint32_t word[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
          for (int u = 0; u < 8; ++u)
            if (n + u < N) dst[u] = static_cast<bf16_t>(word[u / 2] >> (16 * (u % 2)));
        }
      }
    }
    wave_lds_sync();
  }
}

template <int kEpilogue, typename TO, typename T>
__global__ void __launch_bounds__(512) gemm_tall_kernel(TO* __restrict__ out, int64_t ldo, const bf16_t* __restrict__ A, int64_t lda, const bf16_t* __restrict__ W,
                                                        const bf16_t* __restrict__ W2, int64_t ldw, const float* __restrict__ bias, int M, int N, int K, int tiles_m,
                                                        int tiles_n) {
  constexpr int TM = T::TM, TN = T::TN, WN = T::WN, TI = T::TI, TJ = T::TJ, S = T::S, P = T::P;
  constexpr bool kGated = is_gated(kEpilogue), kRows = sizeof(TO) == 2;      // kRows: a lane holds four consecutive columns of one row (bfloat16 outputs, see rows_epilogue)
  static_assert(!kGated || kRows, "gated outputs are bfloat16");
  __shared__ __attribute__((aligned(1024))) char ring[S * T::kStage];
  const TilePlace place = place_tile(blockIdx.x, tiles_m, tiles_n, 1, true);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  const int wm = wave / WN, wn = wave % WN;
  const int m0 = place.bm * TM, n0 = place.bn * (is_gated(kEpilogue) ? TN / 2 : TN);

  // what this lane fetches: instruction i of a unit brings rows 8 (8 i + wave) .. + 7 of the unit, lane l place l % 8 of row l / 8. (A wave whose
  // rows lie past the unit's end brings its first ones again, to the same place: every wave counts the same number of fetches.)
  // Rows beyond M or N come from the last valid row; their results are never stored.
  const int chunk = (lane % 8) ^ swz(8 * wave + lane / 8);      // (units begin at multiples of 32 rows: the same for all of them)
  const bf16_t* src[P][T::most_loads()];
  unsigned to[P][T::most_loads()];
#pragma unroll
  for (int p = 0; p < P; ++p)
#pragma unroll
    for (int i = 0; i < T::loads(p); ++i) {
      const int at = 8 * (8 * i + wave) < T::rows(p) ? 8 * (8 * i + wave) : 8 * wave, r = at + lane / 8;
      const bf16_t* row;
      if (p == 0 && r < TM) {
        row = A + static_cast<int64_t>(min(m0 + r, M - 1)) * lda;
      } else {
        const int x = p == 0 ? r - TM : r, wcol = x / (T::J(p) * 32), j = T::before(p) + x / 32 % T::J(p);
        // (gated: a group of 32 is gate, up, gate, up of eight columns each, so that both halves of an output meet in one lane)
        const int n = n0 + (kGated ? (wcol * TJ + j) * 16 + x % 32 / 16 * 8 + x % 8 : (wcol * TJ + j) * 32 + x % 32);
        row = (kGated && (x & 8) ? W2 : W) + static_cast<int64_t>(min(n, N - 1)) * ldw;
      }
      src[p][i] = row + chunk * 8;
      to[p][i] = static_cast<unsigned>(reinterpret_cast<uintptr_t>(ring)) + (T::first_row(p) + at) * 128;
    }
  // K a multiple of 32: the last slab may be half a slab; the lanes of its other half bring the first half again (it is not multiplied)
  const int slabs = (K + 63) / 64, half_slab = K % 64 ? slabs - 1 : -1, back = chunk >= 4 ? 32 : 0;
  // (written out as an instruction: the compiler, which cannot tell the ring's slabs apart, would wait for every fetch before any read from LDS)
  auto bring = [&](int p, int i, int slab, unsigned stage) __attribute__((always_inline)) {
    const bf16_t* from = src[p][i] + (static_cast<int64_t>(slab) * 64 - (slab == half_slab ? back : 0));
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                 :: "s"(__builtin_amdgcn_readfirstlane(stage + to[p][i])), "v"(from), "r"(ring) : "memory", "m0");
  };
  auto wait = [&](auto n) __attribute__((always_inline)) { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(n.value) : "memory"); };
  auto end_slot = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  f32x16 acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  // fragments: lane l reads row l % 32 of its 32-row group, chunk 2 q + l / 32 in step q of the slab's four
  int place_of[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) place_of[q] = ((2 * q + lane / 32) ^ swz(lane % 32)) * 16 + (lane % 32) * 128;
  bf16x8 a[4][TI], w[4][T::most_j()];

  const bool late = wave >= 4;
#pragma unroll
  for (int x = 0; x < S * P - 1; ++x)      // every unit of the first S slabs but the last
    if (x / P < slabs) {
#pragma unroll
      for (int i = 0; i < T::loads(x % P); ++i) bring(x % P, i, x / P, (x / P) * T::kStage);
    }
  if (slabs >= S) wait(std::integral_constant<int, T::allowed(-1, S, false)>{});
  else wait(std::integral_constant<int, 0>{});
  end_slot();
  if (late) end_slot();
  unsigned stage = 0;
  auto slab_step = [&](int k, auto left) __attribute__((always_inline)) {
    constexpr int R = decltype(left)::value;      // slabs after this one (S: S or more)
    const char* st = ring + stage;
    const unsigned stage_before = stage == 0 ? (S - 1) * T::kStage : stage - T::kStage;      // where slab k - 1 lay and slab k - 1 + S will
    auto phase = [&](auto number) __attribute__((always_inline)) {
      constexpr int p = decltype(number)::value, n = T::J(p);
      if constexpr (p == 0) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int i = 0; i < TI; ++i) a[q][i] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(st + (wm * TI + i) * 32 * 128 + place_of[q]));
      }
      const char* ws = st + (p == 0 ? TM : T::first_row(p)) * 128 + wn * n * 32 * 128;
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int j = 0; j < n; ++j) w[q][j] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(ws + j * 32 * 128 + place_of[q]));
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (late) wait(std::integral_constant<int, T::allowed(p, R, true)>{});
      end_slot();
      // the products, and among them the fetches of the unit whose place the phase before has left
      constexpr int u = p == 0 ? P - 1 : p - 1, ahead = p == 0 ? S - 1 : S, total = 4 * TI * n, loads = T::loads(u);
      constexpr bool more = R >= ahead;
      int sent = 0, done = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (R == 0 && q == 2 && half_slab >= 0) break;      // (uniform: the last slab is half a slab)
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int j = 0; j < n; ++j) {
            acc[i][T::before(p) + j] = kRows ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[q][j], a[q][i], acc[i][T::before(p) + j], 0, 0, 0)
                                             : __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[q][i], w[q][j], acc[i][T::before(p) + j], 0, 0, 0);
            ++done;
            if (more && sent < loads && done * loads * 4 >= (sent + 1) * total * 3) {
              __builtin_amdgcn_sched_barrier(0);
              bring(u, sent, k + ahead, p == 0 ? stage_before : stage);
              __builtin_amdgcn_sched_barrier(0);
              ++sent;
            }
          }
      }
      if (!late) wait(std::integral_constant<int, T::allowed(p, R, false)>{});
      end_slot();
    };
    phase(std::integral_constant<int, 0>{});
    phase(std::integral_constant<int, 1>{});
    if constexpr (P == 3) phase(std::integral_constant<int, 2>{});
    stage = stage == (S - 1) * T::kStage ? 0 : stage + T::kStage;
  };
  int k = 0;
  for (; k + S < slabs; ++k) slab_step(k, std::integral_constant<int, S>{});
  if constexpr (S == 3)
    if (k + 2 < slabs) slab_step(k++, std::integral_constant<int, 2>{});
  if (k + 1 < slabs) slab_step(k++, std::integral_constant<int, 1>{});
  slab_step(k, std::integral_constant<int, 0>{});
  if (!late) end_slot();
  // (behind the last slot's barrier nobody reads the ring any more, and no fetch is on its way)
  if constexpr (kRows) rows_epilogue<kEpilogue, TI, TJ>(acc, ring + wave * kRowsBytes<kEpilogue, TJ>, out, ldo, bias, M, N, m0 + wm * TI * 32, n0 + wn * TJ * (kGated ? 16 : 32), lane);
  else tile_epilogue<kEpilogue, TO, TI, TJ>(acc, out, ldo, bias, M, N, m0, n0, wm, wn, lane);
}

// The forms, and what a tile of each takes: us a slab of 64 with few and with all compute units at work, and us besides (way in and epilogue).
// Measured at 512 to 4,096 rows against 3,584 to 13,824 values of K; with the gate (columns of outputs: half as many as rows of W) fitted to 330 launches of 65 to 4,240 rows against
// K of 768 to 5,120, which it foretells within 3 to 6 %: the form picked is 0.2 % behind the best one on average.
struct TallForm {
  int rows, columns;      // of outputs
  double slab_few, slab_all, besides;
};
constexpr TallForm kPlain[] = {{256, 320, 1.38, 1.95, 17}, {256, 256, 1.15, 1.50, 9}, {256, 192, 1.07, 1.20, 6}, {256, 160, 1.00, 1.13, 5}, {256, 128, 0.83, 0.92, 4}, {128, 192, 0.70, 0.78, 4}, {128, 128, 0.57, 0.60, 3}};
constexpr TallForm kGated[] = {{256, 160, 1.27, 1.91, 9.5}, {256, 128, 1.02, 1.53, 7.1}, {256, 96, 0.93, 1.26, 5.6}, {256, 80, 0.83, 1.14, 5.6}, {256, 64, 0.66, 0.90, 4.8}, {128, 128, 0.89, 0.99, 3.4}, {128, 96, 0.79, 0.84, 3.7}, {128, 64, 0.67, 0.65, 2.9}};

// The form with the least time by that count: whole rounds of the chip, then what is left over; `fill`: its tiles against the compute units.
static int pick_tall(int M, int N, int K, bool gated, double* fill) {
  const TallForm* forms = gated ? kGated : kPlain;
  const int n_forms = gated ? 8 : 7, cus = compute_units();
  const double slabs = (K + 63) / 64;
  int best = 0;
  double least = 1e30;
  for (int f = 0; f < n_forms; ++f) {
    const TallForm& form = forms[f];
    const int64_t tiles = static_cast<int64_t>((M + form.rows - 1) / form.rows) * ((N + form.columns - 1) / form.columns);
    const int64_t whole = tiles / cus, rest = tiles % cus;
    double us = whole * (slabs * form.slab_all + form.besides);
    if (rest) us += slabs * (form.slab_few + (form.slab_all - form.slab_few) * rest / cus) + form.besides;
    if (us < least) least = us, best = f, *fill = tiles >= cus ? 1.0 : static_cast<double>(tiles) / cus;
  }
  return best;
}

// Where the tiled product's other forms stay ahead: tiles that leave too much of the chip idle (their K can be shared out over blocks), all the more the
// shorter K is (a tile is over before the ring has paid for its way in). us, the other forms / these:
//   behind: 4,608 x 3,584 against 512 rows (144 tiles of 128 x 128) 38 / 39, 3,584 x 3,584 against 700 (168) 36 / 39, 3,584 x 18,944 against 512 (56 of 256 x 128) 105 / 237,
//   2,560 x 2,048 against 1,024 (160 of 128 x 128) 21 / 24, 2,048 x 1,536 against 1,536 (192) 18 / 21, 8,960 x 1,536 with the gate against 256 (70) 31 / 36;
//   ahead: 5,120 x 5,120 against 512 (160) 67 / 56, 5,120 x 13,824 against 512 170 / 130, 3,584 x 3,584 against 1,024 (224) 53 / 41, against 2,000 70 / 60, 5,120 x 27,648 against 4,096 1,299 / 891,
//   5,120 x 5,120 260 / 184, 4,608 x 3,584 against 2,000 100 / 72, 2,560 x 2,048 against 1,536 (240) 35 / 25; with the gate: 18,944 x 3,584 against 65 (148 of 128 x 128) 79 / 62, against 2,048
//   523 / 463, 27,648 x 5,120 against 2,048 1,090 / 920, 8,960 x 1,536 against 300 (210) 35 / 29, 13,824 x 5,120 against 2,048 573 / 493.
// Small matrices (under 20 M elements, 40 MB) whose K is not long stay with the other forms until their tiles fill seven and a half tenths: 180 tiles of 128 x 128, 1,280 x 2,048 against 2,262 rows
// 24.5 / 26.3, 2,304 x 4,864 against 1,191 47.0 / 49.6, 2,560 x 4,096 against 1,090 40.6 / 43.3; 154 and 162 tiles, 896 x 8,192 against 2,706 73.3 / 76.4, 2,304 x 8,192 against 1,053 73.1 / 76.5; 189 and 192,
// 896 x 2,560 against 3,432 44.3 / 31.2, 2,048 x 3,072 against 1,465 47.4 / 35.4.
// Where tiles of 128 x 128 are more than one round of the chip, the others' K is not shared out and their second round is nearly empty, while 128 x 192 still come out in one: 11,008 x 4,096 against
// 315 rows (174 tiles of 128 x 192) 82 / 56, 11,008 x 2,048 against 303 47 / 34, 4,224 x 3,584 against 957 (176) 64 / 47, 3,072 x 4,864 against 1,323 78 / 60, 3,072 x 2,560 against 1,385 51 / 38.
// With K of 1,536 too: 8,960 x 1,536 against 397 rows (188) 35 / 27, 18,944 x 1,536 against 150 33 / 27, 3,584 x 1,536 against 1,710 (196 of 256 x 128) 34 / 31.
// But not 256 x 160 where the others come out in two rounds and K is short or the last rows are mostly padding: 8,960 x 1,536 against 787 36 / 41, 18,944 x 2,048 against 269 44 / 47, 18,944 x 5,120
// against 330 89 / 95 (4,608 x 1,792 against 1,907, 540 of 128 x 128, 56 / 42); nor one round of 128 x 128 with that much padding and K under 4,096: 8,960 x 1,536 against 265 (210) 18.0 / 21.0, x 3,584
// 35.4 / 38.0, 13,824 x 2,048 against 140 (216) 21.6 / 25.1 (against 1,536 x 1,536, 2,073 rows, 25 / 22).
// K from 768 to 1,535 (us, the others / these; 0.5B sizes unless said). With the gate wherever the others' tiles of 64 rows x 64 outputs are more than one round: 4,864 x 896 against 171 rows (228 of
// them) 10.9 / 12.9, against 202 (304) 14.3 / 13.1, 467 22.4 / 16.7, 1,041 31.6 / 25.0, 1,430 43.9 / 29.2, 2,048 46.9 / 37.2, 3,967 92.9 / 73.8; 2,816 x 1,024 against 200 (176) 10.1 / 13.0,
// 370 (264) 13.8 / 13.3, 2,803 49.0 / 32.6; 3,072 x 768 against 279 (240) 9.0 / 11.1, 2,968 43.2 / 33.5. Stored as bfloat16 from seven tenths of a round of 128 x 128 on: 1,152 x 896 against 1,162 (90)
// 9.8 / 12.1, 2,453 (180) 12.9 / 12.8, 3,209 (234) 19.1 / 13.5; 4,096 x 1,024 against 398 (128) 10.8 / 13.2, 988 (256) 23.4 / 14.6, 3,302 56.9 / 31.7; 4,864 x 896 against 3,039 55.5 / 29.4. Float outputs,
// whose way out is longer, from eight tenths: 896 x 896 against 2,734 (154) 14.3 / 17.6, 3,760 (210) 20.9 / 18.6.
// With the gate and K from 1,536 from 0.55 of a round on: 8,960 x 1,536 against 268 rows 37.9 / 27.5, 819 77.4 / 55.6, 2,021 140 / 107; 5,632 x 2,048 against 107 (88 tiles of 128 x 64) 22.4 / 23.7, 225 (176)
// 26.4 / 24.4, 2,116 124 / 102. Up to 256 rows against K under 2,048 with few tiles of 128 x 128 stay where they were (5,632 x 1,536 and narrower are even there; 8,960 against 245 36.6 / 26.2 is left).
bool tall_pays(int M, int N, int K, TallKind kind) {
  static const bool switched_off = [] { const char* e = getenv("ALOFA_WIDE_TILES"); return e != nullptr && e[0] == '0'; }();     // (for measurements)
  if (switched_off || M <= 64 || K % 32 != 0 || K < 768) return false;
  const bool gated = kind == kTallGated;
  double fill = 0;
  const int form = pick_tall(M, N, K, gated, &fill), cus = compute_units();
  const int64_t small = static_cast<int64_t>((M + 127) / 128) * ((N + 127) / 128);
  if (gated) {
    if (K < 1536) return static_cast<int64_t>((M + 63) / 64) * ((N + 63) / 64) > cus;
    if (K < 2048 && M <= 256 && 10 * small < 8 * cus) return false;
    return fill >= 0.55;
  }
  if (K < 1536) return 10 * small >= (kind == kTallRows16 ? 7 : 8) * static_cast<int64_t>(cus);
  const int full = (M + kPlain[form].rows - 1) / kPlain[form].rows * kPlain[form].rows;      // rows with the last tile's padding
  if (kPlain[form].columns == 160 && small <= 2 * cus && (K <= 2048 || 4 * M < 3 * full)) return false;
  if (kPlain[form].rows == 128 && kPlain[form].columns == 128 && small <= cus && K < 4096 && 5 * M < 4 * full) return false;
  if (small > cus) return K >= 2048 || fill >= 0.72;
  if (K < 2048) return fill >= 0.80;
  if (K < 8960 && static_cast<int64_t>(N) * K < 20000000) return fill >= 0.735;
  return fill >= (K < 5120 ? 0.70 : 0.57);
}

template <int kEpilogue, typename TO, typename T>
static int launch_form(void* out, int64_t ldo, const void* A, int64_t lda, const void* W, const void* W2, int64_t ldw, const float* bias, int M, int N, int K, hipStream_t stream) {
  constexpr int kOutCols = is_gated(kEpilogue) ? T::TN / 2 : T::TN;
  const int tiles_n = (N + kOutCols - 1) / kOutCols, tiles_m = (M + T::TM - 1) / T::TM;
  gemm_tall_kernel<kEpilogue, TO, T><<<tiles_n * tiles_m, 512, 0, stream>>>(static_cast<TO*>(out), ldo, static_cast<const bf16_t*>(A), lda, static_cast<const bf16_t*>(W),
                                                                          static_cast<const bf16_t*>(W2), ldw, bias, M, N, K, tiles_m, tiles_n);
  return check_launch("gemm_tall");
}

template <int kEpilogue, typename TO>
static int launch_picked(void* out, int64_t ldo, const void* A, int64_t lda, const void* W, const void* W2, int64_t ldw, const float* bias, int M, int N, int K, hipStream_t stream) {
  double fill = 0;
  const int form = pick_tall(M, N, K, is_gated(kEpilogue), &fill);
  if constexpr (is_gated(kEpilogue)) {
    switch (form) {
      case 0: return launch_form<kEpilogue, TO, Tall<256, 320, 4, 2, 2, 2, 2, 1>>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, stream);
      case 1: return launch_form<kEpilogue, TO, Tall<256, 256, 4, 2, 2, 2, 2>>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, stream);
      case 2: return launch_form<kEpilogue, TO, Tall<256, 192, 4, 2, 2, 2, 1>>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, stream);
      case 3: return launch_form<kEpilogue, TO, Tall<256, 160, 8, 1, 3, 3, 2>>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, stream);
      case 4: return launch_form<kEpilogue, TO, Tall<256, 128, 4, 2, 3, 1, 1>>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, stream);
      case 5: return launch_form<kEpilogue, TO, Tall<128, 256, 2, 4, 3, 1, 1>>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, stream);
      case 6: return launch_form<kEpilogue, TO, Tall<128, 192, 4, 2, 3, 2, 1>>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, stream);
      default: return launch_form<kEpilogue, TO, Tall<128, 128, 4, 2, 3, 1, 1>>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, stream);
    }
  } else {
    switch (form) {
      case 0: return launch_form<kEpilogue, TO, Tall<256, 320, 4, 2, 2, 2, 2, 1>>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, stream);
      case 1: return launch_form<kEpilogue, TO, Tall<256, 256, 2, 4, 2, 1, 1>>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, stream);
      case 2: return launch_form<kEpilogue, TO, Tall<256, 192, 4, 2, 2, 2, 1>>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, stream);
      case 3: return launch_form<kEpilogue, TO, Tall<256, 160, 8, 1, 3, 3, 2>>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, stream);
      case 4: return launch_form<kEpilogue, TO, Tall<256, 128, 4, 2, 3, 1, 1>>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, stream);
      case 5: return launch_form<kEpilogue, TO, Tall<128, 192, 4, 2, 3, 2, 1>>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, stream);
      default: return launch_form<kEpilogue, TO, Tall<128, 128, 4, 2, 3, 1, 1>>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, stream);
    }
  }
}

int launch_tall(int epilogue, int o_dtype, void* out, int64_t ldo, const void* A, int64_t lda, const void* W, const void* W2, int64_t ldw, const float* bias, int M, int N, int K,
                hipStream_t stream) {
  if (epilogue == kMfStore && o_dtype == kBF16) return launch_picked<kMfStore, bf16_t>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, stream);
  if (epilogue == kMfStore && o_dtype == kF32) return launch_picked<kMfStore, float>(out, ldo, A, lda, W, W2, ldw, bias, M, N, K, stream);
  if (epilogue == kMfResidual && o_dtype == kF32) return launch_picked<kMfResidual, float>(out, ldo, A, lda, W, W2, ldw, nullptr, M, N, K, stream);
  if (epilogue == kMfSwiglu && o_dtype == kBF16 && W2 != nullptr) return launch_picked<kMfSwiglu, bf16_t>(out, ldo, A, lda, W, W2, ldw, nullptr, M, N, K, stream);
  if (epilogue == kMfGeglu && o_dtype == kBF16 && W2 != nullptr) return launch_picked<kMfGeglu, bf16_t>(out, ldo, A, lda, W, W2, ldw, nullptr, M, N, K, stream);
  ALOFA_REQUIRE(false, "gemm_wide: unsupported epilogue %d with out dtype %d", epilogue, o_dtype);
}

}  // namespace alofa

using namespace alofa;

// Which form the sizes get (its number in kPlain or kGated), whether it is the tiled product's choice or not.
extern "C" int alofa_gemm_wide_form(int M, int N, int K, int gated) {
  double fill = 0;
  return pick_tall(M, N, K, gated != 0, &fill);
}

// Whether alofa_gemm_mfma takes these tiles (gated: 0 float outputs, 1 with the gate, 2 bfloat16 outputs without).
extern "C" int alofa_gemm_wide_pays(int M, int N, int K, int gated) { return tall_pays(M, N, K, static_cast<TallKind>(gated)); }

// The same product by these tiles whatever the sizes (alofa_gemm_mfma takes them where they pay): K a multiple of 32. The operands as for
// alofa_gemm_mfma; norm_w and eps stand where alofa_gemm_skinny has them and must be null and zero (no norm rides on this kernel).
extern "C" int alofa_gemm_wide(void* out, int o_dtype, int64_t ldo, const void* A, int64_t lda, const void* W, const void* W2, int64_t ldw,
                               const float* bias, int M, int N, int K, int epilogue, const float* norm_w, float eps, hipStream_t stream) {
  ALOFA_REQUIRE(M > 0 && N > 0 && K > 0 && K % 32 == 0, "gemm_wide: M=%d N=%d K=%d must be positive, K a multiple of 32", M, N, K);
  ALOFA_REQUIRE(lda % 8 == 0 && ldw % 8 == 0 && lda >= K && ldw >= K && ldo >= N, "gemm_wide: lda=%lld, ldw=%lld must be multiples of 8 and cover K, ldo=%lld cover N",
                static_cast<long long>(lda), static_cast<long long>(ldw), static_cast<long long>(ldo));
  ALOFA_REQUIRE(reinterpret_cast<uintptr_t>(A) % 16 == 0 && reinterpret_cast<uintptr_t>(W) % 16 == 0 && reinterpret_cast<uintptr_t>(W2) % 16 == 0,
                "gemm_wide: operands must be 16-byte aligned");
  ALOFA_REQUIRE(norm_w == nullptr && eps == 0.f, "gemm_wide: no norm rides on this kernel");
  return launch_tall(epilogue, o_dtype, out, ldo, A, lda, W, W2, ldw, bias, M, N, K, stream);
}
