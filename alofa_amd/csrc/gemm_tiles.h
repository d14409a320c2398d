// What the tiled products on the matrix cores share: operand types, the epilogues' numbers, which tile a block
// computes, the order of a slab's 16-byte chunks in LDS, and what a wave does with its finished tiles.
#pragma once

#include "common.h"

namespace alofa {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

enum MfmaEpilogue : int { kMfStore = 0, kMfResidual = 1, kMfSwiglu = 2, kMfArgmax = 3, kMfGeglu = 4, kMfTurn = 5 };

// Which tile a block computes. The chip is eight dies, each with an L2 of its own, and blocks go to the
// dies in turn (block i to die i % 8). Dealt out row by row, every die computes tiles from all over the
// output and pulls all of A and all of W through its L2: fine while both fit there, and measured a few
// percent faster then than the path below; with operands beyond the L2s (projections of 7B-sized models
// and up) it costs up to a fifth of the time. For those (by_die) the tiles are numbered along a path that
// stays within squares of 8 x 8 tiles (8 tile rows at a time, column by column), every die takes one
// contiguous stretch of the path, and the blocks resident on a die together share a handful of A and W
// panels. With K shared out, the shares are the slowest index (blocks of different shares have nothing
// in common).
struct TilePlace {
  int bm, bn, share;
};
__device__ __forceinline__ TilePlace place_tile(int block, int tiles_m, int tiles_n, int shares, bool by_die) {
  constexpr int kDies = 8, kGroup = 8;
  const int tiles = tiles_m * tiles_n, total = tiles * shares;
  if (!by_die) return {block % tiles / tiles_n, block % tiles_n, block / tiles};
  const int die = block % kDies, local = block / kDies;
  const int step = die * (total / kDies) + min(die, total % kDies) + local;   // dies before this one hold that many blocks
  const int t = step % tiles;
  const int per_group = kGroup * tiles_n, first_m = (t / per_group) * kGroup, within = t % per_group;
  const int rows = min(tiles_m - first_m, kGroup);
  return {first_m + within % rows, within / rows, step / tiles};
}

// A row of a slab in LDS is 128 bytes; its eight 16-byte chunks are permuted by the row's number (chunk c of row r lies at
// place c ^ swz(r)), so that the 16 or 32 rows whose fragments are read together fall on distinct banks.
__device__ __forceinline__ int swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// What a wave does with its finished tiles (WTM x WTN of 32 x 32, the block's tile at m0, n0 of the output).
template <int kEpilogue, typename TO, int WTM, int WTN>
__device__ __forceinline__ void tile_epilogue(f32x16 (&acc)[WTM][WTN], TO* __restrict__ out, int64_t ldo,
                                              const float* __restrict__ bias, int M, int N, int m0, int n0, int wm, int wn, int lane) {
  constexpr int kGateTiles = WTN / 2;
  const int col = lane % 32, row_base = (lane / 32) * 4;
  constexpr int kOutTiles = is_gated(kEpilogue) ? kGateTiles : WTN;
#pragma unroll
  for (int i = 0; i < WTM; ++i) {
#pragma unroll
    for (int j = 0; j < kOutTiles; ++j) {
      const int n = n0 + wn * 32 * kOutTiles + j * 32 + col;
      if (n >= N) continue;
      const float b = (bias && kEpilogue == kMfStore) ? bias[n] : 0.f;
      const int m_first = m0 + wm * 32 * WTM + i * 32 + row_base;      // element e: row m_first + 8 * (e / 4) + e % 4
      TO* column = out + n;
      float old[16];
      if (kEpilogue == kMfResidual) {      // all sixteen old values set out before any is needed
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int m = m_first + 8 * (e / 4) + e % 4;
          old[e] = m < M ? load_f32(column + static_cast<int64_t>(m) * ldo) : 0.f;
        }
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = m_first + 8 * (e / 4) + e % 4;
        if (m >= M) continue;
        TO* dst = column + static_cast<int64_t>(m) * ldo;
        if (kEpilogue == kMfStore) {
          store_f32(dst, acc[i][j][e] + b);
        } else if (kEpilogue == kMfResidual) {
          store_f32(dst, old[e] + acc[i][j][e]);
        } else {
          const float g = acc[i][j][e];
          store_f32(dst, gate_of<kEpilogue == kMfGeglu>(g) * acc[i][(j + kGateTiles) % WTN][e]);
        }
      }
    }
  }
}

// (gemm_tall.hip) Tiles of up to 256 x 320 outputs by eight waves, for many rows. `pays`: whether they are the tiled product's choice for these sizes.
// `launch`: the product with the epilogue as above and `out` of type o_dtype; K a multiple of 32. 0, or 1 with the error set.
enum TallKind : int { kTallFloat = 0, kTallGated = 1, kTallRows16 = 2 };      // float outputs, with the gate, bfloat16 outputs
bool tall_pays(int M, int N, int K, TallKind kind);
int launch_tall(int epilogue, int o_dtype, void* out, int64_t ldo, const void* A, int64_t lda, const void* W, const void* W2, int64_t ldw, const float* bias,
                int M, int N, int K, hipStream_t stream);

}  // namespace alofa
