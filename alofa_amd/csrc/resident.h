// What the kernels that run all layers of a decode step in one launch share (decode_resident.hip, decode_groups.hip): the layers' table, the area of places of eight
// bytes that their blocks exchange values in, and the wait for values.
#pragma once

#include "common.h"

#include <float.h>

#include <type_traits>

namespace alofa {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned long long u64;

// (pointers that are read from memory are told to lead to global memory: a load by a pointer of any kind is waited for with LDS's own, at every barrier)
#define ALOFA_GLOBAL __attribute__((address_space(1)))
typedef ALOFA_GLOBAL const char* gbytes;

// one per layer, in device memory
struct ResidentLayer {
  gbytes w_qkv;
  ALOFA_GLOBAL const float* b_qkv;
  gbytes w_o;
  gbytes w_gate;
  gbytes w_up;
  gbytes w_down;
  ALOFA_GLOBAL const float* norm0;
  ALOFA_GLOBAL const float* norm1;
  ALOFA_GLOBAL bf16_t* k_cache;
  ALOFA_GLOBAL bf16_t* v_cache;
};

template <typename V>
__device__ __forceinline__ V load_global(gbytes at) { return *reinterpret_cast<ALOFA_GLOBAL const V*>(at); }

constexpr int kLayerWords = sizeof(ResidentLayer) / 4, kResMaxLayers = 64;
struct LayerWords {
  uint32_t w[kLayerWords];
};

constexpr int kResBlocks = 256, kResThreads = 512, kResWaves = 8;
constexpr int kResMaxWidth = 1024, kResMaxFF = 6144, kResMaxRows = 16, kResMaxParts = 16, kResShares = 8, kResMaxGroup = 8;
// A launch waits until all its blocks are on the chip, and two processes may have one each on their way: a block takes at most half of a compute unit's registers (the launch bounds) and LDS.
// kLdsOf: the bytes of a kernel's __shared__ arrays, all of which are named to it; one that does not fit beside another launch's blocks must not build (its waits would end at their limit).
constexpr int kResMostLds = 80 * 1024;
template <typename... Arrays>
constexpr int kLdsOf = (((static_cast<int>(sizeof(Arrays)) + 15) / 16 * 16) + ...);
constexpr int kLimit = 4 << 20;      // asks of about a microsecond

// where the values lie in the area, in places of eight bytes (the first 32 hold the step counter and `stop`)
constexpr int kAtRowsA = 32, kAtRowsB = kAtRowsA + kResMaxRows * kResMaxWidth, kAtQkv = kAtRowsB + kResMaxRows * kResMaxWidth,
              kAtParts = kAtQkv + kResMaxRows * 4096, kAtAttn = kAtParts + kResBlocks * kResMaxGroup * 66, kAtAct = kAtAttn + kResMaxRows * kResMaxWidth / 2,
              kAtDown = kAtAct + kResMaxRows * kResMaxFF / 2, kAreaPlaces = kAtDown + kResMaxWidth * kResMaxRows * kResShares;
constexpr int kResGroups = 4;      // groups of blocks that take rows of their own through the layers, at most: each has such places of its own, one behind the other

struct ResidentArgs {
  float* hidden;
  const ResidentLayer* layers;
  const int32_t* positions;
  const int32_t* table;
  const int64_t* slots;
  const float* cos_t;
  const float* sin_t;
  u64* area;
  int* failed;
  int n_layers, M, H, FF, heads, kv_heads, max_blocks, bs_shift, parts, has_bias, limit;
  float scale, eps0, eps1;
};

__device__ __forceinline__ void put(u64* at, uint32_t value, uint32_t stamp) {
  __hip_atomic_store(at, (static_cast<u64>(stamp) << 32) | value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void put(u64* at, float value, uint32_t stamp) { put(at, __float_as_uint(value), stamp); }

struct Wait {      // of one wave: the area as a buffer resource (reads past the caches), the stamp waited for, whether waits are over
  __amdgpu_buffer_rsrc_t area;
  u64* words;
  int* failed;
  int limit;      // asks until a wait is given up
  uint32_t stamp;
  bool dead;

  // Two places at once (16 bytes), `at`: the first one's number, even. That such a load sees each of the two stores of eight bytes whole, never a new stamp beside an old
  // value, is how memory serves an aligned piece of sixteen bytes, and taken for granted here (none of 3.9e10 loads beside stores saw half of one): what is promised of a load ends at eight bytes. With loads of eight (64 lanes
  // a run of 64 places, no register in memory) a step of 1, 4, 8, 12 and 16 rows takes 454, 522, 581, 663 and 713 us instead of 449, 499, 529, 599 and 641.
  __device__ __forceinline__ u32x4 two(int at) const {
    constexpr int kPastCaches = 1 | 16;      // sc0, sc1
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(area, at * 8, 0, kPastCaches));
  }
  // whether to go on asking (uniform over the wave)
  __device__ __forceinline__ bool again(int& asked) {
    if ((++asked & 255) == 0 || asked >= limit) {
      dead = asked >= limit || __any(__hip_atomic_load(words + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0);
      if (dead) {
        __hip_atomic_store(words + 1, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(failed, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
    return !dead;
  }
  // N pairs of places at at(i), until all bear the stamp. Where waits are over the values are NaN, in 32 bits and as two numbers of 16: whatever is computed from
  // them is NaN and leaves as such, so that no number that a row ends with comes from a wait that was given up, whichever wave gave it up and when.
  // (told which way is the usual one, the compiler keeps no register in memory: a step of 8 rows 545 -> 529 us, of 12 617 -> 599)
  // (kWhole: the stamps of values that are NaN are set as well; where a wait lies within a loop, what they were before would be kept in registers for that way)
  template <bool kWhole = false, int N, typename At>
  __device__ __forceinline__ void pairs(u32x4 (&v)[N], At&& at) {
    constexpr uint32_t kNaN = 0x7fc07fc0u;
    int asked = 0;
    if (__builtin_expect(!dead, 1)) do {
      asm volatile("" ::: "memory");      // (read anew every time)
#pragma unroll
      for (int i = 0; i < N; ++i)
        v[i] = two(at(i));
      bool here = true;
#pragma unroll
      for (int i = 0; i < N; ++i) here &= v[i][1] == stamp && v[i][3] == stamp;
      if (__builtin_expect(__all(here), 1)) return;
    } while (again(asked));
#pragma unroll
    for (int i = 0; i < N; ++i) {
      v[i][0] = kNaN, v[i][2] = kNaN;
      if constexpr (kWhole) v[i][1] = stamp, v[i][3] = stamp;
    }
  }
};

// (decode_groups.hip) more than sixteen rows; tiled: the layers' gate, up and down are laid out in tiles
int launch_groups(const ResidentArgs& a, bool tiled, hipStream_t stream);

}  // namespace alofa

extern "C" int alofa_resident_rows(int H, int FF, int heads, int kv_heads);
