// A decode step of a layer whose heads keep a state S [dk, dv] (recurrent.hip says what is computed): rotation of the row's query and key, the state's step and its
// read-out, the norm per head, the gate, in one launch, for steps in which every request brings one row (row r is request r).
//
// Launch by launch these were three, which hand a few hundred numbers on: rotation 2.4 to 4.4 us, the recurrence 6.2 to 8.8 (made for many rows: operands by way of LDS in chunks, read-outs in
// parts), norm and gate 2.2 to 4 (4 requests, 16 heads of 64 x 64 in a captured step). What the work cannot do without is the state, read and written once: 16 KB a head.
// 1 to 64 requests of 1 to 32 heads, 1.01 to 2.2 times as fast, but a few (request, head) pairs of the widest heads, whose state one block reads and writes here: those go launch by launch
// (recurrence_step_pays in ops.py has the figures).
// Where the decays come from a projection of few channels (its rank), the block makes its head's share of it too, with the bits of the vector-unit product that makes it by itself: the launch that was
// saved took 2.6 us of a captured step, the products hide behind the state's loads.
// A block takes a head of a request. The state's loads set out first (a thread has four neighbouring columns of every so-manieth row, 16 bytes a load), the row's operands are made meanwhile, each
// once, in LDS; the read-outs' shares meet in LDS in row order. Read-outs stay float up to the norm's end, as they are between the launches.
#include "common.h"

namespace alofa {

enum StepDecay : int { kStepPerHead = 0, kStepSigmoidRoot = 1, kStepExpNegExp = 2 };

struct StepArgs {
  bf16_t* out;
  int64_t out_stride;
  const bf16_t *q, *k, *v, *gate;
  int64_t q_stride, k_stride, v_stride, gate_stride;
  const float* decay;      // per head [heads], or z [rows, heads * dk], or (low not null) z's bias [heads * dk]
  int64_t decay_stride;
  const bf16_t *low, *low_w;      // z = low [rows, rank] low_w^T + bias, low_w [heads * dk, rank]; null: z is given
  int64_t low_stride, low_ld;
  int rank;                       // a multiple of 8, at most kStepRank
  const float* bonus;
  const float* weight;     // of the norm [heads * dv]; null: none
  float* state;
  const int32_t* req_slot;
  const float *cos_t, *sin_t;      // [positions, dk / 2]; null: queries and keys as they are
  const int32_t* positions;
  int heads, dk, dv, decay_kind, before_update;
  float inv_tau, q_scale, k_scale, eps;
};

constexpr int kStepThreads = 512, kStepMost = 256, kStepRank = 64;      // kStepMost: key and value channels of a head
static_assert(kStepRank == 64, "eight sums of eight channels meet");

// kRows: rows of the state a thread has at most
template <int kRows>
__global__ void __launch_bounds__(kStepThreads) recurrence_step_kernel(StepArgs a) {
  __shared__ float qs[kStepMost], ks[kStepMost], ws[kStepMost], us[kStepMost];
  __shared__ __attribute__((aligned(16))) float vs[kStepMost], shares[kStepThreads * 4];
  __shared__ float scratch[kStepThreads / kWave];
  const int h = blockIdx.x, r = blockIdx.y, tid = threadIdx.x, dk = a.dk, dv = a.dv;
  const int quads = dv / 4, every = kStepThreads / quads, quad = tid % quads, first = tid / quads;      // this thread's columns 4 quad .. + 3 of rows first, first + every, ..
  const bool works = first < every;
  float4* S = reinterpret_cast<float4*>(a.state + (static_cast<int64_t>(a.req_slot[r]) * a.heads + h) * dk * dv);
  float4 s[kRows];
#pragma unroll
  for (int n = 0; n < kRows; ++n) {
    const int i = first + n * every;
    s[n] = works && i < dk ? S[static_cast<int64_t>(i) * quads + quad] : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  // the decays' projection: a thread of the second half has a key channel; its weights and the row set out with the state
  uint4 lw[kStepRank / 8], lx[kStepRank / 8];
  const int key = tid - kStepMost;
  const bool projects = a.low != nullptr && key >= 0 && key < dk;
  if (a.low != nullptr) {      // (uniform)
    const int own = projects ? key : 0;
#pragma unroll
    for (int i = 0; i < kStepRank / 8; ++i) {
      const int at = 8 * i < a.rank ? 8 * i : 0;
      lw[i] = *reinterpret_cast<const uint4*>(a.low_w + static_cast<int64_t>(h * dk + own) * a.low_ld + at);
      lx[i] = *reinterpret_cast<const uint4*>(a.low + r * a.low_stride + at);
    }
  }
  float z = 0.f, weight = 1.f;      // of the channel that this thread finishes
  if (tid < dv) {
    z = bf16_to_f32(a.gate[r * a.gate_stride + h * dv + tid]);
    if (a.weight) weight = a.weight[h * dv + tid];
  }
  {
    const bf16_t *q = a.q + r * a.q_stride + h * dk, *k = a.k + r * a.k_stride + h * dk;
    const int half = dk / 2;
    if (a.cos_t) {
      if (tid < half) {
#pragma clang fp contract(off)
        const int64_t at = static_cast<int64_t>(a.positions[r]) * half + tid;
        const float c = a.cos_t[at], sn = a.sin_t[at];
        const float q0 = bf16_to_f32(q[tid]), q1 = bf16_to_f32(q[tid + half]), k0 = bf16_to_f32(k[tid]), k1 = bf16_to_f32(k[tid + half]);
        // (rounded as the rotation in a launch of its own leaves them)
        const uint32_t qr = pack_bf16x2(q0 * c - q1 * sn, q1 * c + q0 * sn), kr = pack_bf16x2(k0 * c - k1 * sn, k1 * c + k0 * sn);
        qs[tid] = __uint_as_float(qr << 16) * a.q_scale;
        qs[tid + half] = __uint_as_float(qr & 0xffff0000u) * a.q_scale;
        ks[tid] = __uint_as_float(kr << 16) * a.k_scale;
        ks[tid + half] = __uint_as_float(kr & 0xffff0000u) * a.k_scale;
      }
    } else if (tid < dk) {
      qs[tid] = bf16_to_f32(q[tid]) * a.q_scale;
      ks[tid] = bf16_to_f32(k[tid]) * a.k_scale;
    }
    if (tid >= kStepMost) {
      const int i = tid - kStepMost;
      if (i < dv) vs[i] = bf16_to_f32(a.v[r * a.v_stride + h * dv + i]);
      if (i < dk) {
        if (a.decay_kind == kStepPerHead) {
          ws[i] = a.decay[h];
        } else {
          float x = a.decay[r * a.decay_stride + h * dk + i];      // (low: the bias, decay_stride 0)
          if (projects) {      // (gemm_rows_kernel's sum: eight channels in order, then the lanes' tree)
            float p[kStepRank / 8];
#pragma unroll
            for (int n = 0; n < kStepRank / 8; ++n) {
              p[n] = dot2(lx[n].w, lw[n].w, dot2(lx[n].z, lw[n].z, dot2(lx[n].y, lw[n].y, dot2(lx[n].x, lw[n].x, 0.f))));
              if (8 * n >= a.rank) p[n] = 0.f;
            }
            x = (((p[0] + p[4]) + (p[2] + p[6])) + ((p[1] + p[5]) + (p[3] + p[7]))) + x;
          }
          ws[i] = a.decay_kind == kStepSigmoidRoot ? expf(-(fmaxf(-x, 0.f) + log1pf(expf(-fabsf(x)))) * a.inv_tau) : expf(-expf(x));
        }
        us[i] = a.bonus ? a.bonus[h * dk + i] : 0.f;
      }
    }
  }
  __syncthreads();
  if (works) {
    const float4 v = reinterpret_cast<const float4*>(vs)[quad];
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int n = 0; n < kRows; ++n) {
      const int i = first + n * every;
      if (i < dk) {
        const float q = qs[i], k = ks[i], w = ws[i];
        const float4 kv = make_float4(k * v.x, k * v.y, k * v.z, k * v.w);
        if (a.before_update) {
          const float u = us[i];
          acc.x += q * (s[n].x + u * kv.x), acc.y += q * (s[n].y + u * kv.y), acc.z += q * (s[n].z + u * kv.z), acc.w += q * (s[n].w + u * kv.w);
        }
        s[n] = make_float4(w * s[n].x + kv.x, w * s[n].y + kv.y, w * s[n].z + kv.z, w * s[n].w + kv.w);
        if (!a.before_update) acc.x += q * s[n].x, acc.y += q * s[n].y, acc.z += q * s[n].z, acc.w += q * s[n].w;
        S[static_cast<int64_t>(i) * quads + quad] = s[n];
      }
    }
    reinterpret_cast<float4*>(shares)[first * quads + quad] = acc;
  }
  __syncthreads();
  float o = 0.f;
  if (tid < dv)
    for (int g = 0; g < every && g < dk; ++g) o += shares[g * dv + tid];
  const float ss = block_sum<float, kStepThreads>(o * o, scratch);
  if (tid < dv) {
    const float inv = 1.f / sqrtf(ss / static_cast<float>(dv) + a.eps);
    float y = o * inv;
    if (a.weight) y *= weight;
    store_f32(a.out + r * a.out_stride + h * dv + tid, y * (z / (1.f + expf(-z))));
  }
}

}  // namespace alofa

using namespace alofa;

extern "C" int alofa_recurrence_step_takes(int dk, int dv) { return dk >= 1 && dk <= kStepMost && dv >= 4 && dv <= kStepMost && dv % 4 == 0; }

// out [rows, heads * dv]: the read-outs of one row a request, normed per head, gated. decay: [heads] (decay_kind 0) or z [rows, heads * dk] (1: sigmoid(z)^(1 / tau), 2: exp(-exp(z))); low not null:
// z = low [rows, rank] low_w [heads * dk, rank]^T + decay [heads * dk] (alofa_gemm_rows' bits).
extern "C" int alofa_recurrence_step(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v, int64_t v_stride,
                                     const void* gate, int64_t gate_stride, const float* decay, int64_t decay_stride, const void* low, int64_t low_stride, const void* low_w, int64_t low_ld, int rank,
                                     const float* bonus, const float* weight, float* state,
                                     const int32_t* req_slot, const float* cos_t, const float* sin_t, const int32_t* positions, int rows, int heads, int dk, int dv,
                                     int decay_kind, float tau, float q_scale, float k_scale, float eps, int before_update, hipStream_t stream) {
  ALOFA_REQUIRE(rows >= 0 && rows <= 65535 && heads > 0 && alofa_recurrence_step_takes(dk, dv), "recurrence_step: bad sizes (rows=%d heads=%d dk=%d dv=%d)", rows, heads, dk, dv);
  ALOFA_REQUIRE(decay_kind >= kStepPerHead && decay_kind <= kStepExpNegExp && decay && (decay_kind != kStepSigmoidRoot || tau > 0.f) && eps > 0.f,
                "recurrence_step: decay kind %d, tau %g, eps %g", decay_kind, static_cast<double>(tau), static_cast<double>(eps));
  ALOFA_REQUIRE(!cos_t || (sin_t && positions && dk % 2 == 0), "recurrence_step: a rotation needs both tables, positions, and an even number of key channels (%d)", dk);
  ALOFA_REQUIRE(reinterpret_cast<uintptr_t>(state) % 16 == 0, "recurrence_step: the state must be 16-byte aligned");
  ALOFA_REQUIRE(!low || (low_w && decay_kind != kStepPerHead && decay_stride == 0 && rank >= 8 && rank <= kStepRank && rank % 8 == 0 && low_stride % 8 == 0 && low_ld % 8 == 0 && low_ld >= rank &&
                         reinterpret_cast<uintptr_t>(low) % 16 == 0 && reinterpret_cast<uintptr_t>(low_w) % 16 == 0), "recurrence_step: the decays' projection takes aligned rows of 8 to %d channels in eights (%d)", kStepRank, rank);
  if (rows == 0) return 0;
  const StepArgs a = {static_cast<bf16_t*>(out), out_stride, static_cast<const bf16_t*>(q), static_cast<const bf16_t*>(k), static_cast<const bf16_t*>(v), static_cast<const bf16_t*>(gate),
                      q_stride, k_stride, v_stride, gate_stride, decay, decay_stride, static_cast<const bf16_t*>(low), static_cast<const bf16_t*>(low_w), low_stride, low_ld, rank, bonus, weight, state, req_slot, cos_t, sin_t, positions, heads, dk, dv, decay_kind, before_update,
                      decay_kind == kStepSigmoidRoot ? 1.f / tau : 0.f, q_scale, k_scale, eps};
  const int every = kStepThreads / (dv / 4), most = (dk + every - 1) / every;
  const dim3 grid(heads, rows);
  if (most <= 2) recurrence_step_kernel<2><<<grid, kStepThreads, 0, stream>>>(a);
  else if (most <= 4) recurrence_step_kernel<4><<<grid, kStepThreads, 0, stream>>>(a);
  else if (most <= 8) recurrence_step_kernel<8><<<grid, kStepThreads, 0, stream>>>(a);
  else if (most <= 16) recurrence_step_kernel<16><<<grid, kStepThreads, 0, stream>>>(a);
  else recurrence_step_kernel<32><<<grid, kStepThreads, 0, stream>>>(a);
  return check_launch("recurrence_step");
}
