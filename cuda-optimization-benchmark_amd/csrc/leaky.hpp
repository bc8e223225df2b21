// leaky kernel template (instantiated by leaky.hip).
//
// Op: tasks/leaky/reference.py:26-37 (the fp32 step loop is also the oracle, :40) and the
// step order of tasks/leaky/prompt.md.
//
// The recurrence is nonlinear (threshold reset), so time stays serial and the
// parallelism is over the B*H neurons.  A thread owns kVec adjacent neurons of one batch
// row and walks all T steps; step t reads x[t] (one 4*kVec-byte load, coalesced across
// the wave) and writes spikes[t].  Inputs are prefetched kDepth steps ahead in a register
// ring so each wave keeps kDepth loads in flight.  Arithmetic is fp32 with contraction
// disabled: each of beta*mem, +x, reset*th and the subtraction rounds once, exactly as
// the eager reference does, so spikes and final_mem are bit-identical to it.
// HBM-bound: 8 algorithmic bytes per neuron-step (4 in, 4 out).
#pragma once

#include <type_traits>

#include "common.hpp"

#pragma clang fp contract(off)

namespace taskops {

namespace leaky_detail {
template <int kVec>
struct Vec;
template <>
struct Vec<1> {
  using T = float;
};
template <>
struct Vec<2> {
  using T = float __attribute__((ext_vector_type(2)));
};
template <>
struct Vec<4> {
  using T = float __attribute__((ext_vector_type(4)));
};

template <bool kNT, class V>
__device__ __forceinline__ V ld(const V* p) {
  if constexpr (kNT) return __builtin_nontemporal_load(p);
  return *p;
}
template <bool kNT, class V>
__device__ __forceinline__ void st(V v, V* p) {
  if constexpr (kNT)
    __builtin_nontemporal_store(v, p);
  else
    *p = v;
}
}  // namespace leaky_detail

template <int kThreads, int kVec, int kDepth, bool kNT>
__global__ __launch_bounds__(kThreads) void leaky_kernel(
    const float* __restrict__ x, const float* __restrict__ mem0, const float* __restrict__ beta,
    const float* __restrict__ threshold, int T, int64_t N, int H, float* __restrict__ spikes,
    float* __restrict__ final_mem) {
  using namespace leaky_detail;
  using V = typename Vec<kVec>::T;
  const int64_t n0 = ((int64_t)blockIdx.x * kThreads + threadIdx.x) * kVec;
  if (n0 >= N) return;
  const int h0 = (int)(n0 % H);

  float b[kVec], th[kVec], m[kVec];
#pragma unroll
  for (int k = 0; k < kVec; ++k) {
    float bb = beta[h0 + k];
    // clamp to [0, 1]; a NaN stays NaN, as torch.clamp leaves it
    bb = bb < 0.0f ? 0.0f : (bb > 1.0f ? 1.0f : bb);
    b[k] = bb;
    th[k] = threshold[h0 + k];
    m[k] = mem0[n0 + k];
  }

  const V* xp = reinterpret_cast<const V*>(x + n0);
  V* sp = reinterpret_cast<V*>(spikes + n0);
  const int64_t stride = N / kVec;  // one time step, in units of V

  V ring[kDepth];
#pragma unroll
  for (int j = 0; j < kDepth; ++j)
    if (j < T) ring[j] = ld<kNT>(xp + (int64_t)j * stride);

  for (int t0 = 0; t0 < T; t0 += kDepth) {
#pragma unroll
    for (int j = 0; j < kDepth; ++j) {
      const int t = t0 + j;
      if (t >= T) break;
      const V xv = ring[j];
      if (t + kDepth < T) ring[j] = ld<kNT>(xp + (int64_t)(t + kDepth) * stride);
      V s;
      const float* xs = reinterpret_cast<const float*>(&xv);
      float* ss = reinterpret_cast<float*>(&s);
#pragma unroll
      for (int k = 0; k < kVec; ++k) {
        const float reset = (m[k] >= th[k]) ? 1.0f : 0.0f;
        const float decayed = b[k] * m[k];
        const float charged = decayed + xs[k];
        const float drop = reset * th[k];
        m[k] = charged - drop;
        ss[k] = (m[k] >= th[k]) ? 1.0f : 0.0f;
      }
      st<kNT>(s, sp + (int64_t)t * stride);
    }
  }
#pragma unroll
  for (int k = 0; k < kVec; ++k) final_mem[n0 + k] = m[k];
}

// ---------------------------------------------------------------------------------------
// leaky_rows_kernel: 64 neurons per wave, one per lane, with the time steps moved four at a time.
//
// What bounds a small layer (few neurons) is how far ahead of the serial step loop its loads
// run: bytes in flight are neurons x 4 x steps ahead, and a wave has at most 63 memory
// operations outstanding, loads and stores together.  One operation here covers 64 neurons x 4
// steps: lane l moves 16 bytes, neurons 4 (l % 16) .. +3 of step 4 b + l / 16 of block b, and
// the wave's own LDS turns blocks between that layout and one neuron per lane.  So kRing
// blocks, 4 kRing steps, are in flight (up to 32 blocks), where one neuron pair per lane and
// step reaches 31 steps (16 as built): T = 160, N = 17000 22.2 -> 9.1 us (21.9 MB, floor 4.3
// and the serial steps at about 20 ns each).  The 16-byte accesses need a float's alignment only, so odd H and any base take
// the same path.  The loop has no branch around a load or store (an offset past the buffer
// reads zero and stores nothing): behind branches the compiler's waits drained the ring.
// Same operations in the same order as leaky_kernel, the same bits.
//
// The last wave takes the last 64 neurons and stores only those no other wave owns.
// ---------------------------------------------------------------------------------------
namespace leaky_detail {
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
constexpr unsigned kOutOfRange = 0x80000000u;

// kPart: kFull, the wave owns its 64 columns; kTail, the last 4 or more of them; kFew, fewer.
enum LeakyPart : int { kFull = 0, kTail = 1, kFew = 2 };
template <int kRing, LeakyPart kPart>
__device__ __forceinline__ void run_rows(const float* __restrict__ x, const float* __restrict__ mem0,
                                         const float* __restrict__ beta, const float* __restrict__ threshold, int T,
                                         int N, int H, float* __restrict__ spikes, float* __restrict__ final_mem,
                                         int n0, int owned, float* lds) {
  const int lane = threadIdx.x % kWave, r = lane / 16, g = 4 * (lane % 16);
  const int n = n0 + lane, h = n % H;
  float b = beta[h];
  b = b < 0.0f ? 0.0f : (b > 1.0f ? 1.0f : b);  // a NaN stays NaN, as torch.clamp leaves it
  const float th = threshold[h];
  // reset * th for reset = 1 and 0: a product each, taken once (0 * th is not 0 for every th).
  const float drop1 = 1.0f * th, drop0 = 0.0f * th;
  float m = mem0[n];
  bool fired = m >= th;

  // (T + 4) * N * 4 bytes fit 31 bits (the launch checks), so no row of a block that is computed
  // wraps.
  const unsigned bytes = (unsigned)T * (unsigned)N * 4u;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x), (short)0, (int)bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(spikes, (short)0, (int)bytes, 0x00020000);
  constexpr int kNT = 2;  // non-temporal
  // Offsets of the next block's load and store, one addition per block.  A store's rows past T
  // lie past the descriptor's end (and so, by wrapping, does the store of block -1).  The loads run
  // up to kRing + 1 blocks ahead: past T they read zero, or, where the offset wraps in a layer of
  // more than 32 M neurons, some row of the input; nothing uses either.
  unsigned lat = ((unsigned)r * (unsigned)N + (unsigned)(n0 + g)) * 4u;
  const unsigned step4 = 16u * (unsigned)N;
  auto load = [&]() {
    const f32x4 v = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, lat, 0, kNT));
    lat += step4;
    return v;
  };
  // A block of the spikes from its LDS stage to memory.  The tail: its own columns c0 .. 63 in
  // 16-byte groups, the last one ending at column 63; fewer than four, one float per lane.
  const int c0 = kWave - owned;
  const int from = kPart == kFull ? g : (kPart == kFew ? min(c0 + lane % 16, kWave - 1) : min(c0 + g, kWave - 4));
  const bool mine = kPart == kFull || (kPart == kFew ? lane % 16 < owned : c0 + g < kWave);
  unsigned sat = ((unsigned)r * (unsigned)N + (unsigned)(n0 + from)) * 4u - step4;
  auto staged = [&](const float* stage) {  // what this lane stores of a block
    u32x4 v = {0u, 0u, 0u, 0u};
    if constexpr (kPart == kFew) {
      v[0] = __float_as_uint(stage[r * kWave + from]);
    } else if constexpr (kPart == kTail) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = __float_as_uint(stage[r * kWave + from + e]);
    } else {
      v = *reinterpret_cast<const u32x4*>(stage + r * kWave + g);
    }
    return v;
  };
  auto store = [&](u32x4 v, unsigned at) {
    const unsigned off = mine ? at : kOutOfRange;
    if constexpr (kPart == kFew)
      __builtin_amdgcn_raw_buffer_store_b32(v[0], rs, off, 0, kNT);
    else
      __builtin_amdgcn_raw_buffer_store_b128(v, rs, off, 0, kNT);
  };
  float* xin = lds;              // [2][4][64]
  float* sout = lds + 8 * kWave;  // [2][4][64]
  // A wave's LDS operations run in order, and the compiler keeps this order because it cannot tell
  // the addresses apart.  A fence that says so changed its schedule: N = 17000, T = 160 8.5 -> 8.4 us,
  // but N = 800,199, T = 60 106 -> 109 and N = 2,096,640, T = 20 59 -> 61.
  auto stage_in = [&](int blk, f32x4 q, float (&xv)[4]) {
    float* st = xin + (blk & 1) * 4 * kWave;
    *reinterpret_cast<f32x4*>(st + r * kWave + g) = q;
#pragma unroll
    for (int k = 0; k < 4; ++k) xv[k] = st[k * kWave + lane];
  };

  // Each load of the prologue is followed by a store that goes nowhere, as every load of the
  // loop is by a block's store: the loop's waits count both, and the compiler takes the
  // smaller count of the two ways into the loop (half the ring stood idle without).
  f32x4 ring[kRing];
#pragma unroll
  for (int j = 0; j < kRing; ++j) {
    ring[j] = load();
    store(u32x4{0u, 0u, 0u, 0u}, kOutOfRange);
  }
  float xv[4], xn[4];
  stage_in(0, ring[0], xv);
  ring[0] = load();
  store(u32x4{0u, 0u, 0u, 0u}, kOutOfRange);

  // Block blk's four steps (kGuard: only those below T).  The previous block's spikes and the
  // next block's inputs are read from LDS before the steps and used after them.
  auto block = [&](int blk, f32x4& next, auto guard) {
    constexpr bool kGuard = decltype(guard)::value;
    const u32x4 done = staged(sout + ((blk - 1) & 1) * 4 * kWave);
    stage_in(blk + 1, next, xn);
    next = load();
    __builtin_amdgcn_sched_barrier(0);
    float* st = sout + (blk & 1) * 4 * kWave;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float decayed = b * m;
      const float charged = decayed + xv[k];
      const float next_m = charged - (fired ? drop1 : drop0);
      if (!kGuard || 4 * blk + k < T) m = next_m;
      fired = m >= th;
      st[k * kWave + lane] = fired ? 1.0f : 0.0f;
    }
    __builtin_amdgcn_sched_barrier(0);
    store(done, sat);
    sat += step4;
#pragma unroll
    for (int k = 0; k < 4; ++k) xv[k] = xn[k];
  };
  const int nblk = (T + 3) / 4;
  int b0 = 0;
  for (; 4 * (b0 + kRing) <= T; b0 += kRing) {
#pragma unroll
    for (int j = 0; j < kRing; ++j) block(b0 + j, ring[(j + 1) % kRing], std::integral_constant<bool, false>{});
  }
#pragma unroll
  for (int j = 0; j < kRing; ++j)
    if (b0 + j < nblk) block(b0 + j, ring[(j + 1) % kRing], std::integral_constant<bool, true>{});
  store(staged(sout + ((nblk - 1) & 1) * 4 * kWave), sat);
  if (kPart == kFull || lane >= c0) final_mem[n] = m;
}
}  // namespace leaky_detail

template <int kWaves, int kRing>
__global__ __launch_bounds__(kWaves * kWave) void leaky_rows_kernel(
    const float* __restrict__ x, const float* __restrict__ mem0, const float* __restrict__ beta,
    const float* __restrict__ threshold, int T, int N, int H, float* __restrict__ spikes,
    float* __restrict__ final_mem) {
  __shared__ __attribute__((aligned(16))) float lds[kWaves][16 * kWave];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int n0 = ((int)blockIdx.x * kWaves + wave) * kWave;
  if (n0 >= N) return;
  if (n0 + kWave <= N)
    leaky_detail::run_rows<kRing, leaky_detail::kFull>(x, mem0, beta, threshold, T, N, H, spikes, final_mem, n0, kWave, lds[wave]);
  else if (N - n0 >= 4)
    leaky_detail::run_rows<kRing, leaky_detail::kTail>(x, mem0, beta, threshold, T, N, H, spikes, final_mem, N - kWave,
                                                       N - n0, lds[wave]);
  else
    leaky_detail::run_rows<kRing, leaky_detail::kFew>(x, mem0, beta, threshold, T, N, H, spikes, final_mem, N - kWave,
                                                      N - n0, lds[wave]);
}

}  // namespace taskops
