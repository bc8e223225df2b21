// efficient_kan on fp32 matrix cores, weights read where they lie: kan_direct.
//
// Op: tasks/efficient_kan/reference.py:33-51, any spline order 1 .. 4 and any knot row of up
// to 32 knots, all arithmetic fp32.
//
// One contraction over the features: per feature 1 + C terms, silu(x) against Wb and the C
// bases against Ws * sc, on v_mfma_f32_16x16x4_f32 (16 batch rows x 16 columns, 4 features
// at a time: lane quarter q supplies feature 4 t + q for the A and the B operand, and the
// 1 + C MFMAs of the four features run over the terms).
//  * Weights go from memory to the B operand's registers with no packed copy in between, so
//    a call moves each weight once per 64 rows of the batch; a wave is the only reader of its
//    16 columns in its workgroup (flat_loads below: how they are read).
//  * Activations are expanded once per workgroup: 16 kR rows x a chunk of features, one pair
//    per thread: the knot interval, the order + 1 nonzero bases by the triangular Cox-de Boor
//    scheme on the interval's own knots, written into a zeroed run of C slots in LDS.  Chunk
//    c + 1 is expanded while chunk c feeds the MFMAs (two LDS stages, one barrier per chunk).
//  * The features are split over workgroups until the chip is full; each split writes its
//    fp32 tile, and the last to arrive (where there are counters, and few splits) or
//    kan_direct_sum adds the splits in order, so the result does not depend on timing.
// Each step's terms are summed from zero and then added to the running sum, so a long sum
// rounds like one of its partial sums: 1.1e-7 .. 1.8e-7 (2-norm, against fp64) where the
// row-wise kernel had 2.3e-7 .. 3.7e-7 and the fp16x3 path 2.2e-7 .. 3.6e-7.
//
// Bound: for batches up to about 32 rows by the weight stream and two launches' latency (B = 8,
// I = O = 1024, G = 5: 42 MB in 15.6 us, 71.4 with the fp16x3 path), above by the fp32 MFMAs
// and the expansion beside them: B = 1024, I = 256, O = 512, G = 16 takes 66.3 us, against
// 11,050 for the row-wise kernel; of its busy cycles the counters give 57 % to the MFMAs and
// 30 % to the VALU, 17 % of them with the LDS in use.
#pragma once

#include "common.hpp"

namespace taskops {
namespace kan_direct {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
constexpr int kCols = 16 * kWaves;     // output columns per workgroup, 16 per wave
constexpr int kMaxKnots = 32;
constexpr int kRawBufferFlags = 0x00020000;
constexpr unsigned kOutOfRange = 0x80000000u;
constexpr int kSystemScope = 17;  // buffer cache policy sc0 | sc1
typedef int i32x4 __attribute__((ext_vector_type(4)));

// Features per chunk: 16 kR rows x these features are the (row, feature) pairs the threads
// expand, one each (half the threads idle for kR = 1 with many bases, whose staged weights
// would not fit otherwise).
template <int kNQ, int kR>
constexpr int chunk_features() { return kR == 1 && kNQ > 4 ? 8 : 16 / kR; }

// Weight loads.  kR = 4 (flat false): each lane reads its own column's bases, which is how
// the MFMA wants them, but 64 lanes then touch 16 columns' lines four lanes at a time, 64 line
// accesses per load: hidden under 64 rows of MFMAs, it is what bounds a small batch (the
// loads alone took 13.6 of 16.4 us at B = 8, I = O = 1024).  kR < 4 (flat true): a wave's 16
// columns' runs of a chunk, kFeat C contiguous floats each, are read as consecutive 16-byte
// units, staged in the wave's own LDS and read back per lane.
template <int kR>
constexpr bool flat_loads() { return kR < 4; }

// Floats between two (feature, row) runs of 4 kNQ slots in LDS: an odd number of 16-byte
// units, so eight consecutive rows' 16-byte reads fall on different banks.
template <int kNQ>
constexpr int slot_stride() { return kNQ % 2 ? 4 * kNQ : 4 * kNQ + 4; }

// LDS, in floats: two stages of the expanded runs and of the silu plane, two of the knot
// rows, then (flat loads) each wave's 16 column runs of Ws, sc and Wb.  A column's runs are
// padded by one 16-byte unit, which spreads a step's reads over the banks.
template <int kNQ, int kR>
constexpr int pairs() { return 16 * kR * chunk_features<kNQ, kR>(); }
template <int kNQ, int kR>
constexpr int act_floats() { return pairs<kNQ, kR>() * slot_stride<kNQ>(); }
template <int kNQ, int kR>
constexpr int knots_at() { return 2 * (act_floats<kNQ, kR>() + pairs<kNQ, kR>()); }
template <int kNQ, int kR>
constexpr int weights_at() { return knots_at<kNQ, kR>() + 2 * chunk_features<kNQ, kR>() * kMaxKnots; }
__host__ __device__ constexpr int run_stride(int feats, int C) { return feats * C + 4; }
__host__ __device__ constexpr int wave_weight_floats(int feats, int C) {
  return 16 * (run_stride(feats, C) + 2 * run_stride(feats, 1));
}
template <int kNQ, int kR>
int lds_bytes(int C) {
  const int staged = flat_loads<kR>() ? kWaves * wave_weight_floats(chunk_features<kNQ, kR>(), C) : 0;
  return (weights_at<kNQ, kR>() + staged) * (int)sizeof(float);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, size_t bytes) {
  const int n = bytes > 0x7fffffffu ? 0x7fffffff : (int)bytes;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, n, kRawBufferFlags);
}

// 1 / d, one Newton step on v_rcp_f32: within an ulp, a third of an IEEE division's cost.
__device__ __forceinline__ float recip(float d) {
  const float r = __builtin_amdgcn_rcpf(d);
  return fmaf(fmaf(-d, r, 1.0f), r, r);
}

// The knot interval of x on the row kn[0..L): j with kn[j] <= x < kn[j + 1]; false when x lies
// outside [kn[0], kn[L - 1]) (or is NaN).  The guess from the first spacing is right for
// uniform rows up to rounding; if it fails for any lane, the wave counts knots <= x.
// kn is padded with +inf to a multiple of four.
__device__ __forceinline__ bool knot_interval(float x, const float* kn, int L, int& j) {
  const float t0 = kn[0];
  j = min(max((int)__builtin_floorf((x - t0) * recip(kn[1] - t0)), 0), L - 2);
  const bool inside = x >= t0 && x < kn[L - 1];
  const bool hit = x >= kn[j] && x < kn[j + 1];
  if (__builtin_amdgcn_ballot_w64(inside && !hit) != 0ull) {
    int cnt = 0;
    for (int q = 0; q < (L + 3) / 4; ++q) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(kn + 4 * q);
      cnt += (int)(x >= v.x) + (int)(x >= v.y) + (int)(x >= v.z) + (int)(x >= v.w);
    }
    j = min(max(cnt - 1, 0), L - 2);
  }
  return inside;
}

// The kOrder + 1 bases j - kOrder .. j on the knot interval j of the row kn[0..L), by the
// triangular scheme, written to their slots of the zeroed run.  Knots past the row's ends are
// replaced by the end knots; they only enter bases outside [0, C), which have no slot.
template <int kNQ, int kOrder>
__device__ __forceinline__ void write_bases(float x, const float* kn, int L, int C, int j, bool inside, float* run) {
  float t[2 * kOrder];  // knots j - kOrder + 1 .. j + kOrder
#pragma unroll
  for (int i = 0; i < 2 * kOrder; ++i) t[i] = kn[min(max(j - kOrder + 1 + i, 0), L - 1)];
  float N[kOrder + 1];
  N[0] = 1.0f;
#pragma unroll
  for (int p = 1; p <= kOrder; ++p) {
    float saved = 0.0f;
#pragma unroll
    for (int r = 0; r < p; ++r) {
      const float hi = t[kOrder + r], lo = t[kOrder - p + r];  // t_{j+1+r}, t_{j+1-p+r}
      const float q = N[r] * recip(hi - lo);
      N[r] = fmaf(hi - x, q, saved);
      saved = (x - lo) * q;
    }
    N[p] = saved;
  }
#pragma unroll
  for (int i = 0; i <= kOrder; ++i) {
    const int b = j - kOrder + i;
    if (inside && (unsigned)b < (unsigned)C) run[b < 4 * (kNQ - 1) ? b : b + 4 * kNQ - C] = N[i];
  }
}

// kNQ: 16-byte groups of a feature's C bases, 4 (kNQ - 1) < C <= 4 kNQ.  The last group is
// read at C - 4, inside the feature's own floats, so its first 4 kNQ - C ("dup") elements
// repeat the group before it: they have no slot and no MFMA.  kR: row blocks of 16.
// nsplit > 1: the features' sums are taken in nsplit parts and added in order.  partial: a tile
// of sums per (split, row tile, column tile), a workgroup per part; counters: null or one
// arrival counter per tile, zero between launches.  kAlone, for calls without that memory: a
// tile's one workgroup takes the parts one after another and keeps their sum in `out`, in the
// same order, so the same bits.  (The loop around the parts costs 27 registers and with them a
// quarter of the waves, so it is a form of its own.)
template <int kNQ, int kR, bool kAlone>
__global__ __launch_bounds__(kThreads) void kan_direct(
    const float* __restrict__ x, const float* __restrict__ grid, const float* __restrict__ wb,
    const float* __restrict__ ws, const float* __restrict__ sc, int order, int L, int C, int B, int I, int O,
    int mtiles, int ctiles, int nsplit, int cper, float* __restrict__ partial, unsigned* __restrict__ counters,
    float* __restrict__ out) {
  constexpr int kFeat = chunk_features<kNQ, kR>();
  constexpr int kPairs = pairs<kNQ, kR>(), kAct = act_floats<kNQ, kR>();
  constexpr bool kFlat = flat_loads<kR>();
  constexpr int kSteps = kFeat / 4;             // 4-feature steps per chunk
  constexpr int kRows = 16 * kR;
  constexpr int kS = slot_stride<kNQ>();
  constexpr int kKnotLoads = kFeat * kMaxKnots / kThreads > 0 ? kFeat * kMaxKnots / kThreads : 1;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  float* act = smem;                           // [2][feature][row][kS]
  float* act0 = smem + 2 * kAct;               // [2][feature][row]: silu
  float* knots = smem + knots_at<kNQ, kR>();   // [2][feature][kMaxKnots]

  // The row tiles of one (column tile, split) read the same weights: they go to one XCD
  // (workgroups are dispatched round-robin over 8) one after another, and share its L2.
  const int shares = kAlone ? 1 : nsplit;  // workgroups of one tile
  const int span = min(8, ctiles * shares), seq = (int)blockIdx.x / span;
  const int pair = seq / mtiles * span + (int)blockIdx.x % span, mt = seq % mtiles;
  if (pair >= ctiles * shares) return;
  const int ct = pair % ctiles;
  int split = pair / ctiles;
  const int m0 = mt * kRows, n0 = ct * kCols;
  const int nchunks = (I + kFeat - 1) / kFeat;
  int c0, c1;
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;

  // This lane's column and feature quarter of the MFMA operands.
  const int fr = lane % 16, fq = lane / 16;
  const int col = n0 + 16 * wave + fr;
  const int ncols = min(kCols, O - n0);
  const __amdgpu_buffer_rsrc_t rwb = make_rsrc(wb + (size_t)n0 * I, (size_t)ncols * I * 4);
  const __amdgpu_buffer_rsrc_t rsc = make_rsrc(sc + (size_t)n0 * I, (size_t)ncols * I * 4);
  const __amdgpu_buffer_rsrc_t rws = make_rsrc(ws + (size_t)n0 * I * C, (size_t)ncols * I * C * 4);
  const int dup = 4 * kNQ - C;

  // Raw weights on their way: per lane and step (direct), or the wave's units of a chunk
  // (flat).  They are reloaded for the next chunk as soon as their values have been used.
  constexpr int kUnits = kFlat ? kFeat * kNQ / 4 : 1;  // 16-byte units per lane, C = 4 kNQ
  f32x4 rw[kFlat ? 1 : kSteps][kNQ], ru[kUnits], rub, rus;
  float rb[kSteps], rs[kSteps];
  const unsigned crow = (unsigned)(col - n0) * (unsigned)I;
  auto load_step = [&](int c, int s) {
    const int f = c * kFeat + 4 * s + fq;
    const bool ok = c < c1 && f < I && col < O;
    const unsigned at = crow + (unsigned)f, o1 = ok ? at * 4u : kOutOfRange;
    rb[s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rwb, o1, 0, 0));
    rs[s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsc, o1, 0, 0));
    const unsigned w0 = at * (unsigned)C;
#pragma unroll
    for (int j = 0; j < kNQ; ++j) {
      const unsigned e = (j < kNQ - 1 ? w0 + 4u * j : w0 + (unsigned)(C - 4)) * 4u;
      rw[s][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rws, ok ? e : kOutOfRange, 0, 0));
    }
  };
  // Flat: unit u of the chunk's run of column k of this wave (kFeat C / 4 units; lanes take
  // consecutive units, column after column).
  float* wst = smem + weights_at<kNQ, kR>() + wave * wave_weight_floats(kFeat, C);  // [16][run] Ws, then sc, then Wb
  const int wrun = run_stride(kFeat, C);
  float* sst = wst + 16 * wrun;
  constexpr int kSrun = run_stride(kFeat, 1);
  float* bst = sst + 16 * kSrun;
  const int ucol = kFeat * C / 4;                   // units per column
  const unsigned umagic = (65536u + ucol - 1) / ucol;  // n / ucol = n * umagic >> 16 (n < 16 ucol <= 2048)
  const unsigned wcol0 = (unsigned)(16 * wave) * (unsigned)I;
  // Unit at float `at` of r, `left` floats of its run from there on.  No branch around the
  // loads (an offset past the buffer reads zero), so a chunk's are in flight together; cut: the
  // chunk's runs end inside a unit (the last chunk, I and C odd), whose floats are read singly.
  auto unit = [&](__amdgpu_buffer_rsrc_t r, bool live, unsigned at, int left, bool cut) {
    f32x4 v = __builtin_bit_cast(
        f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, live && left >= 4 ? at * 4u : kOutOfRange, 0, 0));
    if (cut) {
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        const float t = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                      r, live && left < 4 && e < left ? (at + e) * 4u : kOutOfRange, 0, 0));
        v[e] = left < 4 ? t : v[e];
      }
    }
    return v;
  };
  auto load_flat = [&](int c) {
    const int f0 = c * kFeat, nf = min(kFeat, I - f0);
    const bool wcut = ((nf * C) & 3) != 0;
#pragma unroll
    for (int i = 0; i < kUnits; ++i) {
      const int n = lane + kWave * i, k = (int)((unsigned)n * umagic >> 16), u = n - k * ucol;
      const bool live = c < c1 && n < 16 * ucol && n0 + 16 * wave + k < O;
      ru[i] = unit(rws, live, (wcol0 + (unsigned)k * (unsigned)I + (unsigned)f0) * (unsigned)C + 4u * u, nf * C - 4 * u, wcut);
    }
    constexpr int kQ = kFeat / 4;  // units of a column's sc and Wb
    const int k = lane / kQ, u = lane % kQ;
    const bool live = c < c1 && k < 16 && n0 + 16 * wave + k < O;
    const unsigned at = wcol0 + (unsigned)k * (unsigned)I + (unsigned)(f0 + 4 * u);
    rus = unit(rsc, live, at, nf - 4 * u, (nf & 3) != 0);
    rub = unit(rwb, live, at, nf - 4 * u, (nf & 3) != 0);
  };
  auto stage_flat = [&]() {
#pragma unroll
    for (int i = 0; i < kUnits; ++i) {
      const int n = lane + kWave * i, k = (int)((unsigned)n * umagic >> 16), u = n - k * ucol;
      if (n < 16 * ucol) *reinterpret_cast<f32x4*>(wst + k * wrun + 4 * u) = ru[i];
    }
    constexpr int kQ = kFeat / 4;
    const int k = lane / kQ, u = lane % kQ;
    if (k < 16) {
      *reinterpret_cast<f32x4*>(sst + k * kSrun + 4 * u) = rus;
      *reinterpret_cast<f32x4*>(bst + k * kSrun + 4 * u) = rub;
    }
  };

  // The (row, feature) pair this thread expands.
  const int er = tid % kRows, ef = tid / kRows;
  const int erow = m0 + er;
  const int nrows = min(kRows, B - m0);
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(x + (size_t)m0 * I, (size_t)nrows * I * 4);
  auto load_x = [&](int c) {
    const int f = c * kFeat + ef;
    const unsigned at = (unsigned)er * (unsigned)I + (unsigned)f;
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                         rx, (erow < B && f < I && c < c1) ? at * 4u : kOutOfRange, 0, 0));
  };
  // Knot k of feature f at knots[stage][f][k], +inf past L (a count of knots <= x then ends
  // at L); missing features' rows are never used.
  float kreg[kKnotLoads];
  auto load_knots = [&](int c) {
#pragma unroll
    for (int i = 0; i < kKnotLoads; ++i) {
      const int e = tid + i * kThreads, f = c * kFeat + e / kMaxKnots, k = e % kMaxKnots;
      kreg[i] = (e < kFeat * kMaxKnots && f < I && c < c1 && k < L) ? grid[(size_t)f * L + k] : __builtin_inff();
    }
  };
  auto write_knots = [&](int stage) {
#pragma unroll
    for (int i = 0; i < kKnotLoads; ++i) {
      const int e = tid + i * kThreads;
      if (e < kFeat * kMaxKnots) knots[stage * kFeat * kMaxKnots + e] = kreg[i];
    }
  };

  auto expand = [&](int c, float xv) {
    if (kPairs < kThreads && tid >= kPairs) return;
    const int stage = (c - c0) & 1;
    const float* kn = knots + (stage * kFeat + ef) * kMaxKnots;
    float* run = act + stage * kAct + (ef * kRows + er) * kS;
    const bool present = c * kFeat + ef < I;
    // An infinite x makes every basis of the recursion NaN (0 * inf), and so the row's sum:
    // the silu term carries that.
    const float s = __builtin_isinf(xv) ? __builtin_nanf("") : xv / (1.0f + expf(-xv));
    act0[stage * kPairs + ef * kRows + er] = present ? s : 0.0f;
#pragma unroll
    for (int q = 0; q < kNQ; ++q) *reinterpret_cast<f32x4*>(run + 4 * q) = f32x4{0.f, 0.f, 0.f, 0.f};
    int j;
    const bool inside = knot_interval(xv, kn, L, j) && present;
    switch (order) {
      case 1: write_bases<kNQ, 1>(xv, kn, L, C, j, inside, run); break;
      case 2: write_bases<kNQ, 2>(xv, kn, L, C, j, inside, run); break;
      case 3: write_bases<kNQ, 3>(xv, kn, L, C, j, inside, run); break;
      default: write_bases<kNQ, 4>(xv, kn, L, C, j, inside, run); break;
    }
  };

  f32x4 acc[kR];

  // Step s of chunk c: the lane's weights scaled into their own registers (direct: the raw
  // ones reload for chunk c + 1), then 1 + C MFMAs per row block.
  auto step = [&](int c, int s) {
    float w[4 * kNQ], w0;
    if constexpr (kFlat) {
      const int f = 4 * s + fq;
      const float* src = wst + fr * wrun + f * C;
      const float scale = sst[fr * kSrun + f];
      w0 = bst[fr * kSrun + f];
#pragma unroll
      for (int j = 0; j < 4 * kNQ; ++j)  // slot order: the last group starts at base C - 4
        w[j] = src[j < 4 * (kNQ - 1) ? j : j - dup] * scale;
    } else {
#pragma unroll
      for (int j = 0; j < kNQ; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) w[4 * j + e] = rw[s][j][e] * rs[s];
      w0 = rb[s];
      load_step(c + 1, s);
    }
    const int stage = (c - c0) & 1;
    const float* a = act + stage * kAct + ((4 * s + fq) * kRows + fr) * kS;
    const float* a0 = act0 + stage * kPairs + (4 * s + fq) * kRows + fr;
    f32x4 part[kR];
#pragma unroll
    for (int r = 0; r < kR; ++r)
      part[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[16 * r], w0, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
    for (int j = 0; j < kNQ; ++j) {
      f32x4 av[kR];
#pragma unroll
      for (int r = 0; r < kR; ++r) av[r] = *reinterpret_cast<const f32x4*>(a + 16 * r * kS + 4 * j);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (j == kNQ - 1 && e < dup) continue;  // uniform: this element repeats the group before
#pragma unroll
        for (int r = 0; r < kR; ++r)
          part[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[r][e], w[4 * j + e], part[r], 0, 0, 0);
      }
    }
#pragma unroll
    for (int r = 0; r < kR; ++r) acc[r] += part[r];
  };

  for (;;) {
    c0 = split * cper;
    c1 = min(nchunks, c0 + cper);
#pragma unroll
    for (int r = 0; r < kR; ++r) acc[r] = f32x4{0.f, 0.f, 0.f, 0.f};
    // The activations' loads go out before the weights', whose arrival nothing before the first
    // MFMA waits for (loads return in order).
    load_knots(c0);
    float xv = load_x(c0);
    const float x1 = load_x(c0 + 1);
    write_knots(0);
    load_knots(c0 + 1);
    if constexpr (kFlat) {
      load_flat(c0);
    } else {
#pragma unroll
      for (int s = 0; s < kSteps; ++s) load_step(c0, s);
    }
    barrier_no_vm_drain();
    expand(c0, xv);
    write_knots(1);
    xv = x1;
    load_knots(c0 + 2);
    for (int c = c0; c < c1; ++c) {
      // Chunk c's runs and chunk c + 1's knots are written; every wave is done with the stage
      // chunk c + 1 expands into and with chunk c's knots.
      barrier_no_vm_drain();
      if (c + 1 < c1) {
        expand(c + 1, xv);
        write_knots((c - c0) & 1);
        xv = load_x(c + 2);
        load_knots(c + 3);
      }
      if constexpr (kFlat) {  // the wave's own LDS: its reads of the last chunk came before
        wave_lds_fence();
        stage_flat();
        wave_lds_fence();
        load_flat(c + 1);
      }
#pragma unroll
      for (int s = 0; s < kSteps; ++s) step(c, s);
    }
    if constexpr (!kAlone) break;
    // This part's sum on top of the parts' before it.
    if (col < O) {
#pragma unroll
      for (int r = 0; r < kR; ++r)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = m0 + 16 * r + 4 * fq + e;
          float* at = out + (size_t)row * O + col;
          if (row < B) *at = (split > 0 ? *at : 0.f) + acc[r][e];
        }
    }
    if (++split == nsplit) return;
    __syncthreads();  // the stages are free
  }

  if (nsplit > 1) {
    // Every split stores its tile, 16 bytes per lane and row block.  Without counters
    // kan_direct_sum adds them.  With counters it then arrives on the tile's, and the last adds
    // the splits' tiles in split order, so the result does not depend on which one that is.
    // Its stores and loads are system-scope (sc0 sc1) and go through to the coherence point: a
    // store's completion (vmcnt) means that it got there, and the arrival follows every wave's
    // wait for that.  So no L2 needs writing back or invalidating: with
    // agent-scope fences, one per workgroup, the write-backs queued up (B = 64, I = O = 1024
    // 55 us; a second launch for the sums 27.0).
    constexpr int kTile = kRows * kCols;
    const int tile = mt * ctiles + ct;
    // Split by split, so that what the sum reads together lies together.
    const int stride = mtiles * ctiles * kTile * 4;
    const __amdgpu_buffer_rsrc_t rp =
        make_rsrc(partial + (size_t)tile * kTile, (size_t)(nsplit - 1) * stride + kTile * 4);
    unsigned at[kR];  // missing rows' sums go nowhere: past the descriptor
#pragma unroll
    for (int r = 0; r < kR; ++r)
      at[r] = m0 + 16 * r + 4 * fq < B ? (unsigned)(((wave * kR + r) * kWave + lane) * 16) : kOutOfRange;
    if (counters == nullptr) {
#pragma unroll
      for (int r = 0; r < kR; ++r)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(i32x4, acc[r]), rp, at[r], split * stride, 0);
      return;
    }
#pragma unroll
    for (int r = 0; r < kR; ++r)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(i32x4, acc[r]), rp, at[r], split * stride, kSystemScope);
    __builtin_amdgcn_s_waitcnt((0x7 << 4) | (0xF << 8));  // vmcnt(0): the stores are done
    __syncthreads();  // every wave's; the LDS is free
    unsigned* flag = reinterpret_cast<unsigned*>(smem);
    if (tid == 0) {
      const bool last =
          __hip_atomic_fetch_add(counters + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)nsplit - 1;
      if (last) __hip_atomic_store(counters + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *flag = last;
    }
    __syncthreads();
    if (!*flag) return;
    constexpr int kBatch = 16 / kR;  // splits whose loads are in flight together
#pragma unroll
    for (int r = 0; r < kR; ++r) acc[r] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < nsplit; s += kBatch) {
      f32x4 v[kBatch][kR];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        // Past the last split: the vector offset, the one the descriptor's bound is checked
        // against, lies past the buffer and the load returns zero.
        const bool live = s + u < nsplit;
#pragma unroll
        for (int r = 0; r < kR; ++r)
          v[u][r] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                  rp, live ? at[r] : kOutOfRange, live ? (s + u) * stride : 0, kSystemScope));
      }
#pragma unroll
      for (int u = 0; u < kBatch; ++u)
#pragma unroll
        for (int r = 0; r < kR; ++r) acc[r] += v[u][r];
    }
  }
  if (col < O) {
#pragma unroll
    for (int r = 0; r < kR; ++r)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = m0 + 16 * r + 4 * fq + e;
        if (row < B) out[(size_t)row * O + col] = acc[r][e];
      }
  }
}

// The sums without counters: thread per element of a tile, as kan_direct stored it, the
// splits added in the same order.  4 * kR workgroups per tile.
constexpr int kSumBatch = 16;
template <int kR>
__global__ __launch_bounds__(kThreads) void kan_direct_sum(const float* __restrict__ partial, int B, int O, int mtiles,
                                                           int ctiles, int nsplit, float* __restrict__ out) {
  constexpr int kTile = 16 * kR * kCols;
  const int tile = (int)blockIdx.x / (4 * kR), at = (int)blockIdx.x % (4 * kR) * kThreads + (int)threadIdx.x;
  const int lane = at / 4 % kWave, r = at / 4 / kWave % kR, wave = at / 4 / kWave / kR;
  const int col = tile % ctiles * kCols + 16 * wave + lane % 16;
  const int row = tile / ctiles * 16 * kR + 16 * r + 4 * (lane / 16) + at % 4;
  if (col >= O || row >= B) return;
  const size_t stride = (size_t)mtiles * ctiles * kTile;
  const float* from = partial + (size_t)tile * kTile + at;
  float t = 0.f;
  for (int s = 0; s < nsplit; s += kSumBatch) {  // a batch of loads in flight, added in order
    float v[kSumBatch];
#pragma unroll
    for (int u = 0; u < kSumBatch; ++u) v[u] = s + u < nsplit ? from[(s + u) * stride] : 0.f;
#pragma unroll
    for (int u = 0; u < kSumBatch; ++u) t += v[u];
  }
  out[(size_t)row * O + col] = t;
}

}  // namespace kan_direct
}  // namespace taskops
