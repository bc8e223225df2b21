// fp8_linear's middle kernel (fp8_linear_mid.hip): output tiles of 64 x 64, 64 x 128 and 128 x
// 128, for calls whose 128 x 256 tiles would leave most CUs idle, and for any K and alignment.
//
// 8 waves on a (64 kXI) x (64 kWJ) tile, K in steps of 128: waves 0-3 take the first 64 k of
// every step and waves 4-7 the second, each four a 2 x 2 arrangement of (32 kXI) x (32 kWJ)
// wave tiles of 32x32x64 MFMAs (W is the A operand, as in the wide kernel).  Two waves per
// SIMD cover each other's waits; the halves' sums are added once at the end, through LDS.
//
// kDirect (K % 16 == 0, operands 16-byte aligned): direct-to-LDS copies into a ring of kStages
// steps, kStages - 1 of them in flight, and each step's fragments read during the step
// before's MFMAs (read in their own step, M = 512, K = N = 4096 took 17.9 us instead of 14.0).
// Otherwise 16-byte loads at any alignment into registers two steps ahead and from there into
// two LDS stages; the row's last 16 bytes are loaded from K - 16 on and shifted, so no load
// leaves the operand.
//
// Bound: no unit by itself.  At M = 512, K = N = 4096 (64 x 128 tiles, one workgroup per CU) the
// counters read the MFMAs busy 28 % of a CU's cycles, the LDS 24 % (2 % of that bank
// conflicts) and the VALU 31 %: what is left is a step's chain of loads, barrier and LDS reads,
// and the launch.  Measured (us, against the 128 x 256 form): M = 512, K = N = 4096 14.0 / 24.0, M = 256 9.3 / 24.0, M =
// 1024 19.0 / 24.3; K = 8192, N = 1024, M = 512 13.8 / 41.1.  Against the register-staged 256 x
// 256 kernel that took other K: M = 333, K = 1000, N = 3000 7.0 / 34.9, M = 1000, K = N = 1001
// 6.7 / 138, M = 4096, K = 4088, N = 4096 97 / 103.
#pragma once

#include "fp8_linear.hpp"

namespace taskops {
namespace fp8 {
namespace mid {

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / kWave;
typedef i32x4 __attribute__((aligned(1))) i32x4u;

template <int kXI, int kWJ>
struct Shape {
  static constexpr int kRows = 64 * kXI, kCols = 64 * kWJ;     // output tile
  static constexpr int kStageBytes = (kRows + kCols) * WBK;     // x rows, then w rows
  static constexpr int kCopies = kXI + kWJ;                     // 1 KiB copies (8 rows) per wave and step
  static constexpr int kChunks = (kRows + kCols) * 8 / kThreads;  // 16-byte loads per thread
  static constexpr int kSumBytes = kRows * kCols * 4;           // waves 4-7's sums
  static constexpr int kTileBytes = kRows * kCols * 2;          // the bf16 tile
  static_assert(kCopies * kWaves * 1024 == kStageBytes, "every wave's copies make a stage");
  // The ring or stages (reused by the sums and the tile), then the bias.
  static constexpr int bias_at(int stages) {
    return stages * kStageBytes > kSumBytes + kTileBytes ? stages * kStageBytes : kSumBytes + kTileBytes;
  }
  static constexpr int lds_bytes(int stages) { return bias_at(stages) + kCols * 4; }
};

// Bytes shift .. 15 of v moved down to 0, zeros above (shift uniform, 1 .. 15).
__device__ __forceinline__ i32x4 shift_down(i32x4 v, int shift) {
  const int d = shift / 4;
  const unsigned b = (unsigned)shift % 4;
  const int w0 = d == 0 ? v.x : d == 1 ? v.y : d == 2 ? v.z : v.w, w1 = d == 0 ? v.y : d == 1 ? v.z : d == 2 ? v.w : 0,
            w2 = d == 0 ? v.z : d == 1 ? v.w : 0, w3 = d == 0 ? v.w : 0;
  return i32x4{(int)__builtin_amdgcn_alignbyte(w1, w0, b), (int)__builtin_amdgcn_alignbyte(w2, w1, b),
               (int)__builtin_amdgcn_alignbyte(w3, w2, b), (int)__builtin_amdgcn_alignbyte(0, w3, b)};
}

// kStore: 2 = 16-byte row stores (N % 8 == 0, out 16-byte aligned); 0 = one 2-byte store per
// value.
template <int kXI, int kWJ, int kStages, bool kDirect, int kStore>
__global__ __launch_bounds__(kThreads) void fp8_gemm_mid(
    const uint8_t* __restrict__ x, const uint8_t* __restrict__ w, int M, int N, int K, float inv_scale,
    const uint16_t* __restrict__ bias, uint16_t* __restrict__ out) {
  using S = Shape<kXI, kWJ>;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tm = (M + S::kRows - 1) / S::kRows, tn = (N + S::kCols - 1) / S::kCols;
  int mt, nt;
  tile_of(blockIdx.x, tm, tn, mt, nt);
  const int m0 = mt * S::kRows, n0 = nt * S::kCols;
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int half = wave / 4, wm = wave % 4 / 2, wn = wave % 2;
  const int rows_a = min(S::kRows, M - m0), rows_b = min(S::kCols, N - n0);
  const int fr = lane % 32, fg = lane / 32;
  const int arow = wm * 32 * kXI + fr, brow = S::kRows + wn * 32 * kWJ + fr;  // rows of a stage
  const int nk = (K + WBK - 1) / WBK;

  f32x16 acc[kXI][kWJ];
#pragma unroll
  for (int i = 0; i < kXI; ++i)
#pragma unroll
    for (int j = 0; j < kWJ; ++j) acc[i][j] = f32x16{};

  float* bias_s = reinterpret_cast<float*>(smem + S::bias_at(kDirect ? kStages : 2));
  const __amdgpu_buffer_rsrc_t rbias = make_rsrc(bias + n0, (size_t)rows_b * 2);
  float bias_v = 0.0f;
  if (tid < S::kCols)
    bias_v = bf16_to_f32(__builtin_amdgcn_raw_buffer_load_b16(rbias, tid < rows_b ? (unsigned)tid * 2u : kOutOfRange, 0, 0));

  // A step's fragments of this wave's half, read during the step before's MFMAs.
  struct Frags {
    i32x8 a[kXI], b[kWJ];
  };
  auto read = [&](const uint8_t* stage, Frags& f) {
#pragma unroll
    for (int j = 0; j < kWJ; ++j) f.b[j] = frag128(stage, brow + 32 * j, fg, half);
#pragma unroll
    for (int i = 0; i < kXI; ++i) f.a[i] = frag128(stage, arow + 32 * i, fg, half);
  };
  auto multiply = [&](const Frags& f) {
#pragma unroll
    for (int i = 0; i < kXI; ++i)
#pragma unroll
      for (int j = 0; j < kWJ; ++j) acc[i][j] = mfma32_e4m3(f.b[j], f.a[i], acc[i][j]);
  };
  Frags f0, f1;

  if constexpr (kDirect) {
    const __amdgpu_buffer_rsrc_t xa = make_rsrc(x + (size_t)m0 * K, (size_t)rows_a * K);
    const __amdgpu_buffer_rsrc_t wb = make_rsrc(w + (size_t)n0 * K, (size_t)rows_b * K);
    // This wave's copies of a step, kXI of x and kWJ of w, 8 rows each.  A step past K zero-fills its slot
    // without touching memory.
    auto copy = [&](int step) {
      uint8_t* stage = smem + (step % kStages) * S::kStageBytes;
#pragma unroll
      for (int c = 0; c < kXI; ++c) dma_group128<false>(xa, stage, rows_a, K, step * WBK, wave * kXI + c, lane);
#pragma unroll
      for (int c = 0; c < kWJ; ++c)
        dma_group128<false>(wb, stage + S::kRows * WBK, rows_b, K, step * WBK, wave * kWJ + c, lane);
    };
#pragma unroll
    for (int s = 0; s < kStages; ++s) copy(s);
    wait_vmcnt<(kStages - 1) * S::kCopies>();
    barrier_no_vm_drain();
    read(smem, f0);
    auto step = [&](int kt, const Frags& cur, Frags& nxt) {
      // This wave's copies of step kt + 1 have landed; past the barrier everyone's have, and
      // everyone holds step kt in registers, so its slot takes step kt + kStages.
      wait_vmcnt<(kStages - 2) * S::kCopies>();
      barrier_no_vm_drain();
      read(smem + (kt + 1) % kStages * S::kStageBytes, nxt);
      copy(kt + kStages);
      multiply(cur);
    };
    for (int kt = 0; kt < nk; kt += 2) {
      step(kt, f0, f1);
      if (kt + 1 < nk) step(kt + 1, f1, f0);
    }
    wait_vmcnt<0>();
  } else {
    // Chunk i of this thread: 16 bytes at k = 16 chunk of stage row 64 i + tid / 8 (rows past
    // the operand repeat its last row; their products are never stored).
    const int chunk = tid % 8;
    const uint8_t* src[S::kChunks];
    uint8_t* dst[S::kChunks];
#pragma unroll
    for (int i = 0; i < S::kChunks; ++i) {
      const int r = 64 * i + tid / 8;
      src[i] = (64 * i < S::kRows ? x + (size_t)(m0 + min(r, rows_a - 1)) * K
                                  : w + (size_t)(n0 + min(r - S::kRows, rows_b - 1)) * K) +
               16 * chunk;
      const int rr = 64 * i < S::kRows ? r : r - S::kRows;
      dst[i] = smem + r * WBK + ((chunk ^ swz128(rr)) << 4);
    }
    auto load = [&](int step, i32x4 (&v)[S::kChunks]) {
      const int left = K - step * WBK - 16 * chunk;  // bytes of the row from this chunk on
      if (K < 16) {                                  // uniform: the row byte by byte
#pragma unroll
        for (int i = 0; i < S::kChunks; ++i) {
          v[i] = i32x4{0, 0, 0, 0};
          for (int e = 0; e < left; ++e) v[i][e / 4] |= (int)((unsigned)src[i][e] << (8 * (e % 4)));
        }
      } else if ((step + 1) * WBK <= K) {  // uniform
#pragma unroll
        for (int i = 0; i < S::kChunks; ++i) v[i] = *reinterpret_cast<const i32x4u*>(src[i] + step * WBK);
      } else {
        const int at = left >= 16 ? step * WBK : K - 16 - 16 * chunk;
#pragma unroll
        for (int i = 0; i < S::kChunks; ++i) {
          i32x4 t = *reinterpret_cast<const i32x4u*>(src[i] + at);
          if (left < 16) t = left > 0 ? shift_down(t, 16 - K % 16) : i32x4{0, 0, 0, 0};
          v[i] = t;
        }
      }
    };
    auto write = [&](int stage, const i32x4 (&v)[S::kChunks]) {
#pragma unroll
      for (int i = 0; i < S::kChunks; ++i) *reinterpret_cast<i32x4*>(dst[i] + stage * S::kStageBytes) = v[i];
    };
    i32x4 v0[S::kChunks], v1[S::kChunks];
    load(0, v0);
    if (nk > 1) load(1, v1);
    // Stage kt % 2 is rewritten two steps on, past a barrier that follows its last read.  The
    // fragments are read in their own step.  Read a step ahead, M = 2000, K = 1000, N = 3000 took 21.6
    // us instead of 17.4; its 128 x 128 tiles fit one workgroup per CU either way (98,816 bytes of
    // LDS), so the cause is another one, which was not found.
    for (int kt = 0; kt < nk; kt += 2) {
      write(0, v0);
      if (kt + 2 < nk) load(kt + 2, v0);
      barrier_no_vm_drain();
      read(smem, f0);
      multiply(f0);
      if (kt + 1 < nk) {
        write(1, v1);
        if (kt + 3 < nk) load(kt + 3, v1);
        barrier_no_vm_drain();
        read(smem + S::kStageBytes, f0);
        multiply(f0);
      }
    }
  }
  if (tid < S::kCols) bias_s[tid] = bias_v;
  __syncthreads();  // every copy has landed and every fragment is read: the ring is free

  // Waves 4-7 hand their sums to waves 0-3 (same tile position), 16 KiB per register block.
  f32x4* sums = reinterpret_cast<f32x4*>(smem);
  const int sat = (wm * 2 + wn) * (kXI * kWJ * 4);
  if (half == 1) {
#pragma unroll
    for (int i = 0; i < kXI; ++i)
#pragma unroll
      for (int j = 0; j < kWJ; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          sums[(sat + (i * kWJ + j) * 4 + q) * kWave + lane] =
              f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
  }
  __syncthreads();
  // Tile row r's 16-byte chunk c at chunk c ^ (r % 8): a wave writes 32 rows' 8 bytes at a time.
  uint8_t* tile = smem + S::kSumBytes;
  constexpr int kRowBytes = S::kCols * 2;
  if (half == 0) {
#pragma unroll
    for (int j = 0; j < kWJ; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int c = wn * 32 * kWJ + j * 32 + 8 * q + 4 * fg;  // first of four columns
        const f32x4 bv = *reinterpret_cast<const f32x4*>(bias_s + c);
#pragma unroll
        for (int i = 0; i < kXI; ++i) {
          const f32x4 other = sums[(sat + (i * kWJ + j) * 4 + q) * kWave + lane];
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = fmaf(acc[i][j][4 * q + e] + other[e], inv_scale, bv[e]);
          const int r = wm * 32 * kXI + i * 32 + fr;
          *reinterpret_cast<i32x2*>(tile + r * kRowBytes + (((c / 8) ^ (r % 8)) << 4) + 8 * ((c / 4) & 1)) =
              i32x2{(int)pack_bf16x2(v[0], v[1]), (int)pack_bf16x2(v[2], v[3])};
        }
      }
  }
  __syncthreads();
  if constexpr (kStore == 2) {  // 128 rows of N values within 32-bit offsets (the launch checks)
    const __amdgpu_buffer_rsrc_t ob = make_rsrc(out + (size_t)m0 * N, (size_t)rows_a * N * 2);
    constexpr int kRowChunks = kRowBytes / 16;
#pragma unroll
    for (int s = 0; s < S::kRows * kRowChunks / kThreads; ++s) {
      const int e = tid + s * kThreads, r = e / kRowChunks, c = e % kRowChunks;
      const i32x4 v = *reinterpret_cast<const i32x4*>(tile + r * kRowBytes + ((c ^ (r % 8)) << 4));
      const unsigned off = (r < rows_a && c * 8 < rows_b) ? (unsigned)(r * N + n0 + c * 8) * 2u : kOutOfRange;
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(__attribute__((ext_vector_type(4))) unsigned, v), ob,
                                             off, 0, 0);
    }
  } else {
    uint16_t* dst = out + (size_t)m0 * N + n0;
#pragma unroll 4
    for (int s = 0; s < S::kRows * S::kCols / kThreads; ++s) {
      const int e = tid + s * kThreads, r = e / S::kCols, c = e % S::kCols;
      const uint16_t v = *reinterpret_cast<const uint16_t*>(tile + r * kRowBytes + (((c / 8) ^ (r % 8)) << 4) + 2 * (c % 8));
      if (r < rows_a && c < rows_b) dst[(size_t)r * N + c] = v;
    }
  }
}

}  // namespace mid
}  // namespace fp8
}  // namespace taskops
