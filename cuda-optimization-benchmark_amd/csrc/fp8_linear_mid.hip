// Launches of fp8_linear's middle kernel (fp8_linear_mid.hpp).
#include <algorithm>

#include "fp8_linear_mid.hpp"

namespace taskops {
namespace fp8 {
namespace {

using mid::Shape;

template <int kXI, int kWJ, int kStages, bool kDirect>
hipError_t launch(const uint8_t* x, const uint8_t* w, int M, int N, int K, float inv, const uint16_t* bias,
                  uint16_t* out, hipStream_t stream) {
  using S = Shape<kXI, kWJ>;
  const bool rows16 = N % 8 == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0 && (int64_t)S::kRows * N * 2 <= 0x7fffffff;
  auto kernel = rows16 ? mid::fp8_gemm_mid<kXI, kWJ, kStages, kDirect, 2> : mid::fp8_gemm_mid<kXI, kWJ, kStages, kDirect, 0>;
  // A launch covers at most 2^32 - 1 work-items: whole rows of tiles at a time.
  const int64_t tn = (N + S::kCols - 1) / S::kCols, most = (int64_t)0xffffffff / mid::kThreads / tn * S::kRows;
  for (int64_t m0 = 0; m0 < M; m0 += most) {
    const int rows = (int)std::min<int64_t>(most, M - m0);
    const unsigned tiles = (unsigned)((rows + (int64_t)S::kRows - 1) / S::kRows * tn);
    hipLaunchKernelGGL(kernel, dim3(tiles), dim3(mid::kThreads), S::lds_bytes(kDirect ? kStages : 2), stream,
                       x + m0 * K, w, rows, N, K, inv, bias, out + m0 * N);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

template <int kXI, int kWJ, int kStages>
hipError_t launch_any(bool direct, const uint8_t* x, const uint8_t* w, int M, int N, int K, float inv,
                      const uint16_t* bias, uint16_t* out, hipStream_t stream) {
  if (direct) return launch<kXI, kWJ, kStages, true>(x, w, M, N, K, inv, bias, out, stream);
  return launch<kXI, kWJ, kStages, false>(x, w, M, N, K, inv, bias, out, stream);
}

}  // namespace

// Ring depths: 64 x 64 tiles in four steps (two workgroups fit a CU), the larger ones as many
// as one CU's LDS holds; 8 steps for 64 x 64 measured slower with two workgroups per CU (M = 512,
// K = N = 4096 16.8 against 14.7 us).  Up to 32 rows with one workgroup per CU and a long K, where
// the weights are the stream, 8 steps keep twice the bytes in flight: from memory M = 16, K = 4096,
// N = 8192 12.6 -> 11.3 us, K = 7168 19.1 -> 17.6, the same from the Infinity Cache; K = 1024 4.1 ->
// 4.7 there, and the same at 64 rows, so shorter K and more rows keep four.
hipError_t mid_launch(MidTile tile, bool direct, const uint8_t* x, const uint8_t* w, int M, int N, int K, float inv,
                      const uint16_t* bias, uint16_t* out, hipStream_t stream) {
  switch (tile) {
    case kTile64x64:
      if (direct && M <= 32 && K >= 4096 && (N + 63) / 64 <= device_cu_count())
        return launch<1, 1, 8, true>(x, w, M, N, K, inv, bias, out, stream);
      return launch_any<1, 1, 4>(direct, x, w, M, N, K, inv, bias, out, stream);
    case kTile64x128: return launch_any<1, 2, 6>(direct, x, w, M, N, K, inv, bias, out, stream);
    default: return launch_any<2, 2, 4>(direct, x, w, M, N, K, inv, bias, out, stream);
  }
}

}  // namespace fp8
}  // namespace taskops
