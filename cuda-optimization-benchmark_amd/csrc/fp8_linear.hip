// fp8_linear on gfx950: output = bf16((x/sx) @ (w/sw)^T + bias), OCP e4m3 inputs.
//
// Drop-in signature tasks/fp8_linear/tests/task.json:3, replacing
// reference/fp8_linear/solution.cu:276-321.  Kernels are in fp8_linear.hpp (skinny, wide and its
// 128-row form) and fp8_linear_mid.hpp (64 to 128-row tiles, any K and alignment); the rules
// below choose.
#include "fp8_linear.hpp"

using namespace taskops;
using namespace taskops::fp8;

namespace {

// True when every 32-bit buffer offset of the kernels fits: a workgroup addresses its
// operand rows (at most 256 rows of K bytes above M = 64; all M rows of x and 16 of w in
// the skinny kernels) and, above M = 64, its output rows (at most 256 rows of N bf16
// values) through descriptors of at most 2^31 - 1 bytes.  The skinny grid (16 columns per
// workgroup of kSkinnyThreads) also stays within one launch's 2^32 - 1 work-items; above
// M = 64 the offsets bound N, which keeps that grid far inside it.
bool offsets_fit(int64_t M, int64_t K, int64_t N) {
  const int64_t lim = 0x7fffffff;
  if (M <= kSkinnyMaxM)
    return M * K <= lim && 16 * K <= lim && (N + 15) / 16 * kSkinnyThreads <= (int64_t)0xffffffff;
  return (int64_t)BM * K <= lim && (int64_t)BM * N * 2 <= lim;
}

// The middle kernel's tile for a call, or -1 for the skinny and wide kernels.
//
// M > 64: the smallest tile that gives each CU at most one workgroup, since the work of one
// step is bound by its own LDS traffic and smaller tiles only spread it: us at 64x64 / 64x128 /
// 128x128 / 128x256: M = 256, K = N = 4096 (256 tiles of 64x64) 9.2 / 13.5 / 16.8 / 24.0, M =
// 512 14.7 / 14.0 / 17.1 / 24.0, M = 1024 27 / 26 / 19.0 / 24.3, M = 2048 51 / 51 / 36.9 / 29.8,
// and from there on the wide kernel's forms.  Where they do not apply (K % 16, alignment),
// 128x128 tiles take the rest.
//
// M <= 64: the skinny kernel gives 16 columns to a workgroup and splits K over its waves; a tile
// has four times the columns and walks K alone.  With more than one skinny workgroup per CU the
// skinny kernel's time doubles and the tiles win; below that it depends on K.  us, skinny / tiles,
// weights in the Infinity Cache and (in brackets) from memory:
//  * 17 rows up, more than 16 columns per CU: M = 32, K = 4096, N = 5120 12.8 / 8.3 (13.2 / 11.9),
//    M = 64 16.0 / 8.6 (16.6 / 12.9).  Up to 16 rows from N = 7168 on: M = 16, K = 1024, N = 8192 7.6 /
//    4.1 (7.8 / 5.6), K = 4096 10.1 / 8.3 (10.3 / 11.3), K = 7168 15.9 / 11.8 (16.0 / 17.6), but K =
//    14336 28.2 / 30.5 (28.3 / 30.5): half the CUs hold a tile and do not draw the memory's rate.
//  * 33 to 48 rows at fewer columns: the skinny kernel's waves take 2048 of K a pass, so just beyond
//    one pass the tiles win: M = 43, K = 2176, N = 1632 6.4 / 5.3 (10.1 / 6.3), M = 33, K = 3072, N = 1024
//    7.7 / 6.2 (9.3 / 7.3), K = 4096 7.6 / 7.2 (9.8 / 8.6); at K = 2048 5.1 / 5.1 (5.4 / 6.0), 4.3 / 5.1
//    with the weights in the L2s, and at N = 64, K = 4096 5.7 / 7.0.  Longer K from memory is too much for
//    the few CUs that hold a tile: M = 39, K = 5536, N = 1568 (14.3 / 18.1), M = 48, K = 10352, N =
//    1216 (26.6 / 36.6), although from the Infinity Cache the tiles would be faster.
//  * 33 to 48 rows and short K: M = 42, K = 256, N = 1024 4.1 / 3.3 (4.7 / 3.3), M = 48, K = 768, N = 2048
//    4.9 / 3.8 (5.0 / 4.4), K = 1280 5.1 / 4.4 (5.9 / 5.2); at K = 1536 5.2 / 4.6 (6.1 / 5.5) but 4.8 / 4.7 at
//    N = 3360 and, with the weights in the L2s, 4.1 / 4.6; N = 512: K = 768 3.8 / 3.8, K = 1024 3.8 / 4.0.
//  * 49 rows up at fewer columns: M = 64, K = 1024, N = 512 3.5 / 4.1, K = 2048, N = 4096 5.5 / 5.2 (6.0 /
//    8.0), K = 7168, N = 1024 13.4 / 11.9 (13.7 / 19.3): the skinny kernel.
//  * 33 rows up at less than two columns per CU, where the skinny kernel has few workgroups as well,
//    and K past 4096: M = 54, K = 8000, N = 176 14.9 / 11.3, M = 64, K = 7168, N = 64 12.1 / 10.1.
// With 8-byte rows both move less per load: M = 33, K = 4088, N = 4104 16.6 / 13.8 (18.1 / 18.5), K =
// 1016 4.8 / 5.6 (4.9 / 5.8), N = 8200 6.1 / 5.7 (7.2 / 7.2); M = 64, K = 1016, N = 4104 6.2 / 5.6 (6.2 /
// 6.0).  Other K have no 8-byte loads for the skinny kernel: M = 16, K = 1001, N = 1024 12.3 / 6.1.
int mid_tile(int64_t M, int64_t K, int64_t N, int vec) {
  const int64_t cus = device_cu_count();
  if (M <= kSkinnyMaxM) {
    if (vec == 16 && 64 * K > (int64_t)0x7fffffff) return -1;  // a tile's rows in 32-bit offsets
    const int rb = (int)(M + 15) / 16;
    const bool wide = N > 16 * cus;  // more than one skinny workgroup per CU
    bool tiles = vec == 1;
    if (vec == 16) {
      if (rb == 1) tiles = N >= 28 * cus && (K <= 8192 || N > 32 * cus);
      else if (rb == 2) tiles = N >= 20 * cus;
      else if (rb == 3 && K <= 2048) tiles = wide || K <= 640 || (K <= 1280 && N >= 4 * cus);
      else tiles = wide || (K > 4096 ? N < 2 * cus : rb == 3 && N >= 2 * cus);
    } else if (vec == 8) {
      tiles = wide && (rb == 4 || (rb == 3 && (K > 2048 || N >= 32 * cus)));
    }
    return tiles ? kTile64x64 : -1;
  }
  auto tiles = [&](int rows, int cols) { return ((M + rows - 1) / rows) * ((N + cols - 1) / cols); };
  if (tiles(64, 64) <= cus) return kTile64x64;
  if (tiles(64, 128) <= cus) return kTile64x128;
  if (vec != 16 || tiles(128, 128) <= cus) return kTile128x128;
  return -1;
}

}  // namespace

extern "C" hipError_t taskops_fp8_linear(int32_t M, int32_t K, int32_t N, const uint8_t* x_fp8,
                                         float scale_x, const uint8_t* w_fp8, float scale_w,
                                         const uint16_t* bias, uint16_t* output,
                                         hipStream_t stream) {
  if (M < 0 || K < 0 || N < 0) return hipErrorInvalidValue;
  if (M == 0 || N == 0) return hipSuccess;
  if (!offsets_fit(M, K, N)) return hipErrorInvalidValue;
  const float inv = (float)(1.0 / ((double)scale_x * (double)scale_w));
  const int vec = vec_width(x_fp8, w_fp8, K);
  const int mid = mid_tile(M, K, N, vec);
  if (mid >= 0)
    return mid_launch(static_cast<MidTile>(mid), vec == 16, x_fp8, w_fp8, (int)M, (int)N, (int)K, inv, bias, output,
                      stream);
  if (M <= kSkinnyMaxM) {
    const dim3 grid((N + 15) / 16);
    if (vec == 16) {
      // Flat loads through LDS; M decides the row blocks (and so the K slice per pass).
      switch ((M + 15) / 16) {
        case 1:
          hipLaunchKernelGGL(fp8_gemm_skinny_flat<1>, grid, dim3(kSkinnyThreads), skinny_lds_bytes(1), stream,
                             x_fp8, w_fp8, (int)M, (int)N, (int)K, inv, bias, output);
          break;
        case 2:
          hipLaunchKernelGGL(fp8_gemm_skinny_flat<2>, grid, dim3(kSkinnyThreads), skinny_lds_bytes(2), stream,
                             x_fp8, w_fp8, (int)M, (int)N, (int)K, inv, bias, output);
          break;
        case 3:
          hipLaunchKernelGGL(fp8_gemm_skinny_flat<3>, grid, dim3(kSkinnyThreads), skinny_lds_bytes(3), stream,
                             x_fp8, w_fp8, (int)M, (int)N, (int)K, inv, bias, output);
          break;
        default:
          hipLaunchKernelGGL(fp8_gemm_skinny_flat<4>, grid, dim3(kSkinnyThreads), skinny_lds_bytes(4), stream,
                             x_fp8, w_fp8, (int)M, (int)N, (int)K, inv, bias, output);
          break;
      }
    } else
      hipLaunchKernelGGL(fp8_gemm_skinny, grid, dim3(kSkinnyThreads), 0, stream, x_fp8, w_fp8, (int)M, (int)N, (int)K,
                         inv, bias, output);
    return hipGetLastError();
  }
  const int tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
  const size_t wide_lds = kWideLdsBytes;
  const uintptr_t o = reinterpret_cast<uintptr_t>(output);
  if (2 * tiles <= device_cu_count()) {
    // At most half a 256x256 tile per CU: 128x256 tiles, twice as many workgroups.
    const dim3 hgrid(((M + kHalfRows - 1) / kHalfRows) * ((N + BN - 1) / BN));
    const size_t half_lds = kHalfLaunchLdsBytes;
    if (N % 8 == 0 && (o & 15) == 0)
      hipLaunchKernelGGL(fp8_gemm_half<2>, hgrid, dim3(kThreads), half_lds, stream, x_fp8, w_fp8, (int)M,
                         (int)N, (int)K, inv, bias, output);
    else if (N % 4 == 0 && (o & 7) == 0)
      hipLaunchKernelGGL(fp8_gemm_half<1>, hgrid, dim3(kThreads), half_lds, stream, x_fp8, w_fp8, (int)M,
                         (int)N, (int)K, inv, bias, output);
    else
      hipLaunchKernelGGL(fp8_gemm_half<0>, hgrid, dim3(kThreads), half_lds, stream, x_fp8, w_fp8, (int)M,
                         (int)N, (int)K, inv, bias, output);
    return hipGetLastError();
  }
  // K % 128 == 0: copies without per-lane bounds tests (copy_offset; the 128x256 form
  // measured no faster with them dropped).
  if (N % 8 == 0 && (o & 15) == 0 && K % WBK == 0)
    hipLaunchKernelGGL((fp8_gemm_wide<2, true>), dim3(tiles), dim3(kThreads), wide_lds, stream, x_fp8, w_fp8,
                       (int)M, (int)N, (int)K, inv, bias, output);
  else if (N % 8 == 0 && (o & 15) == 0)
    hipLaunchKernelGGL(fp8_gemm_wide<2>, dim3(tiles), dim3(kThreads), wide_lds, stream, x_fp8, w_fp8,
                       (int)M, (int)N, (int)K, inv, bias, output);
  else if (N % 4 == 0 && (o & 7) == 0)
    hipLaunchKernelGGL(fp8_gemm_wide<1>, dim3(tiles), dim3(kThreads), wide_lds, stream, x_fp8, w_fp8,
                       (int)M, (int)N, (int)K, inv, bias, output);
  else
    hipLaunchKernelGGL(fp8_gemm_wide<0>, dim3(tiles), dim3(kThreads), wide_lds, stream, x_fp8, w_fp8,
                       (int)M, (int)N, (int)K, inv, bias, output);
  return hipGetLastError();
}
