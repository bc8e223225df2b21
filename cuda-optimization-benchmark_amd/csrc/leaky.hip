// leaky on gfx950: leaky integrate-and-fire layer (snnTorch Leaky, reset by subtraction).
//
// Drop-in signature tasks/leaky/tests/task.json:3, replacing
// reference/leaky/solution.cu:106-138.  The kernels are in leaky.hpp: leaky_kernel for layers
// that fill the chip with neuron pairs, leaky_rows_kernel for small and odd ones.
#include "leaky.hpp"

namespace taskops {
namespace {
constexpr int kThreads = 256;
constexpr int kDepth = 16;
constexpr bool kNonTemporal = true;

// The four-step kernel's launch: waves per workgroup and ring blocks by how many waves the
// neurons make.  Up to one wave per CU, single waves that look 64 steps ahead; then fewer
// steps and wider workgroups, whose waves read adjacent 256 bytes.  us at <1, 16> / <2, 12> /
// <4, 6>: N = 4096, T = 512 14.7 / 17.5 / 21.9; N = 17000, T = 160 9.9 / 9.1 / 12.2; N = 64000, T =
// 160 17.4 / 16.9 / 15.7; N = 180180 (odd H), T = 100 47.3 / 43.9 / 38.1.
template <int kWaves, int kRing>
hipError_t launch_rows(const float* x, const float* mem0, const float* beta, const float* th, int T, int N, int H,
                       float* spikes, float* final_mem, hipStream_t stream) {
  const unsigned per = kWaves * kWave;
  hipLaunchKernelGGL((leaky_rows_kernel<kWaves, kRing>), dim3(((unsigned)N + per - 1) / per), dim3(per), 0, stream, x,
                     mem0, beta, th, T, N, H, spikes, final_mem);
  return hipGetLastError();
}
}  // namespace
}  // namespace taskops

using namespace taskops;

extern "C" hipError_t taskops_leaky(const float* input_current, const float* mem0,
                                    const float* beta, const float* threshold, int32_t T,
                                    int32_t B, int32_t H, float* spikes, float* final_mem,
                                    hipStream_t stream) {
  if (T < 0 || B < 0 || H < 0) return hipErrorInvalidValue;
  const int64_t N = (int64_t)B * H;
  if (N == 0) return hipSuccess;
  const uintptr_t bits = reinterpret_cast<uintptr_t>(input_current) |
                         reinterpret_cast<uintptr_t>(spikes);
  int vec = 1;
  if (H % 2 == 0 && (bits & 7) == 0) vec = 2;
  // Neuron pairs (leaky_kernel) need even H, aligned rows and enough neurons to fill the chip:
  // at 262,144 they are the faster (90.0 against 98 us, T = 256), at 163,840 30.2 against 26.3,
  // at 17,000 22.2 against 9.1.  Odd H gains at every size (T = 310, N = 67,768 170 against 50,
  // T = 60, N = 800,400 96 against 78).  The four-step kernel addresses a block's rows, up to
  // three past T, in 31 bits, and a wave needs 64 neurons.
  const int64_t cus = device_cu_count(), waves = (N + kWave - 1) / kWave;
  if (T > 0 && N >= kWave && ((int64_t)T + 4) * N * 4 <= 0x7fffffff && (vec == 1 || waves <= 12 * cus)) {
    auto launch = waves <= cus ? launch_rows<1, 16> : (waves <= 2 * cus ? launch_rows<2, 12> : launch_rows<4, 6>);
    return launch(input_current, mem0, beta, threshold, (int)T, (int)N, (int)H, spikes, final_mem, stream);
  }
  const int64_t threads = N / vec;
  // One launch covers at most 2^32 - 1 work-items: B*H up to 2^32 - 256 neurons on either path.
  if (N > (int64_t(1) << 32) - kThreads) return hipErrorInvalidValue;
  const unsigned blocks = (unsigned)((threads + kThreads - 1) / kThreads);
  if (vec == 2)
    hipLaunchKernelGGL((leaky_kernel<kThreads, 2, kDepth, kNonTemporal>), dim3(blocks), dim3(kThreads), 0,
                       stream, input_current, mem0, beta, threshold, (int)T, N, (int)H, spikes, final_mem);
  else
    hipLaunchKernelGGL((leaky_kernel<kThreads, 1, kDepth, kNonTemporal>), dim3(blocks), dim3(kThreads), 0,
                       stream, input_current, mem0, beta, threshold, (int)T, N, (int)H, spikes, final_mem);
  return hipGetLastError();
}
