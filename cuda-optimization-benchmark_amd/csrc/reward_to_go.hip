// reward_to_go on gfx950: batched discounted reward-to-go with done flags.
//
// Drop-in signature tasks/reward_to_go/tests/task.json:3, replacing
// reference/reward_to_go/solution.cu:237-264.  The kernel is in reward_to_go.hpp.  Launch
// shape, measured on MI355X at B = T = 4096 (cold, µs per call): one workgroup per row;
// lanes own 4 steps, so every load and store instruction of a wave covers 1 KiB of
// contiguous memory; 4 waves of 4 chunks each cover 4096 steps, a BASELINE row in one
// segment; loads and stores are non-temporal.  That is 27.4 us against 30.5 us for 8 waves
// of one 8-step-per-lane chunk (whose 16-byte accesses cover every other 16 bytes per
// instruction, and which slows to 39 us with non-temporal stores).  Shorter rows use fewer
// waves and chunks per wave, so no wave idles.
#include <algorithm>
#include <cmath>

#include "reward_to_go.hpp"

namespace taskops {
namespace {

constexpr int kPerLane = 4;
// Cache policies (kNT of the kernel): aligned rows, non-temporal loads (bit 0) and stores
// (policy 2 in bits 1-2).  Unaligned rows share the lines at their ends with the next load, so
// theirs are ordinary loads: B = 4096, T = 4095 31.3 us against 34.0 with non-temporal ones
// (39.4 with ordinary stores too; 65.1 element by element, which such rows took before).
template <RtgAccess kAccess>
constexpr int policy() { return kAccess == kUnaligned ? 4 : 5; }

// Rows of 4 waves x 4 chunks (T > 2048) run with at most this many workgroups per CU,
// held there by the LDS each one reserves (the kernel's own LDS is a few bytes).  At the
// kernel's 68 VGPRs the registers allow 7; 4 measured fastest at B = T = 4096 (25.53
// against 25.76 us per call, 5 and 6 slower, 3 slower still) and at B = 3000 (20.15 against
// 20.63 us), and the same at B = 8192 and 1024 (one MI355X, cold rotating inputs).
constexpr int kLongRowWorkgroupsPerCU = 4;

// Dynamic LDS that lets at most `per_cu` workgroups share a CU: more than 1/(per_cu+1) of it.
size_t occupancy_lds(int per_cu) { return (size_t)device_lds_per_cu() / (per_cu + 1) + 1; }

// One workgroup per row, and one launch covers at most 2^32 - 1 work-items in a dimension,
// so rows go out in launches of at most kRowsPerLaunch (one launch for every B up to it).
constexpr int kRowsPerLaunch = 1 << 23;

template <int kWaves, int kSeg, RtgAccess kAccess>
void launch(const float* reward, const uint8_t* done, double g, int B, int T, float* out, hipStream_t stream) {
  const size_t lds = (kWaves == 4 && kSeg == 4) ? occupancy_lds(kLongRowWorkgroupsPerCU) : 0;
  for (int b0 = 0; b0 < B; b0 += kRowsPerLaunch) {
    const int nb = B - b0 < kRowsPerLaunch ? B - b0 : kRowsPerLaunch;
    const size_t off = (size_t)b0 * (size_t)T;  // T % 4 == 0 on the aligned path: alignment kept
    hipLaunchKernelGGL((reward_to_go_kernel<kWaves, kPerLane, kSeg, kAccess, policy<kAccess>()>), dim3(nb),
                       dim3(kWaves * kWave), lds, stream, reward + off, done + off, g, nb, T, out + off, RtgArgs<kWhole>{});
  }
}

// Few long rows.  A workgroup walks its row one segment of 4096 steps after another, about 2.2
// us each, so such rows are split into parts over workgroups: one launch composes each part's
// map, a second scans each part from the maps after it, reading the rewards again (from the
// caches).  Whole row against split, us per call: 16 x 65536 33-39 / 7.4, 1 x 131072 71 / 6.5,
// 6 x 18592 12.4 / 5.8, 33 x 109969 75-140 / 13.4, 128 x 131072 82.7 / 39.5, 256 x 65536 46.2 / 38.7, 1 x
// 1048576 600 / 12.9, 256 x 1048576 689 / 691.
// Rows of at most 12288 steps (three segments) or more than 256 of them keep the whole-row
// form: 1 x 8000 5.7 / 8.0, 229 x 9751 11.5 / 11.6, 256 x 16384 13.3 / 13.3, 512 x 8192 9.5 / 13.3.
constexpr int kSplitMaxRows = 256, kSplitMinChunks = 48;
// Chunks in all up to which parts have 4 chunks and 8, one and two per wave; beyond, four per wave
// in 16 or more: at 4, 8 and 16 16 x 65536 7.8, 7.4 and 8.4 us, 64 x 16384 7.7, 7.3 and 8.4, 8 x 65536
// 6.6, 6.7 and 8.1, 4 x 65536 6.0 and 6.5.  More parts would not find room for their maps either.
constexpr int kPart4Chunks = 1024, kPart8Chunks = 4096;
static_assert(kPart4Chunks / 4 <= 4 * kRtgMapsPerChunk && kPart8Chunks / 8 <= 8 * kRtgMapsPerChunk, "room for the maps");
// Chunks per part of a call in parts of 16 or more: more where a part's outputs have no room for
// the maps after it (rows past 4.2 M steps), and beyond what fills the chip where the maps'
// copies, one to each earlier part, add up: 8 x 2097152 71.6 us in 512 parts a row, 46.4 in 256.
int long_part(int B, int nchunks) {
  const int64_t nseg = ((int64_t)nchunks + 15) / 16;
  int64_t m = std::max<int64_t>((nseg + 16 * kRtgMapsPerChunk - 1) / (16 * kRtgMapsPerChunk), B * nseg / 4096);
  for (m = std::max<int64_t>(m, 1);; ++m) {
    const int64_t n = (nseg + m - 1) / m;  // parts of a row
    if (B * n <= 1024 || (B * n <= 4096 && n <= 128 * m)) return (int)(16 * m);
  }
}

// The factor of two composed maps.  Where it is too small for a double it stays the smallest one,
// not zero: only a done step makes a factor zero, and 0 * inf would turn the infinity that an
// infinite reward sends up its row into NaN.
double rtg_factor(double a, double b) {
  const double p = a * b;
  return p == 0.0 && a != 0.0 && b != 0.0 ? 0x1p-1074 : p;
}

template <int kSeg, RtgAccess kAccess>
hipError_t launch_split(const float* reward, const uint8_t* done, double g, int B, int T, float* out, int nparts,
                        int cpart, hipStream_t stream) {
  constexpr int kWaves = 4;
  double gpart = 1.0, power = g;  // g^(256 cpart)
  for (int e = kWave * kPerLane * cpart; e > 0; e >>= 1, power = rtg_factor(power, power))
    if (e & 1) gpart = rtg_factor(gpart, power);
  // Ordinary loads in the first pass, so that the second finds the rewards in the caches.
  hipLaunchKernelGGL((reward_to_go_kernel<kWaves, kPerLane, kSeg, kAccess, 0, kMaps>), dim3(B * nparts),
                     dim3(kWaves * kWave), 0, stream, reward, done, g, B, T, out, RtgArgs<kMaps>{nparts, cpart});
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((reward_to_go_kernel<kWaves, kPerLane, kSeg, kAccess, policy<kAccess>(), kApply>), dim3(B * nparts),
                     dim3(kWaves * kWave), 0, stream, reward, done, g, B, T, out, RtgArgs<kApply>{nparts, cpart, gpart});
  return hipGetLastError();
}

// Whether a call's output shares memory with an input (each workgroup reads its rewards before
// it writes there, so the whole-row form allows that; the maps of split rows do not).
bool overlaps(const float* reward, const uint8_t* done, int B, int T, const float* out) {
  const uintptr_t n = (uintptr_t)B * (uintptr_t)T, o = reinterpret_cast<uintptr_t>(out);
  auto with = [&](uintptr_t p, uintptr_t bytes) { return p < o + 4 * n && o < p + bytes; };
  return with(reinterpret_cast<uintptr_t>(reward), 4 * n) || with(reinterpret_cast<uintptr_t>(done), n);
}

template <RtgAccess kAccess>
hipError_t run(const float* reward, const uint8_t* done, double g, int B, int T, float* out, hipStream_t stream) {
  const int nchunks = (int)(((int64_t)T + kWave * kPerLane - 1) / (kWave * kPerLane));  // chunks of 256 steps
  if constexpr (kAccess != kElements) {
    // |g| <= 1: a part's a = g^steps cannot overflow (inf * 0 would make the carry NaN).
    if (B <= kSplitMaxRows && nchunks > kSplitMinChunks && std::fabs(g) <= 1.0) {
      const int64_t all = (int64_t)B * nchunks;
      const int cpart = all <= kPart4Chunks ? 4 : (all <= kPart8Chunks ? 8 : long_part(B, nchunks));
      const int nparts = (nchunks + cpart - 1) / cpart;
      if (!overlaps(reward, done, B, T, out)) {
        auto split = cpart == 4 ? launch_split<1, kAccess> : (cpart == 8 ? launch_split<2, kAccess> : launch_split<4, kAccess>);
        return split(reward, done, g, B, T, out, nparts, cpart, stream);
      }
    }
  }
  if (nchunks <= 1)
    launch<1, 1, kAccess>(reward, done, g, B, T, out, stream);
  else if (nchunks <= 2)
    launch<2, 1, kAccess>(reward, done, g, B, T, out, stream);
  else if (nchunks <= 4)
    launch<4, 1, kAccess>(reward, done, g, B, T, out, stream);
  else if (nchunks <= 8)
    launch<4, 2, kAccess>(reward, done, g, B, T, out, stream);
  else
    launch<4, 4, kAccess>(reward, done, g, B, T, out, stream);
  return hipGetLastError();
}

}  // namespace
}  // namespace taskops

using namespace taskops;

extern "C" hipError_t taskops_reward_to_go(const float* reward, const bool* done, float gamma,
                                           int32_t B, int32_t T, float* output,
                                           hipStream_t stream) {
  if (B <= 0 || T <= 0) return hipSuccess;  // nothing to write
  const uint8_t* d = reinterpret_cast<const uint8_t*>(done);
  const double g = (double)gamma;
  // The 16-byte paths' buffer stores address a row in 32-bit bytes (store_row16).
  if (T >= (1 << 30)) return run<kElements>(reward, d, g, B, T, output, stream);
  const bool aligned = (T % 4) == 0 &&
                       ((reinterpret_cast<uintptr_t>(reward) | reinterpret_cast<uintptr_t>(output)) & 15) == 0 &&
                       (reinterpret_cast<uintptr_t>(d) & 3) == 0;
  if (aligned) return run<kAligned>(reward, d, g, B, T, output, stream);
  return run<kUnaligned>(reward, d, g, B, T, output, stream);
}
