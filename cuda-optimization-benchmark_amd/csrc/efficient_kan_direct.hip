// Host side of efficient_kan's direct fp32 path (efficient_kan_direct.hpp).
#include <hip/hip_ext.h>

#include <algorithm>
#include <optional>

#include "efficient_kan_direct.hpp"

namespace taskops {
namespace {

using namespace kan_direct;

// Row blocks of 16 per workgroup: as few as hold the batch, so small batches do no MFMAs
// for missing rows, up to 4, which read each weight once per 64 rows.
int row_blocks(int B) { return B <= 16 ? 1 : (B <= 32 ? 2 : 4); }

// Up to this many splits the tile's last arrival adds them; it reads them all by itself, so
// beyond that a second launch, spread over the chip, is faster although it costs 2 to 4 us: us
// with one launch / two at 2 splits (B = 70, I = 5, O = 30, G = 7) 6.7 / 8.6, 6 (B = 1024, I = 256,
// O = 512, G = 16) 66.3 / 71.6, 10 (B = 1, I = 77, O = 301, G = 23) 12.9 / 13.5, 26 (B = 6, I = 208, O = 448,
// G = 20) 11.1 / 10.4, 42 (B = 20, I = 333, O = 131, G = 10) 12.1 / 11.5.
constexpr int kMaxArrivals = 16;

// A call's launch: workgroups the chip holds at once, at most four per CU: the features are
// split until the grid has that many, in one round.  At 1, 2 and 4 per CU B = 8, I = O = 1024 took
// 19.7, 17.5 and 17.5 us (its LDS allows two); B = 4096, I = 256, O = 512 took 200 us at 3 and 178 at
// 4.  nsplit splits of at most cper chunks each, none empty.
struct Plan {
  size_t lds;
  int mtiles, ctiles, nchunks, per_cu, nsplit, cper, features;
  void split(int n) {
    cper = (nchunks + n - 1) / n;
    nsplit = (nchunks + cper - 1) / cper;
  }
};

template <int kNQ, int kR>
Plan make_plan(int C, int B, int I, int O) {
  Plan p;
  p.features = chunk_features<kNQ, kR>();
  p.mtiles = (B + 16 * kR - 1) / (16 * kR);
  p.ctiles = (O + kCols - 1) / kCols;
  p.nchunks = (I + p.features - 1) / p.features;
  p.lds = (size_t)lds_bytes<kNQ, kR>(C);
  p.per_cu = std::max(1, std::min<int>(4, (int)(device_lds_per_cu() / p.lds)));
  const int64_t want = (int64_t)p.per_cu * device_cu_count() / ((int64_t)p.mtiles * p.ctiles);
  p.split((int)std::min<int64_t>(p.nchunks, std::max<int64_t>(want, 1)));
  return p;
}

template <int kNQ, int kR>
hipError_t launch(const float* x, const float* grid, const float* wb, const float* ws, const float* sc, int order,
                  int L, int C, int B, int I, int O, float* out, size_t shared_bytes, hipStream_t stream) {
  Plan plan = make_plan<kNQ, kR>(C, B, I, O);
  const int mtiles = plan.mtiles, ctiles = plan.ctiles;
  const int64_t tiles = (int64_t)mtiles * ctiles;
  const size_t per_split = (size_t)tiles * 16 * kR * kCols * sizeof(float);
  const int nsplit = plan.nsplit;
  unsigned* counters = nullptr;
  float* partial = nullptr;
  std::optional<StreamScratch> scratch;
  if (shared_bytes > 0) {
    void* p = nullptr;
    size_t have = 0;
    const hipError_t e = workspace_if_possible(kSlotKan, std::max(shared_bytes, nsplit * per_split), stream, &p, &have);
    if (e != hipSuccess) return e;
    if (have >= nsplit * per_split) partial = static_cast<float*>(p);
  } else if (nsplit > 1) {
    scratch.emplace(nsplit * per_split, stream);
    counters = scratch->counters;
    partial = static_cast<float*>(scratch->ptr);
  }
  const int shares = partial != nullptr ? nsplit : 1;  // workgroups of one tile
  if (shares > kMaxArrivals || tiles > kScratchCounters) counters = nullptr;
  const int64_t pairs = (int64_t)ctiles * shares, span = std::min<int64_t>(8, pairs), padded = (pairs + span - 1) / span * span;
  auto enqueue = [&](bool last, auto kernel, dim3 groups, size_t lds, auto... args) {
    const hipEvent_t done = last && scratch && scratch->ptr != nullptr ? scratch->done : nullptr;
    if (done != nullptr)
      hipExtLaunchKernelGGL(kernel, groups, dim3(kThreads), (unsigned)lds, stream, nullptr, done, 0, args...);
    else
      hipLaunchKernelGGL(kernel, groups, dim3(kThreads), lds, stream, args...);
    const hipError_t e = hipGetLastError();
    if (done != nullptr && e == hipSuccess) scratch->ended();
    return e;
  };
  const bool one = shares == 1 || counters != nullptr;
  auto kernel = shares < nsplit ? kan_direct::kan_direct<kNQ, kR, true> : kan_direct::kan_direct<kNQ, kR, false>;
  const hipError_t e = enqueue(one, kernel, dim3((unsigned)(padded * mtiles)), plan.lds, x, grid, wb, ws, sc, order, L, C, B,
                               I, O, mtiles, ctiles, nsplit, plan.cper, partial, counters, out);
  if (e != hipSuccess || one) return e;
  return enqueue(true, kan_direct_sum<kR>, dim3((unsigned)(tiles * 4 * kR)), (size_t)0,
                 static_cast<const float*>(partial), B, O, mtiles, ctiles, nsplit, out);
}

template <int kNQ>
hipError_t launch_rows(const float* x, const float* grid, const float* wb, const float* ws, const float* sc, int order,
                       int L, int C, int B, int I, int O, float* out, size_t shared_bytes, hipStream_t stream) {
  switch (row_blocks(B)) {
    case 1: return launch<kNQ, 1>(x, grid, wb, ws, sc, order, L, C, B, I, O, out, shared_bytes, stream);
    case 2: return launch<kNQ, 2>(x, grid, wb, ws, sc, order, L, C, B, I, O, out, shared_bytes, stream);
    default: return launch<kNQ, 4>(x, grid, wb, ws, sc, order, L, C, B, I, O, out, shared_bytes, stream);
  }
}

}  // namespace

// Orders 1 .. 4 (the triangular scheme's instantiations), four or more bases (a feature's
// bases are read 16 bytes at a time), 32-bit offsets for one workgroup's rows and columns,
// and a grid one launch covers (2^32 - 1 work-items; the split never takes the grid past
// four workgroups per CU).
bool kan_direct_fits(int order, int C, int B, int I, int O) {
  const int64_t lim = 0x7fffffff;
  if (order < 1 || order > 4 || C < 4 || I < 1) return false;
  if ((int64_t)kCols * I * C * 4 > lim || (int64_t)64 * I * 4 > lim) return false;
  const int rows = 16 * row_blocks(B);
  const int64_t tiles = (((int64_t)O + kCols - 1) / kCols + 7) / 8 * 8 * (((int64_t)B + rows - 1) / rows);
  return tiles <= (int64_t)0xffffffff / kThreads;
}

namespace {
template <int kNQ>
Plan plan_rows(int C, int B, int I, int O) {
  switch (row_blocks(B)) {
    case 1: return make_plan<kNQ, 1>(C, B, I, O);
    case 2: return make_plan<kNQ, 2>(C, B, I, O);
    default: return make_plan<kNQ, 4>(C, B, I, O);
  }
}
}  // namespace

// About how long a call takes, in us, for the choice between the two paths (C at most 12 there):
// each CU's share of (16-row block, feature) pairs, padding of the tiles and splits included, at
// 27 ns for the expansion and 4 ns a term.  Within 10% of 80% of 370 measured calls of 15 to 100 us.
double kan_direct_us(int C, int B, int I, int O) {
  const Plan p = C <= 4 ? plan_rows<1>(C, B, I, O) : (C <= 8 ? plan_rows<2>(C, B, I, O) : plan_rows<3>(C, B, I, O));
  const double pairs = (double)p.mtiles * p.ctiles * p.nsplit * p.cper * p.features * row_blocks(B) / device_cu_count();
  return 14.3 + pairs * (0.027 + 0.004 * (1 + C));
}

// shared_bytes: 0 for calls with no workspace of their own (the splits' sums then go to the
// stream's scratch memory); else the size to which the shared workspace is grown, which holds
// them.  Where there is no room a tile's one workgroup takes all splits, with the same bits.  The arrival counters are the scratch memory's
// alone: two streams' calls at once could leave shared ones wrong for every later call.
hipError_t kan_direct_launch(const float* x, const float* grid, const float* wb, const float* ws, const float* sc,
                             int order, int L, int C, int B, int I, int O, float* out, size_t shared_bytes,
                             hipStream_t stream) {
#define TASKOPS_KAN_NQ(q) \
  case q: return launch_rows<q>(x, grid, wb, ws, sc, order, L, C, B, I, O, out, shared_bytes, stream)
  switch ((C + 3) / 4) {
    TASKOPS_KAN_NQ(1);
    TASKOPS_KAN_NQ(2);
    TASKOPS_KAN_NQ(3);
    TASKOPS_KAN_NQ(4);
    TASKOPS_KAN_NQ(5);
    TASKOPS_KAN_NQ(6);
    TASKOPS_KAN_NQ(7);
    TASKOPS_KAN_NQ(8);
    default: return hipErrorInvalidValue;
  }
#undef TASKOPS_KAN_NQ
}

}  // namespace taskops
