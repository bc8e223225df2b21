// Host runtime of libtaskops: per-device cached workspaces and device facts.
#include <mutex>
#include <vector>

#include "common.hpp"

namespace taskops {

struct StreamRegion {
  hipStream_t stream = nullptr;
  void* ptr = nullptr;
  size_t bytes = 0;
  hipEvent_t event = nullptr;
  bool ended = false;  // the last use has its event
  uint64_t used = 0;   // g_scratch_uses at the last use
};

namespace {

constexpr int kMaxDevices = 64;

struct Region {
  void* ptr = nullptr;
  size_t bytes = 0;
};

std::mutex g_mu;
std::mutex g_scratch_mu;
StreamRegion g_scratch[kMaxDevices][kMaxScratchStreams];
uint64_t g_scratch_uses = 0;
Region g_regions[kMaxDevices][kNumSlots];
// Buffers replaced by a larger one stay allocated until exit: a kernel enqueued before
// the replacement may still be using them, and freeing would need a host sync.
std::vector<void*> g_retired;
int g_cus[kMaxDevices] = {0};
int g_lds_per_cu[kMaxDevices] = {0};

// Zero fill as a kernel rather than hipMemsetAsync: no library call enqueues memset work,
// which keeps memset nodes out of any graph a caller captures.
__global__ void zero_fill(uint4* p, size_t n16) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (size_t)gridDim.x * blockDim.x)
    p[i] = uint4{0u, 0u, 0u, 0u};
}

}  // namespace

namespace {

// The current device, when `stream` (NULL = the default stream) belongs to it.  The workspace
// is the current device's; kernels run on the stream's device.  A stream of another device is
// refused rather than handed memory it cannot use.
hipError_t stream_device(hipStream_t stream, int* dev) {
  hipError_t e = hipGetDevice(dev);
  if (e != hipSuccess) return e;
  if (*dev < 0 || *dev >= kMaxDevices) return hipErrorInvalidDevice;
  if (stream != nullptr) {
    hipDevice_t sdev = 0;
    e = hipStreamGetDevice(stream, &sdev);
    if (e != hipSuccess) return e;
    if (sdev != *dev) return hipErrorInvalidValue;
  }
  return hipSuccess;
}

// While this lives, the calling thread's HIP calls do not count against a capture that another
// stream is making: in the default, global capture mode an allocation on any thread is refused
// and that capture invalidated.  For allocations whose own stream is not capturing.
struct RelaxedCapture {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  const bool on = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
  ~RelaxedCapture() {
    if (on) (void)hipThreadExchangeStreamCaptureMode(&mode);
  }
};

// Makes region r at least `bytes` large (g_mu held).
hipError_t grow(Region& r, size_t bytes, hipStream_t stream) {
  const size_t want = ((bytes < 4096 ? 4096 : bytes) + 15) / 16 * 16;
  void* p = nullptr;
  hipError_t e = hipMalloc(&p, want);
  if (e != hipSuccess) return e;
  const size_t n16 = want / 16;
  const unsigned blocks = (unsigned)(n16 / 256 < 4096 ? (n16 + 255) / 256 : 4096);
  hipLaunchKernelGGL(zero_fill, dim3(blocks), dim3(256), 0, stream, static_cast<uint4*>(p), n16);
  e = hipGetLastError();
  if (e != hipSuccess) {
    (void)hipFree(p);
    return e;
  }
  if (r.ptr) g_retired.push_back(r.ptr);
  r.ptr = p;
  r.bytes = want;
  return hipSuccess;
}

}  // namespace

hipError_t workspace(WorkspaceSlot slot, size_t bytes, hipStream_t stream, void** out) {
  int dev = 0;
  hipError_t e = stream_device(stream, &dev);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lock(g_mu);
  Region& r = g_regions[dev][slot];
  if (r.bytes < bytes) {
    e = grow(r, bytes, stream);
    if (e != hipSuccess) return e;
  }
  *out = r.ptr;
  return hipSuccess;
}

hipError_t workspace_if_possible(WorkspaceSlot slot, size_t bytes, hipStream_t stream, void** out, size_t* have) {
  int dev = 0;
  hipError_t e = stream_device(stream, &dev);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lock(g_mu);
  Region& r = g_regions[dev][slot];
  if (r.bytes < bytes) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    // The default stream cannot capture; asking about it while another stream captures is an
    // error, and then nothing may be allocated either.
    e = hipStreamIsCapturing(stream, &status);
    if (e != hipSuccess) (void)hipGetLastError();
    if (e == hipSuccess && status == hipStreamCaptureStatusNone) {
      const RelaxedCapture relaxed;
      e = grow(r, bytes, stream);
      if (e != hipSuccess) return e;
    }
  }
  *out = r.ptr;
  *have = r.bytes;
  return hipSuccess;
}

namespace {

// The region of `stream`: its own, an unused one, or the least recently used one whose last use
// is known to have completed; null when there is none (g_scratch_mu held).
StreamRegion* region_for(hipStream_t stream, int dev) {
  for (StreamRegion& s : g_scratch[dev])
    if (s.ptr != nullptr && s.stream == stream) return &s;
  for (StreamRegion& s : g_scratch[dev])
    if (s.ptr == nullptr) return &s;
  StreamRegion* r = nullptr;
  const RelaxedCapture relaxed;
  for (StreamRegion& s : g_scratch[dev]) {
    if (!s.ended || (r != nullptr && s.used > r->used)) continue;
    if (hipEventQuery(s.event) == hipSuccess) r = &s;
    else (void)hipGetLastError();
  }
  return r;
}

}  // namespace

StreamScratch::StreamScratch(size_t bytes, hipStream_t stream) {
  constexpr size_t kHead = kScratchCounters * sizeof(unsigned);
  int dev = 0;
  if (bytes > kMaxScratchBytes - kHead || stream == hipStreamPerThread || stream_device(stream, &dev) != hipSuccess) return;
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &status) != hipSuccess) {
    (void)hipGetLastError();
    return;
  }
  if (status != hipStreamCaptureStatusNone) return;
  lock_ = std::unique_lock<std::mutex>(g_scratch_mu);
  StreamRegion* r = region_for(stream, dev);
  if (r == nullptr) return;
  if (r->bytes < kHead + bytes) {
    size_t want = r->bytes > 0 ? 2 * r->bytes : (size_t)1 << 18;
    while (want < kHead + bytes) want *= 2;
    void* p = nullptr;
    const RelaxedCapture relaxed;
    if ((r->event == nullptr && hipEventCreateWithFlags(&r->event, hipEventDisableTiming) != hipSuccess) ||
        hipMalloc(&p, want) != hipSuccess) {
      (void)hipGetLastError();
      return;
    }
    hipLaunchKernelGGL(zero_fill, dim3(1), dim3(256), 0, stream, static_cast<uint4*>(p), kHead / 16);
    if (hipGetLastError() != hipSuccess) {
      (void)hipFree(p);
      return;
    }
    if (r->ptr != nullptr) {
      std::lock_guard<std::mutex> retire(g_mu);
      g_retired.push_back(r->ptr);
    }
    r->ptr = p;
    r->bytes = want;
  }
  r->stream = stream;
  r->used = ++g_scratch_uses;
  r->ended = false;
  for (const StreamRegion& s : g_scratch[dev])
    if (s.ptr != nullptr && &s != r) done = r->event;
  region_ = r;
  counters = static_cast<unsigned*>(r->ptr);
  ptr = static_cast<char*>(r->ptr) + kHead;
}

void StreamScratch::ended() { region_->ended = done != nullptr; }

int device_cu_count() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 256;
  int n = __atomic_load_n(&g_cus[dev], __ATOMIC_RELAXED);
  if (n > 0) return n;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
    n = 256;
  __atomic_store_n(&g_cus[dev], n, __ATOMIC_RELAXED);
  return n;
}

int device_lds_per_cu() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 160 * 1024;
  int n = __atomic_load_n(&g_lds_per_cu[dev], __ATOMIC_RELAXED);
  if (n > 0) return n;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev) != hipSuccess || n <= 0)
    n = 160 * 1024;
  __atomic_store_n(&g_lds_per_cu[dev], n, __ATOMIC_RELAXED);
  return n;
}

}  // namespace taskops

extern "C" int taskops_version(void) { return 1; }
