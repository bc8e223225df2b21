/* A HIP runtime for tests of the host side on a machine without a GPU: it runs no kernel,
 * records what the library asks for, and answers as one MI355X would (256 CUs, 160 KiB of LDS
 * each).  tests/test_host_paths.py builds it with gcc and loads it with RTLD_GLOBAL before
 * libtaskops.so, whose hip* calls then bind to it.
 *
 * Kernels go by their mangled device name, which __hipRegisterFunction gives for each host
 * stub; that call is forwarded to nothing, so no code object is loaded.  Device memory is
 * calloc'd.  Streams are small integers cast to hipStream_t.
 */
#define _GNU_SOURCE
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <hip/hip_runtime_api.h>

/* ---- what the test sets ---- */
static int s_capturing[64];      /* by stream handle */
static int s_global_capture;     /* another stream captures in global mode: see unsafe() */
static int s_malloc_fails;
static int s_busy[64];           /* by stream handle: events on it have not completed */

void stub_set_capturing(int stream, int on) { s_capturing[stream] = on; }
void stub_set_global_capture(int on) { s_global_capture = on; }
void stub_set_malloc_fails(int on) { s_malloc_fails = on; }
void stub_set_busy(int stream, int on) { s_busy[stream] = on; }

/* ---- the record: one line per call of interest ---- */
static char* g_log;
static size_t g_len, g_cap;
#define NOTE(...)                                                   \
  do {                                                              \
    char line_[512];                                                \
    int n_ = snprintf(line_, sizeof line_, __VA_ARGS__);            \
    if (n_ >= (int)sizeof line_) n_ = sizeof line_ - 1;             \
    if (g_len + n_ + 2 > g_cap) g_log = realloc(g_log, g_cap = 2 * g_cap + 4096); \
    memcpy(g_log + g_len, line_, n_);                               \
    g_len += n_;                                                    \
    g_log[g_len++] = '\n';                                          \
    g_log[g_len] = 0;                                               \
  } while (0)
const char* stub_log(void) { return g_log ? g_log : ""; }
void stub_clear(void) { g_len = 0; if (g_log) g_log[0] = 0; }

/* ---- code objects ---- */
static struct { const void* host; const char* name; } g_fn[1024];
static int g_nfn;
void** __hipRegisterFatBinary(const void* data) { (void)data; static void* h; return &h; }
void __hipUnregisterFatBinary(void** m) { (void)m; }
void __hipRegisterFunction(void** m, const void* host, char* dev, const char* name, unsigned limit, void* a, void* b,
                           void* c, void* d, int* w) {
  (void)m; (void)dev; (void)limit; (void)a; (void)b; (void)c; (void)d; (void)w;
  if (g_nfn < 1024) { g_fn[g_nfn].host = host; g_fn[g_nfn++].name = strdup(name); }
}
void __hipRegisterVar(void** m, void* v, char* h, char* d, int e, size_t s, int c, int g) {
  (void)m; (void)v; (void)h; (void)d; (void)e; (void)s; (void)c; (void)g;
}

/* ---- capture rules ----
 * While a stream captures in the default (global) mode, a call that allocates or asks about
 * completion is refused on every thread, and the capture is invalid from then on, unless the
 * thread has exchanged its own mode for relaxed. */
static __thread hipStreamCaptureMode t_mode = hipStreamCaptureModeGlobal;
static int unsafe(const char* what) {
  if (!s_global_capture || t_mode == hipStreamCaptureModeRelaxed) return 0;
  NOTE("capture_broken %s", what);
  return 1;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) {
  const hipStreamCaptureMode was = t_mode;
  t_mode = *m;
  *m = was;
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
  if (s == NULL && s_global_capture) return hipErrorStreamCaptureImplicit;
  *st = s_capturing[(size_t)s % 64] ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}

/* ---- device ---- */
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t* d) { (void)s; *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int d) {
  (void)d;
  *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 160 * 1024;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int threads, size_t lds) {
  (void)f; (void)threads;
  *n = lds >= 60000 ? 2 : 4;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* sym) { (void)sym; *p = calloc(1, 1 << 20); return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }

/* ---- memory ---- */
hipError_t hipMalloc(void** p, size_t n) {
  if (unsafe("hipMalloc")) return hipErrorStreamCaptureUnsupported;
  if (s_malloc_fails) return hipErrorOutOfMemory;
  *p = malloc(64);
  NOTE("malloc %zu -> %p", n, *p);
  return hipSuccess;
}
hipError_t hipFree(void* p) { NOTE("free %p", p); free(p); return hipSuccess; }

/* ---- events: each stands for the stream of its last record ---- */
static size_t g_event_stream[1024];
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned f) {
  static size_t n;
  (void)f;
  *e = (hipEvent_t)(++n);
  return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) {
  if (unsafe("hipEventQuery")) return hipErrorStreamCaptureUnsupported;
  return s_busy[g_event_stream[(size_t)e]] ? hipErrorNotReady : hipSuccess;
}

/* ---- launches ---- */
static __thread struct { dim3 g, b; size_t lds; hipStream_t s; } t_cfg;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
  t_cfg.g = g; t_cfg.b = b; t_cfg.lds = lds; t_cfg.s = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
  *g = t_cfg.g; *b = t_cfg.b; *lds = t_cfg.lds; *s = t_cfg.s;
  return hipSuccess;
}
static hipError_t launch(const void* f, dim3 g, dim3 b, size_t lds, hipStream_t s, hipEvent_t stop) {
  const char* name = "?";
  for (int i = 0; i < g_nfn; ++i)
    if (g_fn[i].host == f) name = g_fn[i].name;
  if ((unsigned long long)g.x * b.x > 0xffffffffull || (unsigned long long)g.y * b.y > 0xffffffffull || g.x == 0) {
    NOTE("refused %s", name);
    return hipErrorInvalidConfiguration;
  }
  if (stop) g_event_stream[(size_t)stop] = (size_t)s % 64;
  NOTE("launch %s grid %u %u block %u lds %zu stream %zu%s", name, g.x, g.y, b.x, lds, (size_t)s, stop ? " event" : "");
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void** a, size_t lds, hipStream_t s) {
  (void)a;
  return launch(f, g, b, lds, s, NULL);
}
hipError_t hipExtLaunchKernel(const void* f, dim3 g, dim3 b, void** a, size_t lds, hipStream_t s, hipEvent_t e0,
                              hipEvent_t e1, int flags) {
  (void)a; (void)e0; (void)flags;
  return launch(f, g, b, lds, s, e1);
}
