/* A HIP runtime for host tests without a device.  Device memory is host memory,
 * kernels are not run: each launch is written to a log with its kernel's
 * name, grid and first argument.  Loaded before librfxhip.so with its symbols
 * global, it takes the place of the real runtime for that library alone
 * (the test's process imports nothing else that uses HIP). */
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

typedef struct {
  uint32_t x, y, z;
} dim3_;

static char g_log[1 << 20];
static size_t g_at;
static int g_fail_at = -1;        /* allocations until one fails, -1: none */
static long long g_limit = -1;    /* larger allocations fail, -1: none */
static long long g_live, g_peak, g_last_pinned;
static int g_capture;             /* what hipStreamIsCapturing says */
static int g_mask_cus = -1;       /* compute units of every stream's mask, -1: all */
static int g_mode;                /* this thread's capture mode (0: global) */
static struct {
  const void* fn;
  char name[160];
} g_fn[512];
static int g_nfn;
static struct {
  dim3_ grid, block;
  size_t shmem;
  void* stream;
} g_cfg;

static void logf_(const char* fmt, ...) {
  va_list a;
  va_start(a, fmt);
  if (g_at + 512 < sizeof(g_log)) g_at += (size_t)vsnprintf(g_log + g_at, 512, fmt, a);
  va_end(a);
}

/* ---- the test's own side ---- */
const char* fake_log(void) { return g_log; }
void fake_clear(void) { g_at = 0, g_log[0] = 0; }
void fake_fail_at(int n) { g_fail_at = n; }
void fake_limit(long long bytes) { g_limit = bytes; }
void fake_capture(int on) { g_capture = on; }
void fake_mask(int cus) { g_mask_cus = cus; }
long long fake_live(void) { return g_live; }
long long fake_peak(void) { const long long p = g_peak; g_peak = 0; return p; }
uint32_t* fake_pinned(void) { return (uint32_t*)(uintptr_t)g_last_pinned; }

/* ---- memory ---- */
int hipMalloc(void** p, size_t n) {
  if (g_mode == 0) logf_("malloc-global %zu\n", n);
  if (g_fail_at >= 0 && g_fail_at-- == 0) return 2;
  if (g_limit >= 0 && (long long)n > g_limit) return 2;
  if ((long long)n > g_peak) g_peak = (long long)n;
  ++g_live;
  *p = calloc(1, n < (64u << 20) ? n : 64);   /* (nothing runs on the large ones) */
  return *p ? 0 : 2;
}
int hipFree(void* p) {
  if (p) --g_live;
  free(p);
  return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned flags) {
  (void)flags;
  *p = calloc(1, n);
  g_last_pinned = (long long)(uintptr_t)*p;
  return *p ? 0 : 2;
}
int hipHostFree(void* p) {
  free(p);
  return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int k) {
  (void)k;
  memcpy(d, s, n);
  return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* st) {
  (void)st;
  return hipMemcpy(d, s, n, k);
}
int hipMemsetAsync(void* d, int v, size_t n, void* st) {
  (void)d, (void)v, (void)n, (void)st;
  return 0;
}
int hipGetSymbolAddress(void** p, const void* sym) {
  static char scratch[1 << 24];
  (void)sym;
  *p = scratch;
  return 0;
}

/* ---- device, streams, events, graphs ---- */
int hipGetDevice(int* d) { return *d = 0; }
int hipDeviceGetAttribute(int* v, int attr, int dev) {
  (void)attr, (void)dev;
  *v = 256;
  return 0;
}
int hipDeviceGetPCIBusId(char* s, int n, int dev) {
  (void)dev;
  const char* bus = getenv("FAKE_HIP_BUS");
  snprintf(s, (size_t)n, "%s", bus ? bus : "fake");
  return 0;
}
int hipGetLastError(void) { return 0; }
const char* hipGetErrorString(int e) { return e ? "fake error" : "no error"; }
int hipThreadExchangeStreamCaptureMode(int* mode) {
  const int m = g_mode;
  g_mode = *mode;
  *mode = m;
  return 0;
}
int hipExtStreamGetCUMask(void* s, uint32_t n, uint32_t* m) {
  (void)s;
  int left = g_mask_cus < 0 ? 256 : g_mask_cus;
  for (uint32_t w = 0; w < n; ++w) {
    m[w] = left >= 32 ? ~0u : left > 0 ? (1u << left) - 1u : 0u;
    left -= 32;
  }
  return 0;
}
int hipStreamCreateWithFlags(void** s, unsigned f) {
  (void)f;
  *s = malloc(8);
  return 0;
}
int hipStreamDestroy(void* s) {
  free(s);
  return 0;
}
int hipStreamSynchronize(void* s) {
  (void)s;
  return 0;
}
int hipStreamIsCapturing(void* s, int* st) {
  (void)s;
  *st = g_capture;
  return 0;
}
int hipStreamBeginCapture(void* s, int mode) {
  (void)s, (void)mode;
  return 0;
}
int hipStreamEndCapture(void* s, void** g) {
  (void)s;
  *g = malloc(8);
  return 0;
}
int hipStreamWaitEvent(void* s, void* e, unsigned f) {
  (void)s, (void)e, (void)f;
  return 0;
}
int hipEventCreateWithFlags(void** e, unsigned f) {
  (void)f;
  *e = malloc(8);
  return 0;
}
int hipEventCreate(void** e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void* e) {
  free(e);
  return 0;
}
int hipEventRecord(void* e, void* s) {
  (void)e, (void)s;
  return 0;
}
int hipEventSynchronize(void* e) {
  (void)e;
  return 0;
}
int hipEventElapsedTime(float* ms, void* a, void* b) {
  (void)a, (void)b;
  *ms = 1.f;
  return 0;
}
int hipGraphInstantiate(void** x, void* g, void* n, char* b, size_t z) {
  (void)g, (void)n, (void)b, (void)z;
  *x = malloc(8);
  return 0;
}
int hipGraphDestroy(void* g) {
  free(g);
  return 0;
}
int hipGraphExecDestroy(void* g) {
  free(g);
  return 0;
}
int hipGraphLaunch(void* g, void* s) {
  (void)g;
  logf_("graph 1 1 1 %p\n", s);
  return 0;
}

/* ---- kernels ---- */
void** __hipRegisterFatBinary(const void* d) {
  static void* handle;
  (void)d;
  return &handle;
}
void __hipUnregisterFatBinary(void** m) { (void)m; }
void __hipRegisterFunction(void** m, const void* host, char* dev, const char* name, unsigned lim,
                           void* tid, void* bid, void* bd, void* gd, int* ws) {
  (void)m, (void)dev, (void)lim, (void)tid, (void)bid, (void)bd, (void)gd, (void)ws;
  if (g_nfn == 512) abort();
  g_fn[g_nfn].fn = host;
  snprintf(g_fn[g_nfn++].name, sizeof(g_fn[0].name), "%s", name);
}
void __hipRegisterVar(void** m, void* var, char* host, const char* dev, int ext, size_t n, int c,
                      int g) {
  (void)m, (void)var, (void)host, (void)dev, (void)ext, (void)n, (void)c, (void)g;
}
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t sh, void* s) {
  g_cfg.grid = g, g_cfg.block = b, g_cfg.shmem = sh, g_cfg.stream = s;
  return 0;
}
int __hipPopCallConfiguration(dim3_* g, dim3_* b, size_t* sh, void** s) {
  *g = g_cfg.grid, *b = g_cfg.block, *sh = g_cfg.shmem, *s = g_cfg.stream;
  return 0;
}
int hipLaunchKernel(const void* fn, dim3_ g, dim3_ b, void** args, size_t sh, void* s) {
  (void)b, (void)sh, (void)s;
  const char* name = "?";
  for (int i = 0; i < g_nfn; ++i)
    if (g_fn[i].fn == fn) name = g_fn[i].name;
  logf_("%s %u %u %u %p\n", name, g.x, g.y, g.z, *(void**)args[0]);
  return 0;
}
