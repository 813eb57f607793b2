/* A stand-in for the HIP runtime calls that libmask_srbcrs.so makes, for CPU
 * tests of its host code: device memory is host memory, kernels do nothing but
 * are counted by name, and calls can be made to fail.  Loaded with RTLD_GLOBAL
 * before the library, whose calls then come here.  What a kernel would have
 * counted is put into the library's device-to-host copies by fake_d2h. */
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

enum { kOk = 0, kOutOfMemory = 2, kUnsupportedInCapture = 900, kMax = 65536 };

typedef struct { unsigned x, y, z; } dim3_t;

static struct { void *p; size_t n; } g_live[kMax];
static int g_n_live;
static size_t g_live_bytes;
static long g_calls;             /* memset, copy and launch calls */
static long g_mallocs, g_syncs;
static long g_fail_malloc_from = -1, g_fail_malloc_count;
static long g_fail_sync_from = -1;
static int g_capturing;
static int g_last;
static const void *g_fn[4096];
static const char *g_fn_name[4096];
static long g_fn_launches[4096];
static int g_n_fn;
static struct { size_t n; unsigned char data[64]; } g_d2h[16];
static int g_n_d2h;

/* ---- the tests' side ---- */
size_t fake_live_bytes(void) { return g_live_bytes; }
int fake_live_blocks(void) { return g_n_live; }
long fake_calls(void) { return g_calls; }
long fake_mallocs(void) { return g_mallocs; }
/* the next `skip` hipMalloc calls work, the `count` after them fail */
void fake_fail_malloc(long skip, long count) { g_fail_malloc_from = g_mallocs + skip; g_fail_malloc_count = count; }
/* every synchronisation after the next `skip` ones fails; skip < 0: none does */
void fake_fail_sync(long skip) { g_fail_sync_from = skip < 0 ? -1 : g_syncs + skip; }
void fake_capture(int on) { g_capturing = on; }
/* device-to-host copies of n bytes give these bytes (n = 0: forget all) */
void fake_d2h(size_t n, const void *data) {
  if (n == 0) { g_n_d2h = 0; return; }
  for (int i = 0; i < g_n_d2h; ++i)
    if (g_d2h[i].n == n) { memcpy(g_d2h[i].data, data, n); return; }
  if (n > 64 || g_n_d2h == 16) abort();
  g_d2h[g_n_d2h].n = n;
  memcpy(g_d2h[g_n_d2h++].data, data, n);
}
long fake_launches(const char *part) {
  long n = 0;
  for (int i = 0; i < g_n_fn; ++i)
    if (strstr(g_fn_name[i], part)) n += g_fn_launches[i];
  return n;
}

/* ---- the runtime's side ---- */
int hipMalloc(void **p, size_t n) {
  const long i = g_mallocs++;
  *p = NULL;
  if (g_fail_malloc_from >= 0 && i >= g_fail_malloc_from && i < g_fail_malloc_from + g_fail_malloc_count)
    return g_last = kOutOfMemory;
  if (g_capturing) return g_last = kUnsupportedInCapture;
  if (g_n_live == kMax || !(*p = calloc(1, n ? n : 1))) return g_last = kOutOfMemory;
  g_live[g_n_live].p = *p;
  g_live[g_n_live++].n = n;
  g_live_bytes += n;
  return kOk;
}
int hipFree(void *p) {
  for (int i = 0; i < g_n_live; ++i)
    if (g_live[i].p == p) {
      g_live_bytes -= g_live[i].n;
      g_live[i] = g_live[--g_n_live];
      free(p);
      return kOk;
    }
  if (p) abort();   /* freed twice, or never allocated */
  return kOk;
}
static int sync_result(void) {
  const long i = g_syncs++;
  if (g_capturing) return g_last = kUnsupportedInCapture;
  return g_fail_sync_from >= 0 && i >= g_fail_sync_from ? (g_last = 719) : kOk;
}
int hipStreamSynchronize(void *s) { (void)s; return sync_result(); }
int hipDeviceSynchronize(void) { return sync_result(); }
int hipMemsetAsync(void *p, int v, size_t n, void *s) { (void)s; ++g_calls; memset(p, v, n); return kOk; }
static int copy(void *d, const void *s, size_t n, int kind) {
  ++g_calls;
  memmove(d, s, n);
  if (kind == 2)
    for (int i = 0; i < g_n_d2h; ++i)
      if (g_d2h[i].n == n) memcpy(d, g_d2h[i].data, n);
  return kOk;
}
int hipMemcpy(void *d, const void *s, size_t n, int kind) { return copy(d, s, n, kind); }
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st) { (void)st; return copy(d, s, n, kind); }
int hipStreamIsCapturing(void *s, int *status) { (void)s; *status = g_capturing; return kOk; }
int hipThreadExchangeStreamCaptureMode(int *mode) { (void)mode; return kOk; }
int hipGetLastError(void) { const int e = g_last; g_last = kOk; return e; }
const char *hipGetErrorString(int e) {
  return e == kOutOfMemory ? "out of memory" : e == kUnsupportedInCapture ? "not permitted under capture" : "error";
}
int hipGetDevice(int *d) { *d = 0; return kOk; }
int hipSetDevice(int d) { (void)d; return kOk; }
int hipGetStreamDeviceId(void *s) { (void)s; return 0; }
int hipDeviceGetAttribute(int *v, int a, int d) { (void)a; (void)d; *v = 256; return kOk; }
int hipGetDevicePropertiesR0600(void *p, int d) { (void)d; memset(p, 0, 256); return kOk; }
int hipGetSymbolAddress(void **p, const void *s) { *p = (void *)s; return kOk; }
int hipEventCreate(void **e) { *e = (void *)1; return kOk; }
int hipEventDestroy(void *e) { (void)e; return kOk; }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return kOk; }
int hipEventSynchronize(void *e) { (void)e; return kOk; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 1.f; return kOk; }
int hipLaunchKernel(const void *f, dim3_t g, dim3_t b, void **args, size_t lds, void *s) {
  (void)g; (void)b; (void)args; (void)lds; (void)s;
  ++g_calls;
  for (int i = 0; i < g_n_fn; ++i)
    if (g_fn[i] == f) ++g_fn_launches[i];
  return kOk;
}
static struct { dim3_t g, b; size_t lds; void *s; } g_cfg;
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t lds, void *s) {
  g_cfg.g = g; g_cfg.b = b; g_cfg.lds = lds; g_cfg.s = s;
  return kOk;
}
int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *lds, void **s) {
  *g = g_cfg.g; *b = g_cfg.b; *lds = g_cfg.lds; *s = g_cfg.s;
  return kOk;
}
void **__hipRegisterFatBinary(const void *d) { static void *h; (void)d; return &h; }
void __hipUnregisterFatBinary(void **h) { (void)h; }
void __hipRegisterVar(void **h, void *v, char *a, char *b, int c, size_t n, int d, int e) {
  (void)h; (void)v; (void)a; (void)b; (void)c; (void)n; (void)d; (void)e;
}
void __hipRegisterFunction(void **h, const void *f, char *dn, const char *name, unsigned t, void *a, void *b, void *c,
                           void *d, int *w) {
  (void)h; (void)dn; (void)t; (void)a; (void)b; (void)c; (void)d; (void)w;
  if (g_n_fn < 4096) { g_fn[g_n_fn] = f; g_fn_name[g_n_fn++] = strdup(name); }
}
