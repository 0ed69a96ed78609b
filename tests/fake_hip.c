/* Stand-ins for the HIP runtime calls of the host library, preloaded by
 * test_async_sources.py: device memory is host memory, kernels do nothing,
 * and an asynchronous copy takes place only at the next wait (of any stream
 * or event, or hipFree, which waits for the device), as the interface allows.
 * Its source has to be alive then. */
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

enum { kOps = 4096 };
static struct {
  void *dst;
  const void *src; /* null: a fill with value */
  int value;
  size_t n;
} g_op[kOps];
static int g_ops;

static int flush(void) {
  for (int i = 0; i < g_ops; ++i) {
    if (g_op[i].src) memcpy(g_op[i].dst, g_op[i].src, g_op[i].n);
    else memset(g_op[i].dst, g_op[i].value, g_op[i].n);
  }
  g_ops = 0;
  return 0;
}
static int put(void *dst, const void *src, int value, size_t n) {
  if (g_ops == kOps) abort();
  g_op[g_ops].dst = dst;
  g_op[g_ops].src = src;
  g_op[g_ops].value = value;
  g_op[g_ops++].n = n;
  return 0;
}
static int handle(void **p) {
  *p = malloc(1);
  return 0;
}

int hipGetDeviceCount(int *n) { return *n = 1, 0; }
int hipGetDevice(int *d) { return *d = 0; }
int hipSetDevice(int d) { return d; }
int hipGetLastError(void) { return 0; }
const char *hipGetErrorString(int e) { return e ? "error" : "no error"; }
int hipMalloc(void **p, size_t n) { return (*p = calloc(1, n)) ? 0 : 2; }
int hipHostMalloc(void **p, size_t n, unsigned f) { return (*p = calloc(1, n)) ? 0 : (int)f + 2; }
int hipFree(void *p) { return flush(), free(p), 0; }
int hipHostFree(void *p) { return flush(), free(p), 0; }
int hipGetSymbolAddress(void **p, const void *s) { return (*p = calloc(1, 64u << 20)) ? 0 : s != 0; }
int hipFuncGetAttributes(void *a, const void *f) { return !a || !f; }
int hipFuncSetAttribute(const void *f, int a, int v) { return !f && a && v; }
int hipEventCreate(void **e) { return handle(e); }
int hipEventCreateWithFlags(void **e, unsigned f) { return (void)f, handle(e); }
int hipEventDestroy(void *e) { return free(e), 0; }
int hipEventElapsedTime(float *ms, void *a, void *b) { return *ms = 1.f, !a || !b; }
int hipEventRecord(void *e, void *s) { return (void)s, !e; }
int hipEventSynchronize(void *e) { return (void)e, flush(); }
int hipStreamCreateWithFlags(void **s, unsigned f) { return (void)f, handle(s); }
int hipStreamIsCapturing(void *s, int *st) { return (void)s, *st = 0; }
int hipStreamSynchronize(void *s) { return (void)s, flush(); }
int hipStreamWaitEvent(void *s, void *e, unsigned f) { return (void)s, (void)e, (int)f; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) {
  return (void)k, (void)st, put(d, s, 0, n);
}
int hipMemsetAsync(void *d, int v, size_t n, void *st) { return (void)st, put(d, 0, v, n); }
typedef struct {
  uint32_t x, y, z;
} Dim;
int hipLaunchKernel(const void *f, Dim g, Dim b, void **a, size_t l, void *s) {
  return (void)f, (void)g, (void)b, (void)a, (void)l, (void)s, 0;
}
