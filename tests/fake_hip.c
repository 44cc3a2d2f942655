/* A HIP runtime of two devices without a GPU, for tests of what the library asks of the runtime:
 * device memory is host memory, copies are done, kernels are not run.  Every launch, stream and
 * graph is written to a log of lines "launch <kernel> grid <blocks> block <threads> device <d>",
 * d being the device that the work would run on: the stream's, or for the null stream the current
 * one.  Handles are small structs that start with their device. */
#define _GNU_SOURCE
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

typedef struct { unsigned x, y, z; } dim3;
typedef struct { int device, capturing; } stream_t;
enum { OK = 0, INVALID = 1, CONFIG = 9 };

static int current, lastError;
static char *text;
static size_t used;
static int fail(int e) { return lastError = e; }

__attribute__((format(printf, 1, 2))) static void note(const char *fmt, ...) {
  if (!text) text = calloc(1, 1 << 22);
  __builtin_va_list ap;
  __builtin_va_start(ap, fmt);
  if (used < (1 << 22) - 512) used += vsnprintf(text + used, 512, fmt, ap);
  __builtin_va_end(ap);
}
const char *fake_log(void) { return text ? text : ""; }
void fake_log_clear(void) { if (text) text[used = 0] = 0; }

/* memory */
static struct { char *p; size_t n; int device; } mem[4096];
static int find(const void *p) {
  for (int k = 0; k < 4096; k++)
    if (mem[k].p && (char *)p >= mem[k].p && (char *)p < mem[k].p + mem[k].n) return k;
  return -1;
}
int hipMalloc(void **p, size_t n) {
  for (int k = 0; k < 4096; k++)
    if (!mem[k].p) {
      void *q = mmap(NULL, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
      if (q == MAP_FAILED) return fail(2);
      mem[k].p = *p = q, mem[k].n = n, mem[k].device = current;
      return OK;
    }
  return fail(2);
}
int hipFree(void *p) {
  const int k = find(p);
  if (k < 0 || mem[k].p != p) return fail(INVALID);
  munmap(p, mem[k].n);
  mem[k].p = NULL;
  return OK;
}
int hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; return (*p = calloc(1, n)) ? OK : fail(2); }
int hipHostFree(void *p) { free(p); return OK; }
typedef struct { int type, device; void *dev, *host; int managed; unsigned flags; } attributes;
int hipPointerGetAttributes(attributes *a, const void *p) {
  const int k = find(p);
  if (k < 0) return fail(INVALID);
  memset(a, 0, sizeof *a);
  a->type = 2; /* device */
  a->device = mem[k].device;
  return OK;
}
int hipMemGetAddressRange(void **base, size_t *n, void *p) {
  const int k = find(p);
  if (k < 0) return fail(INVALID);
  *base = mem[k].p, *n = mem[k].n;
  return OK;
}
int hipMemcpy(void *d, const void *s, size_t n, int k) { (void)k; memcpy(d, s, n); return OK; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, stream_t *st) { (void)st; return hipMemcpy(d, s, n, k); }
int hipMemset(void *d, int v, size_t n) { if (v || n < 1 << 20) memset(d, v, n); return OK; }
int hipMemsetAsync(void *d, int v, size_t n, stream_t *s) { (void)s; return hipMemset(d, v, n); }

/* devices, streams, events, graphs */
int hipGetDevice(int *d) { *d = current; return OK; }
int hipSetDevice(int d) { return d < 0 || d > 1 ? fail(101) : (current = d, OK); }
int hipGetDeviceCount(int *n) { *n = 2; return OK; }
int hipGetDevicePropertiesR0600(void *p, int d) { (void)p, (void)d; return fail(INVALID); }
int hipDeviceGetAttribute(int *v, int a, int d) { (void)a, (void)d; *v = 256; return OK; }
int hipDeviceSynchronize(void) { return OK; }
int hipStreamCreateWithFlags(stream_t **s, unsigned f) {
  (void)f;
  *s = calloc(1, sizeof **s);
  (*s)->device = current;
  note("stream device %d\n", current);
  return OK;
}
int hipStreamDestroy(stream_t *s) { free(s); return OK; }
int hipStreamSynchronize(stream_t *s) { (void)s; return OK; }
int hipStreamWaitEvent(stream_t *s, void *e, unsigned f) { (void)s, (void)e, (void)f; return OK; }
int hipStreamBeginCapture(stream_t *s, int m) { (void)m; s->capturing = 1; return OK; }
int hipStreamEndCapture(stream_t *s, void **g) { s->capturing = 0; *g = calloc(1, 8); return OK; }
int hipStreamIsCapturing(stream_t *s, int *c) { *c = s ? s->capturing : 0; return OK; }
int hipEventCreate(void **e) { *e = calloc(1, 8); return OK; }
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; return hipEventCreate(e); }
int hipEventDestroy(void *e) { free(e); return OK; }
int hipEventRecord(void *e, stream_t *s) { (void)e, (void)s; return OK; }
int hipEventSynchronize(void *e) { (void)e; return OK; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a, (void)b; *ms = 1; return OK; }
int hipGraphInstantiate(void **x, void *g, void *n, char *l, size_t z) {
  (void)g, (void)n, (void)l, (void)z;
  *x = calloc(1, 8);
  return OK;
}
int hipGraphDestroy(void *g) { free(g); return OK; }
int hipGraphExecDestroy(void *x) { free(x); return OK; }
int hipGraphUpload(void *x, stream_t *s) { (void)x, (void)s; return OK; }
int hipGraphLaunch(void *x, stream_t *s) { (void)x; note("graph device %d\n", s ? s->device : current); return OK; }
int hipGetLastError(void) { const int e = lastError; lastError = OK; return e; }
const char *hipGetErrorString(int e) { (void)e; return "fake error"; }

/* kernels */
static struct { const void *fn; const char *name; } kernels[4096];
static int nKernels;
void **__hipRegisterFatBinary(const void *d) { (void)d; static void *h; return &h; }
void __hipUnregisterFatBinary(void **h) { (void)h; }
void __hipRegisterFunction(void **h, const void *fn, char *d, const char *name, unsigned l, void *a, void *b, void *c,
                           void *e, int *w) {
  (void)h, (void)d, (void)l, (void)a, (void)b, (void)c, (void)e, (void)w;
  if (nKernels < 4096) kernels[nKernels].fn = fn, kernels[nKernels++].name = name;
}
void __hipRegisterVar(void **h, void *v, char *a, const char *n, int x, size_t z, int c, int g) {
  (void)h, (void)v, (void)a, (void)n, (void)x, (void)z, (void)c, (void)g;
}
int hipGetSymbolAddress(void **p, const void *s) { *p = (void *)s; return OK; }
int hipFuncGetAttributes(void *a, const void *fn) { (void)fn; memset(a, 0, 64); return OK; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *fn, int t, size_t l) {
  (void)fn, (void)l;
  *n = 1024 / t;
  return OK;
}
static struct { dim3 g, b; size_t l; stream_t *s; } pushed;
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t l, stream_t *s) {
  pushed.g = g, pushed.b = b, pushed.l = l, pushed.s = s;
  return OK;
}
int __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *l, stream_t **s) {
  *g = pushed.g, *b = pushed.b, *l = pushed.l, *s = pushed.s;
  return OK;
}
static int launch(const char *how, const void *fn, dim3 g, dim3 b, stream_t *s) {
  const char *name = "?";
  for (int k = 0; k < nKernels; k++)
    if (kernels[k].fn == fn) name = kernels[k].name;
  const uint64_t blocks = (uint64_t)g.x * g.y * g.z, threads = (uint64_t)b.x * b.y * b.z;
  /* the runtime's limit on a grid's work-items, per dimension */
  if (!blocks || (uint64_t)g.x * b.x >> 32 || (uint64_t)g.y * b.y >> 32 || threads > 1024) return fail(CONFIG);
  note("%s %s grid %llu block %llu device %d\n", how, name, (unsigned long long)blocks, (unsigned long long)threads,
       s ? s->device : current);
  return OK;
}
int hipLaunchKernel(const void *fn, dim3 g, dim3 b, void **a, size_t l, stream_t *s) {
  (void)a, (void)l;
  return launch("launch", fn, g, b, s);
}
int hipLaunchCooperativeKernel(const void *fn, dim3 g, dim3 b, void **a, unsigned l, stream_t *s) {
  (void)a, (void)l;
  return launch("cooperative", fn, g, b, s);
}
