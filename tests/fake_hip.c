/* A HIP runtime of two devices without hardware, for test_device_selection.py:
 * memory is host memory with its device noted, copies are done, kernels are
 * not run.  fake_faults() counts what a two-GPU node would do wrong: a launch
 * on a stream of another device than the current one, a copy between a stream
 * and memory of another device. */
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

typedef struct { uint32_t x, y, z; } dim3;
typedef struct { int dev; } stream_t;
struct block { char *p; size_t n; int dev; };

static int cur, faults, nblocks;
static struct block blocks[4096];

static int device_of(const void *p) {
  for (int k = 0; k < nblocks; ++k)
    if ((const char *)p >= blocks[k].p && (const char *)p < blocks[k].p + blocks[k].n)
      return blocks[k].dev;
  return -1; /* host memory */
}

static int stream_device(const stream_t *s) { return s ? s->dev : cur; }

int fake_faults(void) { int f = faults; faults = 0; return f; }

int hipGetDeviceCount(int *n) { *n = 2; return 0; }
int hipSetDevice(int d) { cur = d; return 0; }
int hipGetDevice(int *d) { *d = cur; return 0; }
const char *hipGetErrorString(int e) { (void)e; return "fake"; }
int hipGetLastError(void) { return 0; }

int hipMalloc(void **p, size_t n) {
  if (nblocks == 4096) return 2;
  *p = calloc(1, n + 1);
  blocks[nblocks++] = (struct block){*p, n, cur};
  return 0;
}
int hipFree(void *p) {
  for (int k = 0; k < nblocks; ++k)
    if (blocks[k].p == p) {
      blocks[k] = blocks[--nblocks];
      break;
    }
  free(p);
  return 0;
}
int hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; *p = calloc(1, n + 1); return 0; }
int hipHostFree(void *p) { free(p); return 0; }
int hipHostGetDevicePointer(void **d, void *h, unsigned f) { (void)f; *d = h; return 0; }
int hipGetSymbolAddress(void **d, const void *s) { (void)d; (void)s; return 1; }

int hipStreamCreateWithFlags(stream_t **s, unsigned f) {
  (void)f;
  *s = malloc(sizeof(stream_t));
  (*s)->dev = cur;
  return 0;
}
int hipStreamDestroy(stream_t *s) { free(s); return 0; }
int hipStreamSynchronize(stream_t *s) { (void)s; return 0; }
int hipStreamQuery(stream_t *s) { (void)s; return 0; }
int hipStreamWaitEvent(stream_t *s, void *e, unsigned f) { (void)s; (void)e; (void)f; return 0; }
int hipEventCreate(void **e) { *e = malloc(1); return 0; }
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; *e = malloc(1); return 0; }
int hipEventDestroy(void *e) { free(e); return 0; }
int hipEventRecord(void *e, stream_t *s) { (void)e; (void)s; return 0; }
int hipEventSynchronize(void *e) { (void)e; return 0; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 1.0f; return 0; }

int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, stream_t *st) {
  (void)kind;
  const int dd = device_of(d), ds = device_of(s);
  if ((dd >= 0 && dd != stream_device(st)) || (ds >= 0 && ds != stream_device(st))) ++faults;
  memcpy(d, s, n);
  return 0;
}
int hipMemsetAsync(void *d, int v, size_t n, stream_t *st) {
  if (device_of(d) != stream_device(st)) ++faults;
  memset(d, v, n);
  return 0;
}
int hipLaunchKernel(const void *f, dim3 g, dim3 b, void **a, size_t lds, stream_t *st) {
  (void)f; (void)g; (void)b; (void)a; (void)lds;
  if (stream_device(st) != cur) ++faults;
  return 0;
}

static dim3 cfg_g, cfg_b;
static size_t cfg_l;
static stream_t *cfg_s;
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t l, stream_t *s) {
  cfg_g = g;
  cfg_b = b;
  cfg_l = l;
  cfg_s = s;
  return 0;
}
int __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *l, stream_t **s) {
  *g = cfg_g;
  *b = cfg_b;
  *l = cfg_l;
  *s = cfg_s;
  return 0;
}
void **__hipRegisterFatBinary(const void *p) { (void)p; static void *h; return &h; }
void __hipRegisterFunction(void **m, const void *f, char *d, const char *n, unsigned t, void *a,
                           void *b, dim3 *c, dim3 *e, int *w) {
  (void)m; (void)f; (void)d; (void)n; (void)t; (void)a; (void)b; (void)c; (void)e; (void)w;
}
void __hipRegisterVar(void **m, void *v, char *a, char *b, int e, size_t s, int c, int g) {
  (void)m; (void)v; (void)a; (void)b; (void)e; (void)s; (void)c; (void)g;
}
void __hipUnregisterFatBinary(void **m) { (void)m; }
