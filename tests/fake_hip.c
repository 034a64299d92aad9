/* A host-memory stand-in for the HIP runtime calls of libatrip_hip.so, for tests
 * of its memory handling on the CPU: allocations come from host memory up to a
 * limit, copies are copies, kernels take a settable time and do nothing (so
 * energies are zero). */
#include <pthread.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

enum { OK = 0, OUT_OF_MEMORY = 2, MAX_BLOCKS = 4096 };
static struct { void *p; size_t n; } block[MAX_BLOCKS];
static size_t limit = SIZE_MAX, used;

static pthread_mutex_t lock = PTHREAD_MUTEX_INITIALIZER;
static unsigned launch_us;

void fake_set_limit(size_t bytes) { limit = bytes; }
size_t fake_used(void) { return used; }
void fake_set_launch_us(unsigned us) { launch_us = us; }

static int take(void **p, size_t n) {
  *p = NULL;
  if (n > limit || used > limit - n) return OUT_OF_MEMORY;
  for (int q = 0; q < MAX_BLOCKS; q++)
    if (!block[q].p) {
      if (!(*p = calloc(1, n))) return OUT_OF_MEMORY;
      block[q].p = *p;
      block[q].n = n;
      used += n;
      return OK;
    }
  return OUT_OF_MEMORY;
}
static int give(void *p) {
  for (int q = 0; q < MAX_BLOCKS && p; q++)
    if (block[q].p == p) {
      used -= block[q].n;
      block[q].p = NULL;
      free(p);
      return OK;
    }
  return p ? 1 : OK;
}
int hipMalloc(void **p, size_t n) {
  pthread_mutex_lock(&lock);
  const int e = take(p, n);
  pthread_mutex_unlock(&lock);
  return e;
}
int hipFree(void *p) {
  pthread_mutex_lock(&lock);
  const int e = give(p);
  pthread_mutex_unlock(&lock);
  return e;
}
int hipHostMalloc(void **p, size_t n, unsigned flags) {
  (void)flags;
  return (*p = malloc(n)) ? OK : OUT_OF_MEMORY;
}
int hipHostFree(void *p) { free(p); return OK; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st) {
  (void)kind; (void)st;
  memcpy(d, s, n);
  return OK;
}
int hipMemsetAsync(void *d, int v, size_t n, void *st) {
  (void)st;
  memset(d, v, n);
  return OK;
}
int hipGetDeviceCount(int *n) { *n = 1; return OK; }
int hipSetDevice(int d) { (void)d; return OK; }
int hipDeviceGetAttribute(int *v, int a, int d) { (void)a; (void)d; *v = 4; return OK; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t l) {
  (void)f; (void)b; (void)l;
  *n = 2;
  return OK;
}
int hipFuncSetAttribute(const void *f, int a, int v) { (void)f; (void)a; (void)v; return OK; }
int hipGetSymbolAddress(void **p, const void *s) { (void)s; *p = NULL; return 1; }
int hipStreamCreate(void **s) { *s = malloc(1); return OK; }
int hipStreamDestroy(void *s) { free(s); return OK; }
int hipStreamSynchronize(void *s) { (void)s; return OK; }
int hipEventCreate(void **e) { *e = malloc(1); return OK; }
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; *e = malloc(1); return OK; }
int hipEventDestroy(void *e) { free(e); return OK; }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return OK; }
int hipEventSynchronize(void *e) { (void)e; return OK; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 1.f; return OK; }
const char *hipGetErrorString(int e) {
  return e == OUT_OF_MEMORY ? "out of memory" : e ? "failure" : "no error";
}
int hipGetLastError(void) { return OK; }
typedef struct { unsigned x, y, z; } dims;
int hipLaunchKernel(const void *f, dims g, dims b, void **a, size_t l, void *s) {
  (void)f; (void)g; (void)b; (void)a; (void)l; (void)s;
  if (launch_us) usleep(launch_us);
  return OK;
}
int __hipPushCallConfiguration(dims g, dims b, size_t l, void *s) {
  (void)g; (void)b; (void)l; (void)s;
  return OK;
}
int __hipPopCallConfiguration(dims *g, dims *b, size_t *l, void **s) {
  memset(g, 0, sizeof *g);
  memset(b, 0, sizeof *b);
  *l = 0;
  *s = NULL;
  return OK;
}
void **__hipRegisterFatBinary(const void *d) { (void)d; static void *h; return &h; }
void __hipUnregisterFatBinary(void **h) { (void)h; }
void __hipRegisterFunction(void **h, const void *f, char *d, const char *n, unsigned t,
                           void *a, void *b, void *c, void *e, int *w) {
  (void)h; (void)f; (void)d; (void)n; (void)t; (void)a; (void)b; (void)c; (void)e; (void)w;
}
void __hipRegisterVar(void *h, void *v, char *a, char *b, int e, size_t n, int c, int g) {
  (void)h; (void)v; (void)a; (void)b; (void)e; (void)n; (void)c; (void)g;
}
