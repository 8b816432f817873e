// A HIP runtime on host memory for tests of the host code without a GPU (preloaded before libamdhip64): allocations are the
// heap's, copies are copies, kernels are counted by name and not run.  A chosen allocation can be made to fail.
#include <stddef.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

enum { OK = 0, OUT_OF_MEMORY = 2, H2D = 1 };
typedef struct { unsigned x, y, z; } dim3;

static struct { const void *host; const char *name; long count; } kernels[4096];
static int       nkernels;
static long long h2d_bytes, dev_bytes;
static long      fail_malloc = -1, fail_host_malloc = -1;  // how many more succeed before one fails

long long fake_h2d_bytes(void) { return h2d_bytes; }
long long fake_dev_bytes(void) { return dev_bytes; }
void      fake_fail_malloc(long after) { fail_malloc = after; }
void      fake_fail_host_malloc(long after) { fail_host_malloc = after; }
long      fake_launches(const char *part) {
  long n = 0;
  for (int i = 0; i < nkernels; i++)
    if (strstr(kernels[i].name, part)) n += kernels[i].count;
  return n;
}

int hipGetDeviceCount(int *n) { return *n = 1, OK; }
int hipGetDevice(int *d) { return *d = 0, OK; }
int hipSetDevice(int d) { return OK; }
int hipDeviceGetAttribute(int *v, int attr, int d) { return *v = 256, OK; }
int hipGetLastError(void) { return OK; }
const char *hipGetErrorName(int e) { return e ? "hipErrorOutOfMemory" : "hipSuccess"; }
const char *hipGetErrorString(int e) { return hipGetErrorName(e); }
int hipMalloc(void **p, size_t n) {
  *p = NULL;
  if (fail_malloc >= 0 && fail_malloc-- == 0) return OUT_OF_MEMORY;
  dev_bytes += (long long)n;
  return (*p = calloc(1, n ? n : 1)) ? OK : OUT_OF_MEMORY;
}
int hipFree(void *p) { return free(p), OK; }
int hipHostMalloc(void **p, size_t n, unsigned flags) {
  *p = NULL;
  if (fail_host_malloc >= 0 && fail_host_malloc-- == 0) return OUT_OF_MEMORY;
  return (*p = calloc(1, n ? n : 1)) ? OK : OUT_OF_MEMORY;
}
int hipHostFree(void *p) { return free(p), OK; }
int hipHostGetDevicePointer(void **d, void *h, unsigned flags) { return *d = h, OK; }
int hipMemcpy(void *d, const void *s, size_t n, int kind) {
  if (kind == H2D) h2d_bytes += (long long)n;
  return memcpy(d, s, n), OK;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *stream) { return hipMemcpy(d, s, n, kind); }
int hipMemsetAsync(void *d, int v, size_t n, void *stream) { return memset(d, v, n), OK; }
int hipStreamCreate(void **s) { return *s = NULL, OK; }
int hipStreamDestroy(void *s) { return OK; }
int hipStreamSynchronize(void *s) { return OK; }
int hipEventCreateWithFlags(void **e, unsigned f) { return *e = NULL, OK; }
int hipEventDestroy(void *e) { return OK; }
int hipEventRecord(void *e, void *s) { return OK; }
int hipEventElapsedTime(float *t, void *a, void *b) { return *t = 0, OK; }
int hipGetSymbolAddress(void **p, const void *symbol) {  // the fixed scratch: 96 MiB, of which nothing is touched
  static void *scratch;
  if (!scratch) scratch = calloc(96, 1 << 20);
  return *p = scratch, scratch ? OK : OUT_OF_MEMORY;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int block, size_t lds) { return *n = 2, OK; }
int hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t lds, void *stream) {
  for (int i = 0; i < nkernels; i++)
    if (kernels[i].host == f) return kernels[i].count++, OK;
  fprintf(stderr, "fake_hip: launch of an unregistered kernel\n");
  abort();
}
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, void *stream) { return OK; }
int __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, void **stream) {
  *grid = *block = (dim3){1, 1, 1};
  return *lds = 0, *stream = NULL, OK;
}
void **__hipRegisterFatBinary(const void *data) {
  static void *module;
  return &module;
}
void __hipRegisterFunction(void **m, const void *host, char *stub, const char *name, unsigned limit, void *t, void *b, void *bd, void *gd, int *w) {
  if (nkernels == 4096) abort();
  kernels[nkernels].host = host, kernels[nkernels++].name = name;
}
void __hipRegisterVar(void **m, void *var, char *stub, char *name, int ext, size_t size, int constant, int global) {}
void __hipUnregisterFatBinary(void **m) {}
