/* A HIP runtime on the host for tests of the host code's error paths, put in
 * front of libamdhip64 by LD_PRELOAD: memory is host memory, copies are
 * memcpy, streams and events do nothing, kernels are not run.  fake_fail(name,
 * n) makes the n-th launch from then on of the kernels whose (mangled) name
 * holds name fail: the error stays until hipGetLastError takes it.
 * fake_grid(name): workgroups along x of their last launch. */
#include <stdlib.h>
#include <string.h>

enum { MAX_KERNELS = 4096, LAUNCH_FAILED = 719 };
static struct {
  const void *host;
  const char *name;
  unsigned grid;
} kernels[MAX_KERNELS];
static int nkernel, last, fail_at, token;
static char fail_name[64];

void fake_fail(const char *name, int n) {
  strncpy(fail_name, name, sizeof fail_name - 1);
  fail_at = n;
  last = 0;
}

unsigned fake_grid(const char *name) {
  for (int k = 0; k < nkernel; k++)
    if (kernels[k].grid && strstr(kernels[k].name, name)) return kernels[k].grid;
  return 0;
}

struct dim3 {
  unsigned x, y, z;
};
static struct dim3 grid_pushed;
int __hipPushCallConfiguration(struct dim3 grid) { return grid_pushed = grid, 0; }
int __hipPopCallConfiguration(struct dim3 *grid) { return *grid = grid_pushed, 0; }
int hipLaunchKernel(const void *f, struct dim3 grid) {
  int k;
  for (k = 0; k < nkernel && kernels[k].host != f;) k++;
  if (k == nkernel) return 0;
  if (fail_at > 0 && strstr(kernels[k].name, fail_name) && --fail_at == 0) return last = LAUNCH_FAILED;
  kernels[k].grid = grid.x;
  return 0;
}
int hipGetLastError(void) {
  const int e = last;
  last = 0;
  return e;
}
const char *hipGetErrorString(int e) { return e ? "fake failure" : "no error"; }

void **__hipRegisterFatBinary(const void *data) { return (void **)&token; }
void __hipRegisterFunction(void **m, const void *host, char *device, const char *name) {
  if (nkernel < MAX_KERNELS) {
    kernels[nkernel].host = host;
    kernels[nkernel++].name = name;
  }
}
void __hipRegisterVar(void) {}
void __hipUnregisterFatBinary(void) {}

static int alloc(void **p, size_t n) { return (*p = calloc(1, n ? n : 1)) ? 0 : 2; }
int hipMalloc(void **p, size_t n) { return alloc(p, n); }
int hipHostMalloc(void **p, size_t n, unsigned flags) { return alloc(p, n); }
int hipGetSymbolAddress(void **p, const void *symbol) { return alloc(p, 1 << 26); }
int hipFree(void *p) { return free(p), 0; }
int hipHostFree(void *p) { return free(p), 0; }
int hipMemcpy(void *d, const void *s, size_t n) { return memmove(d, s, n), 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n) { return memmove(d, s, n), 0; }
int hipMemset(void *d, int v, size_t n) { return memset(d, v, n), 0; }
int hipMemsetAsync(void *d, int v, size_t n) { return memset(d, v, n), 0; }
int hipGetDeviceCount(int *n) { return *n = 1, 0; }
int hipEventCreate(void **e) { return *e = &token, 0; }
int hipEventCreateWithFlags(void **e) { return *e = &token, 0; }
int hipStreamCreateWithFlags(void **s) { return *s = &token, 0; }
int hipEventElapsedTime(float *ms) { return *ms = 0.f, 0; }
int hipPointerGetAttributes(void) { return 1; }
int hipEventDestroy(void) { return 0; }
int hipEventRecord(void) { return 0; }
int hipEventSynchronize(void) { return 0; }
int hipFuncSetAttribute(void) { return 0; }
int hipSetDevice(void) { return 0; }
int hipStreamDestroy(void) { return 0; }
int hipStreamSynchronize(void) { return 0; }
int hipStreamWaitEvent(void) { return 0; }
