/* A stand-in for the HIP runtime: one "device" in host memory, of a size that
 * the caller sets, with as much pinned host memory as the caller allows.
 * Copies are made at once, kernels do nothing, and fresh device memory holds
 * the numbers 0, 1, 2, ... as 32-bit words.  Loaded before libiamx.so with its
 * symbols global, it lets the host code run its allocation and transfer paths,
 * out-of-memory ones among them, where there is no GPU. */
#include <hip/hip_runtime_api.h>
#include <pthread.h>
#include <stdlib.h>
#include <string.h>

static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static size_t dev_limit = (size_t)8 << 30, dev_used, pin_limit = (size_t)8 << 30, pin_used, pin_peak;

void fake_limits(size_t device, size_t pinned) {
  dev_limit = device;
  pin_limit = pinned;
}
size_t fake_device_used(void) { return dev_used; }
size_t fake_pinned_peak(void) { return pin_peak; }

static __thread hipError_t last = hipSuccess;
static hipError_t error(hipError_t e) { return last = e; }

static void *take(size_t n, size_t *used, size_t limit) {
  pthread_mutex_lock(&mu);
  size_t *p = *used + n <= limit ? aligned_alloc(4096, ((n + 4095) & ~(size_t)4095) + 4096) : NULL;
  if (p) *used += n;
  if (pin_used > pin_peak) pin_peak = pin_used;
  pthread_mutex_unlock(&mu);
  if (!p) return NULL;
  *p = n;
  return (char *)p + 4096;
}
static void give(void *v, size_t *used) {
  if (!v) return;
  size_t *p = (size_t *)((char *)v - 4096);
  pthread_mutex_lock(&mu);
  *used -= *p;
  pthread_mutex_unlock(&mu);
  free(p);
}

hipError_t hipMalloc(void **p, size_t n) {
  if (!(*p = take(n, &dev_used, dev_limit))) return error(hipErrorOutOfMemory);
  for (size_t i = 0; i < n / 4; i++) ((unsigned *)*p)[i] = (unsigned)i;
  return hipSuccess;
}
hipError_t hipFree(void *p) { return give(p, &dev_used), hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned flags) {
  return (*p = take(n, &pin_used, pin_limit)) ? hipSuccess : error(hipErrorOutOfMemory);
}
hipError_t hipHostFree(void *p) { return give(p, &pin_used), hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned flags) { return *d = h, hipSuccess; }
hipError_t hipMemGetInfo(size_t *f, size_t *t) { return *f = dev_limit - dev_used, *t = dev_limit, hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) {
  return memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, hipMemcpyKind k,
                            hipStream_t st) {
  for (size_t i = 0; i < h; i++) memcpy((char *)d + i * dp, (const char *)s + i * sp, w);
  return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) { return memset(d, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st) { return memset(d, v, n), hipSuccess; }

hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int d) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int d) {
  memset(p, 0, sizeof(*p));
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipGetLastError(void) {
  const hipError_t e = last;
  return last = hipSuccess, e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
static char symbol[1 << 20];
hipError_t hipGetSymbolAddress(void **p, const void *s) { return *p = symbol, hipSuccess; }
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **a, size_t s, hipStream_t st) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, hipStream_t *st) {
  g->x = g->y = g->z = b->x = b->y = b->z = 1;
  return *s = 0, *st = NULL, hipSuccess;
}

static int handle;
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned f) { return *s = (hipStream_t)&handle, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned f) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t)&handle, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned f) { return *e = (hipEvent_t)&handle, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) { return *ms = 0, hipSuccess; }
