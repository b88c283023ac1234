/* A HIP runtime without a device for tests of the library's host paths: memory is
 * the host's, kernels do nothing, and a launch or an allocation is refused when
 * the environment says so.  Preloaded into a process of its own
 * (test_host_refusals.py); never used where kernels should run. */
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static struct {
  const void *host;
  const char *name;
} kernels[4096];
static int n_kernels;
static hipError_t last = hipSuccess;
static size_t host_bytes;           /* pinned memory held */

size_t fake_hip_host_bytes(void) { return host_bytes; }

void **__hipRegisterFatBinary(const void *data)
{
  static void *module;
  (void)data;
  return &module;
}
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterFunction(void **m, const void *host, char *dev, const char *name, unsigned n, void *a, void *b,
                           void *c, void *d, int *e)
{
  (void)m, (void)dev, (void)n, (void)a, (void)b, (void)c, (void)d, (void)e;
  if (strstr(name, "nrg") && n_kernels < 4096) {   /* not those of other libraries in the process */
    kernels[n_kernels].host = host;
    kernels[n_kernels++].name = name;
  }
}
void __hipRegisterVar(void **m, void *v, char *h, char *d, int e, size_t s, int c, int g)
{
  (void)m, (void)v, (void)h, (void)d, (void)e, (void)s, (void)c, (void)g;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st)
{
  (void)g, (void)b, (void)s, (void)st;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, hipStream_t *st)
{
  memset(g, 0, sizeof *g);
  memset(b, 0, sizeof *b);
  *s = 0;
  *st = 0;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t s, hipStream_t st)
{
  const char *refuse = getenv("FAKE_HIP_REFUSE_LAUNCH");
  (void)g, (void)b, (void)args, (void)s, (void)st;
  for (int i = 0; refuse && i < n_kernels; ++i)
    if (kernels[i].host == f && strstr(kernels[i].name, refuse)) last = hipErrorLaunchOutOfResources;
  return last;
}
hipError_t hipGetLastError(void)
{
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "refused"; }
hipError_t hipMalloc(void **p, size_t n) { return (*p = calloc(1, n ? n : 1)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p)
{
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned flags)
{
  (void)flags;
  *p = NULL;
  if (getenv("FAKE_HIP_REFUSE_PINNED")) return last = hipErrorOutOfMemory;
  size_t *q = calloc(1, n + 64);
  if (!q) return hipErrorOutOfMemory;
  *q = n;
  host_bytes += n;
  *p = (char *)q + 64;
  return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
  if (p) {
    size_t *q = (size_t *)((char *)p - 64);
    host_bytes -= *q;
    free(q);
  }
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k)
{
  (void)k;
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st)
{
  (void)st;
  return hipMemcpy(d, s, n, k);
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st)
{
  (void)st;
  memset(d, v, n);
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n)
{
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int d)
{
  (void)d;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int d)
{
  (void)d;
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t s)
{
  (void)f, (void)b, (void)s;
  *n = 4;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *sym)
{
  static void *mem;
  (void)sym;
  if (!mem) mem = calloc(1, 64u << 20);
  *p = mem;
  return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t *s)
{
  *s = (hipStream_t)calloc(1, 8);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
  free(s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s)
{
  (void)s;
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e)
{
  *e = (hipEvent_t)calloc(1, 8);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e)
{
  free(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
  (void)e, (void)s;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e)
{
  (void)e;
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b)
{
  (void)a, (void)b;
  *ms = 0.0f;
  return hipSuccess;
}
