/* A host stand-in for the HIP runtime calls of libflutas_amd.so: "device"
 * memory is host memory with a limit, and a launch is recorded instead of run.
 * Loaded ahead of the library, it shows on the CPU what the host side of a call
 * allocates, launches and waits for, and what it does when memory is short. */
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <pthread.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

/* The header maps these names to versioned ones. */
#ifndef hipGetDeviceProperties
#error "hipGetDeviceProperties is expected to be a macro"
#endif

enum { MAXB = 4096, MAXK = 8192, MAXL = 4096, MAXS = 1 << 16 };
static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static struct { void *p; size_t n; } blk[MAXB];
static size_t used, peak, limit = (size_t)1 << 62;
static long long n_malloc, n_devsync, n_refused_launch;
static struct { const void *f; char name[512]; size_t lds_set, lds_max; int lowered; } kern[MAXK];
static int nkern;
static struct { int k; unsigned g[3], b[3]; size_t lds; void *s; } log_[MAXL];
static int nlog;

/* ---- what a test asks ---- */
void sim_limit(size_t n) { limit = n; }
size_t sim_used(void) { return used; }
size_t sim_peak(void) { return peak; }
void sim_reset(void) { nlog = 0; peak = used; n_malloc = n_devsync = n_refused_launch = 0; }
long long sim_count(int what) { return what == 0 ? n_malloc : what == 1 ? n_devsync : n_refused_launch; }
int sim_launches(void) { return nlog; }
const char *sim_launch(int i, unsigned *grid_block, size_t *lds, void **stream) {
  memcpy(grid_block, log_[i].g, sizeof log_[i].g);
  memcpy(grid_block + 3, log_[i].b, sizeof log_[i].b);
  *lds = log_[i].lds;
  *stream = log_[i].s;
  return kern[log_[i].k].name;
}
/* kernels whose dynamic LDS limit was ever set below an earlier setting */
int sim_lowered(void) {
  int n = 0;
  for (int i = 0; i < nkern; ++i) n += kern[i].lowered;
  return n;
}

static int kernel_of(const void *f) {
  for (int i = 0; i < nkern; ++i)
    if (kern[i].f == f) return i;
  if (nkern == MAXK) abort();
  kern[nkern].f = f;
  return nkern++;
}

/* ---- memory ---- */
static __thread hipError_t last;  /* what hipGetLastError returns */
hipError_t hipMalloc(void **p, size_t n) {
  hipError_t e = hipErrorOutOfMemory;
  *p = NULL;
  pthread_mutex_lock(&mu);
  ++n_malloc;
  if (n <= limit && used <= limit - n) {
    int i = 0;
    while (i < MAXB && blk[i].p) ++i;
    void *q = i < MAXB ? mmap(NULL, n ? n : 1, PROT_READ | PROT_WRITE,
                              MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0) : MAP_FAILED;
    if (q != MAP_FAILED) {
      blk[i].p = q;
      blk[i].n = n;
      used += n;
      if (used > peak) peak = used;
      *p = q;
      e = hipSuccess;
    }
  }
  pthread_mutex_unlock(&mu);
  if (e != hipSuccess) last = e;
  return e;
}
hipError_t hipFree(void *p) {
  if (!p) return hipSuccess;
  hipError_t e = hipErrorInvalidValue;
  pthread_mutex_lock(&mu);
  for (int i = 0; i < MAXB; ++i)
    if (blk[i].p == p) {
      munmap(p, blk[i].n ? blk[i].n : 1);
      used -= blk[i].n;
      blk[i].p = NULL;
      e = hipSuccess;
      break;
    }
  pthread_mutex_unlock(&mu);
  return e;
}
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t s) { (void)s; return hipMalloc(p, n); }
hipError_t hipFreeAsync(void *p, hipStream_t s) { (void)s; return hipFree(p); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; *p = calloc(1, n); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned f) { (void)f; *d = h; return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { (void)k; memmove(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) { (void)k; (void)st; memmove(d, s, n); return hipSuccess; }
hipError_t hipMemset(void *d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) { (void)p; memset(a, 0, sizeof *a); return hipSuccess; }

/* ---- device, streams, events ---- */
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int d) {
  (void)d;
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d) {
  (void)d;
  *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 0;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize(void) { ++n_devsync; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipGetLastError(void);
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "hipsim error"; }

/* ---- kernels ---- */
hipError_t hipGetLastError(void) { hipError_t e = last; last = hipSuccess; return e; }
static __thread struct { dim3 g, b; size_t lds; hipStream_t s; } call;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
  call.g = g; call.b = b; call.lds = lds; call.s = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
  *g = call.g; *b = call.b; *lds = call.lds; *s = call.s;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t lds, hipStream_t s) {
  (void)args;
  hipError_t e = hipSuccess;
  pthread_mutex_lock(&mu);
  const int k = kernel_of(f);
  /* the runtime's own limits: no empty grid, fewer than 2^32 threads in x */
  if (!g.x || !g.y || !g.z || !b.x || !b.y || !b.z ||
      (unsigned long long)g.x * b.x >> 32 || g.y > 65535 || g.z > 65535)
    e = hipErrorInvalidConfiguration;
  if (lds > 64 * 1024 && lds > kern[k].lds_set) e = hipErrorInvalidValue;
  if (e != hipSuccess) ++n_refused_launch;
  else if (nlog < MAXL) {
    log_[nlog].k = k;
    log_[nlog].g[0] = g.x; log_[nlog].g[1] = g.y; log_[nlog].g[2] = g.z;
    log_[nlog].b[0] = b.x; log_[nlog].b[1] = b.y; log_[nlog].b[2] = b.z;
    log_[nlog].lds = lds;
    log_[nlog].s = (void *)s;
    ++nlog;
  }
  pthread_mutex_unlock(&mu);
  last = e;
  return e;
}
hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute a, int v) {
  pthread_mutex_lock(&mu);
  const int k = kernel_of(f);
  if (a == hipFuncAttributeMaxDynamicSharedMemorySize) {
    if ((size_t)v < kern[k].lds_max) kern[k].lowered = 1;
    else kern[k].lds_max = v;
    kern[k].lds_set = v;
  }
  pthread_mutex_unlock(&mu);
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int t, size_t lds) {
  (void)f; (void)t; (void)lds;
  *n = 2;
  return hipSuccess;
}
void **__hipRegisterFatBinary(const void *d) { static void *m; (void)d; return &m; }
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterVar(void **m, void *v, char *hv, const char *n, int e, size_t s, int c, int g) { (void)m; (void)v; (void)hv; (void)n; (void)e; (void)s; (void)c; (void)g; }
void __hipRegisterFunction(void **m, const void *f, char *df, const char *name, unsigned t, void *a, void *b, void *c, void *d, int *w) {
  (void)m; (void)df; (void)t; (void)a; (void)b; (void)c; (void)d; (void)w;
  snprintf(kern[kernel_of(f)].name, sizeof kern[0].name, "%s", name);
}
