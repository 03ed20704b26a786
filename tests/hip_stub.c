/* A HIP runtime without a device, preloaded under the library in tests of its host code:
 * device memory is host memory, kernels do not run, and every call that orders or moves
 * something is written to the log. */
#define _GNU_SOURCE
#define __HIP_PLATFORM_AMD__ 1
#include <dlfcn.h>
#include <errno.h>
#include <hip/hip_runtime_api.h>
#include <pthread.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static char logbuf[1 << 22];
static size_t loglen;
static int no_threads, fail_after = -1;
static char fail_name[64];
static void (*on_sync)(const char*);
static struct { char* p; size_t n; int type; } mem[4096];
static int nmem;
static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;

const char* stub_log(void) { return logbuf; }
void stub_clear(void) { loglen = 0; logbuf[0] = 0; }
void stub_no_threads(int on) { no_threads = on; }
void stub_on_sync(void (*f)(const char*)) { on_sync = f; }
/* From now on let `n` calls of `name` succeed and fail all that follow. */
void stub_fail(const char* name, int n) {
  snprintf(fail_name, sizeof fail_name, "%s", name);
  fail_after = n;
}
/* The last pinned allocation of n bytes. */
void* stub_pinned(size_t n) {
  for (int i = nmem - 1; i >= 0; --i)
    if (mem[i].type == hipMemoryTypeHost && mem[i].n == n) return mem[i].p;
  return NULL;
}

static void say(const char* fmt, ...) {
  va_list a;
  pthread_mutex_lock(&mu);
  va_start(a, fmt);
  if (loglen < sizeof logbuf - 256) loglen += (size_t)vsnprintf(logbuf + loglen, 256, fmt, a);
  va_end(a);
  pthread_mutex_unlock(&mu);
}
static int failing(const char* name) {
  if (fail_after < 0 || strcmp(name, fail_name)) return 0;
  return fail_after == 0 ? 1 : (--fail_after, 0);
}
static hipError_t alloc(void** p, size_t n, int type) {
  *p = aligned_alloc(4096, (n + 4095) / 4096 * 4096);
  memset(*p, 0, n);
  pthread_mutex_lock(&mu);
  mem[nmem].p = *p;
  mem[nmem].n = n;
  mem[nmem++].type = type;
  pthread_mutex_unlock(&mu);
  return hipSuccess;
}
static int find(const void* p) {
  for (int i = nmem - 1; i >= 0; --i)
    if ((char*)p >= mem[i].p && (char*)p < mem[i].p + mem[i].n) return i;
  return -1;
}

int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* x) {
  static int (*real)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
  if (no_threads) return EAGAIN;
  if (!real) *(void**)&real = dlsym(RTLD_NEXT, "pthread_create");
  return real(t, a, f, x);
}

hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int d) { return (void)d, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int d) { return (void)a, (void)d, *v = 256, hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return (void)e, "stub error"; }
hipError_t hipGetSymbolAddress(void** p, const void* s) { return *p = (void*)s, hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
  say("malloc %zu\n", n);
  return alloc(p, n, hipMemoryTypeDevice);
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned f) { return (void)f, alloc(p, n, hipMemoryTypeHost); }
static hipError_t release(void* p) {
  const int i = find(p);
  if (i >= 0) mem[i].n = 0;
  return hipSuccess;
}
hipError_t hipFree(void* p) { return release(p); }
hipError_t hipHostFree(void* p) { return release(p); }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  const int i = find(p);
  memset(a, 0, sizeof *a);
  a->type = i < 0 ? hipMemoryTypeUnregistered : (enum hipMemoryType)mem[i].type;
  return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t* base, size_t* n, hipDeviceptr_t p) {
  const int i = find(p);
  if (i < 0) return hipErrorNotFound;
  *base = mem[i].p;
  *n = mem[i].n;
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) {
  say("copy %p %p %zu %d\n", d, s, n, (int)k);
  memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t st) {
  (void)st;
  return hipMemcpy(d, s, n, k);
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t s) { return (void)s, memset(d, v, n), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned f) {
  (void)f;
  if (failing("hipStreamCreateWithFlags")) return hipErrorOutOfMemory;
  *s = (hipStream_t)malloc(16);
  say("stream %p\n", (void*)*s);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  say("destroy %p\n", (void*)s);
  return hipSuccess;
}
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t* d) { return (void)s, *d = 0, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  say("sync %p\n", (void*)s);
  if (on_sync) on_sync("stream");
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned f) {
  (void)f;
  if (failing("hipStreamWaitEvent")) return hipErrorOutOfMemory;
  say("wait %p %p\n", (void*)s, (void*)e);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned f) {
  (void)f;
  if (failing("hipEventCreateWithFlags")) return hipErrorOutOfMemory;
  *e = (hipEvent_t)malloc(16);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { return (void)e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (failing("hipEventRecord")) return hipErrorOutOfMemory;
  say("record %p %p\n", (void*)s, (void*)e);
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  say("event %p\n", (void*)e);
  if (on_sync) on_sync("event");
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float* t, hipEvent_t a, hipEvent_t b) { return (void)a, (void)b, *t = 0, hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode m) { return (void)s, (void)m, hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) { return (void)s, *g = (hipGraph_t)malloc(16), hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t* n, char* l, size_t z) {
  (void)g, (void)n, (void)l, (void)z;
  *e = (hipGraphExec_t)malloc(16);
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { return (void)g, hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { return (void)e, hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s) {
  say("graph %p %p\n", (void*)s, (void*)e);
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void** a, size_t l, hipStream_t s) {
  (void)a, (void)l;
  say("launch %p %p %u %u\n", (void*)s, f, g.x, b.x);
  return hipSuccess;
}

static __thread struct { dim3 g, b; size_t l; hipStream_t s; } call;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t l, hipStream_t s) {
  call.g = g;
  call.b = b;
  call.l = l;
  call.s = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* l, hipStream_t* s) {
  *g = call.g;
  *b = call.b;
  *l = call.l;
  *s = call.s;
  return hipSuccess;
}
void** __hipRegisterFatBinary(const void* d) {
  static void* h;
  return (void)d, &h;
}
void __hipUnregisterFatBinary(void** h) { (void)h; }
void __hipRegisterFunction(void** h, const void* f, char* d, const char* n, unsigned l, void* t, void* b, void* bd,
                           void* gd, int* w) {
  (void)h, (void)f, (void)d, (void)n, (void)l, (void)t, (void)b, (void)bd, (void)gd, (void)w;
}
void __hipRegisterVar(void** h, void* v, char* hv, char* dv, int e, size_t n, int c, int g) {
  (void)h, (void)v, (void)hv, (void)dv, (void)e, (void)n, (void)c, (void)g;
}
