/* A HIP runtime without a device, for tests of the host side of
 * librapt_hip.so: loaded globally in front of the library, its symbols are the
 * ones the library calls.  Device memory is host memory under a budget,
 * copies copy, kernels do nothing (their grids are counted by name). */
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>
#include <stdlib.h>
#include <string.h>

enum { MAXK = 4096 };
static struct {
  const void* fn;
  const char* name;
} kernels[MAXK];
static int n_kernels;

/* what a test sets and reads */
size_t fake_budget = (size_t)1 << 40, fake_used; /* bytes that may be allocated, and are */
int fake_fail_copy = -1;   /* asynchronous copies that succeed before one fails; -1: all do */
int fake_pending;          /* operations since the stream was last synchronised */
size_t fake_overflow_bytes; /* the next copy from the device of this many bytes is all
                               "too many points" (-20), then the option is off */
int fake_pinned_lookup;    /* 1: every host pointer is one of the runtime's */
int fake_copies;           /* asynchronous copies */
size_t fake_largest_copy;  /* bytes, of those from the device */
const char *fake_last_kernel = "", *fake_epoch_kernel = ""; /* ..., of those captured */
static int capturing;
unsigned fake_last_grid, fake_last_block, fake_epoch_lanes;
static hipError_t last;

static hipError_t ret(hipError_t e) {
  if (e != hipSuccess) last = e;
  return e;
}

hipError_t hipMalloc(void** p, size_t n) {
  if (fake_used + n > fake_budget) return ret(hipErrorOutOfMemory);
  size_t* m = calloc(1, n + 256);
  if (!m) return ret(hipErrorOutOfMemory);
  m[0] = n;
  fake_used += n;
  *p = (char*)m + 256;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!p) return hipSuccess;
  size_t* m = (size_t*)((char*)p - 256);
  fake_used -= m[0];
  free(m);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  *t = fake_budget;
  *f = fake_budget - fake_used;
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) {
  (void)flags;
  *p = malloc(n);
  return *p ? hipSuccess : ret(hipErrorOutOfMemory);
}
hipError_t hipHostFree(void* p) {
  free(p);
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  (void)p;
  memset(a, 0, sizeof *a);
  a->type = fake_pinned_lookup ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return fake_pinned_lookup ? hipSuccess : ret(hipErrorInvalidValue);
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) {
  (void)k;
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t st) {
  (void)st;
  if (fake_fail_copy == 0) return ret(hipErrorUnknown);
  if (fake_fail_copy > 0) --fake_fail_copy;
  ++fake_pending;
  ++fake_copies;
  if (k == hipMemcpyDeviceToHost && n > fake_largest_copy) fake_largest_copy = n;
  memcpy(d, s, n);
  if (k == hipMemcpyDeviceToHost && n && n == fake_overflow_bytes) {
    for (size_t i = 0; i < n / 4; ++i) ((int*)d)[i] = -20;
    fake_overflow_bytes = 0;
  }
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t st) {
  (void)st;
  ++fake_pending;
  memset(d, v, n);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t st) {
  (void)st;
  fake_pending = 0;
  return hipSuccess;
}

static void launched(const char* name, unsigned grid, unsigned block) {
  ++fake_pending;
  fake_last_kernel = name;
  if (capturing && strstr(name, "k_trace")) {
    fake_epoch_kernel = name;
    fake_epoch_lanes = grid * block;
  }
  fake_last_grid = grid;
  fake_last_block = block;
}
hipError_t hipLaunchKernel(const void* fn, dim3 g, dim3 b, void** args, size_t sh,
                           hipStream_t st) {
  (void)args, (void)sh, (void)st;
  for (int i = 0; i < n_kernels; ++i)
    if (kernels[i].fn == fn) {
      launched(kernels[i].name, g.x, b.x);
      return hipSuccess;
    }
  return ret(hipErrorInvalidDeviceFunction);
}
static dim3 cfg_g, cfg_b;
static size_t cfg_sh;
static hipStream_t cfg_st;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t st) {
  cfg_g = g, cfg_b = b, cfg_sh = sh, cfg_st = st;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, hipStream_t* st) {
  *g = cfg_g, *b = cfg_b, *sh = cfg_sh, *st = cfg_st;
  return hipSuccess;
}
void** __hipRegisterFatBinary(const void* data) {
  static void* module;
  (void)data;
  return &module;
}
void __hipUnregisterFatBinary(void** m) { (void)m; }
void __hipRegisterFunction(void** m, const void* fn, char* dev, const char* name, unsigned lim,
                           void* tid, void* bid, dim3* bd, dim3* gd, int* ws) {
  (void)m, (void)dev, (void)lim, (void)tid, (void)bid, (void)bd, (void)gd, (void)ws;
  if (n_kernels < MAXK) {
    kernels[n_kernels].fn = fn;
    kernels[n_kernels++].name = name;
  }
}
void __hipRegisterVar(void** m, void* var, char* host, const char* dev, int ext, size_t n, int c,
                      int g) {
  (void)m, (void)var, (void)host, (void)dev, (void)ext, (void)n, (void)c, (void)g;
}
hipError_t hipGetSymbolAddress(void** p, const void* sym) {
  static unsigned long long mem[4096];
  (void)sym;
  *p = mem;
  return hipSuccess;
}

hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int d) {
  (void)d;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int d) {
  (void)d;
  *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 0;
  return hipSuccess;
}
hipError_t hipGetLastError(void) {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t e) {
  (void)e;
  return "error of the test's runtime";
}
hipError_t hipStreamCreate(hipStream_t* s) {
  static int token;
  *s = (hipStream_t)&token;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  (void)s;
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) {
  static int token;
  *e = (hipEvent_t)&token;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned f) {
  (void)f;
  return hipEventCreate(e);
}
hipError_t hipEventDestroy(hipEvent_t e) {
  (void)e;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  (void)e, (void)s;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  (void)e;
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
  (void)a, (void)b;
  *ms = 0.0f;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode m) {
  (void)s, (void)m;
  capturing = 1;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
  static int token;
  (void)s;
  capturing = 0;
  *g = (hipGraph_t)&token;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t g, hipGraphNode_t* n, char* log,
                               size_t sz) {
  static int token;
  (void)g, (void)n, (void)log, (void)sz;
  *x = (hipGraphExec_t)&token;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t s) {
  (void)x, (void)s;
  ++fake_pending;
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
  (void)g;
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x) {
  (void)x;
  return hipSuccess;
}
