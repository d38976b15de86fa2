/* A stand-in for the HIP runtime, for tests of the library's host code on a
 * machine without a GPU: device memory is host memory (zeroed), copies are
 * memcpy, kernels do nothing, and allocations can be counted, limited and made
 * to fail.  A failed call leaves its error for hipGetLastError, as HIP's do.
 * Loaded with RTLD_GLOBAL before libgpuseed.so, whose calls it then answers. */
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <pthread.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#define EXPORT __attribute__((visibility("default")))

typedef struct Block {
  struct Block* next;
  void* p;
  size_t bytes;
} Block;

static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static Block* blocks[2];  /* 0: device, 1: pinned host */
static uint64_t held[2], calls[2];
static uint64_t total_limit[2] = {~0ull, ~0ull}; /* bytes that may be held */
static uint64_t block_limit[2] = {~0ull, ~0ull}; /* bytes of one allocation */
static __thread hipError_t last_error = hipSuccess;
static uint64_t chain_rows; /* rows that direct_chains reports as visited */
static const void* chains_stub;

/* what the tests see and set (kind 0: device, 1: pinned host memory) */
EXPORT uint64_t fake_held(int kind) { return held[kind]; }
EXPORT uint64_t fake_calls(int kind) { return calls[kind]; }
EXPORT void fake_limit(int kind, uint64_t total, uint64_t block) {
  total_limit[kind] = total;
  block_limit[kind] = block;
}
EXPORT void fake_chain_rows(uint64_t rows) { chain_rows = rows; }

static hipError_t fail(hipError_t e) {
  last_error = e;
  return e;
}

static hipError_t get(int kind, void** out, size_t bytes) {
  hipError_t e = hipSuccess;
  pthread_mutex_lock(&mu);
  ++calls[kind];
  Block* b = NULL;
  void* p = NULL;
  if (bytes > block_limit[kind] || held[kind] + bytes > total_limit[kind] || !(b = malloc(sizeof *b)) ||
      !(p = calloc(bytes / 64 + 1, 64))) {
    free(b);
    e = hipErrorOutOfMemory;
  } else {
    b->p = p;
    b->bytes = bytes;
    b->next = blocks[kind];
    blocks[kind] = b;
    held[kind] += bytes;
    *out = p;
  }
  pthread_mutex_unlock(&mu);
  return e == hipSuccess ? e : fail(e);
}

static hipError_t put(int kind, void* p) {
  if (!p) return hipSuccess;
  hipError_t e = hipErrorInvalidValue;
  pthread_mutex_lock(&mu);
  for (Block** q = &blocks[kind]; *q; q = &(*q)->next)
    if ((*q)->p == p) {
      Block* b = *q;
      *q = b->next;
      held[kind] -= b->bytes;
      free(b->p);
      free(b);
      e = hipSuccess;
      break;
    }
  pthread_mutex_unlock(&mu);
  return e == hipSuccess ? e : fail(e);
}

EXPORT hipError_t hipMalloc(void** p, size_t n) { return get(0, p, n); }
EXPORT hipError_t hipFree(void* p) { return put(0, p); }
EXPORT hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) { return get(1, p, n); }
EXPORT hipError_t hipHostFree(void* p) { return put(1, p); }
EXPORT hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) {
  if (n) memcpy(d, s, n);
  return hipSuccess;
}
EXPORT hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t st) {
  return hipMemcpy(d, s, n, k);
}
EXPORT hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t st) {
  memset(d, v, n);
  return hipSuccess;
}
EXPORT hipError_t hipGetLastError(void) {
  hipError_t e = last_error;
  last_error = hipSuccess;
  return e;
}
EXPORT hipError_t hipPeekAtLastError(void) { return last_error; }

EXPORT hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
EXPORT hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
EXPORT hipError_t hipSetDevice(int d) { return hipSuccess; }
EXPORT hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int d) {
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  p->warpSize = 64;
  return hipSuccess;
}
EXPORT hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int d) {
  *v = 256;
  return hipSuccess;
}
EXPORT hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int block, size_t lds) {
  *n = 8;
  return hipSuccess;
}
EXPORT int hipGetStreamDeviceId(hipStream_t st) { return 0; }
EXPORT hipError_t hipDeviceSynchronize(void) { return hipSuccess; }

static uint64_t handle; /* every stream, event and graph */
EXPORT hipError_t hipStreamCreate(hipStream_t* st) { *st = (hipStream_t)&handle; return hipSuccess; }
EXPORT hipError_t hipStreamCreateWithFlags(hipStream_t* st, unsigned f) { return hipStreamCreate(st); }
EXPORT hipError_t hipStreamDestroy(hipStream_t st) { return hipSuccess; }
EXPORT hipError_t hipStreamSynchronize(hipStream_t st) { return hipSuccess; }
EXPORT hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)&handle; return hipSuccess; }
EXPORT hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned f) { return hipEventCreate(e); }
EXPORT hipError_t hipEventDestroy(hipEvent_t e) { return hipSuccess; }
EXPORT hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) { return hipSuccess; }
EXPORT hipError_t hipEventSynchronize(hipEvent_t e) { return hipSuccess; }
EXPORT hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) { *ms = 0; return hipSuccess; }

/* the library's fixed device array */
EXPORT hipError_t hipGetSymbolAddress(void** p, const void* symbol) {
  static void* array;
  if (!array) array = calloc(1, 256u << 20);
  *p = array;
  return array ? hipSuccess : fail(hipErrorOutOfMemory);
}

/* kernels: registered by name, launched as nothing */
static uint64_t module;
EXPORT void** __hipRegisterFatBinary(const void* data) { return (void**)&module; }
EXPORT void __hipUnregisterFatBinary(void** m) {}
EXPORT void __hipRegisterVar(void** m, void* var, char* hv, char* dv, int ext, size_t size, int constant, int global) {}
EXPORT void __hipRegisterFunction(void** m, const void* stub, char* name, const char* dname, unsigned limit, void* tid,
                                  void* bid, void* bdim, void* gdim, int* wsize) {
  if (strstr(dname, "direct_chains")) chains_stub = stub;
}
static __thread struct {
  dim3 grid, block;
  size_t lds;
  hipStream_t st;
} call;
EXPORT hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t st) {
  call.grid = grid;
  call.block = block;
  call.lds = lds;
  call.st = st;
  return hipSuccess;
}
EXPORT hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* st) {
  *grid = call.grid;
  *block = call.block;
  *lds = call.lds;
  *st = call.st;
  return hipSuccess;
}
EXPORT hipError_t hipLaunchKernel(const void* stub, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t st) {
  if (stub == chains_stub) { /* {.., uint32_t* err}: rows visited in err[2..3] */
    uint32_t* err = *(uint32_t**)args[6];
    err[2] = (uint32_t)chain_rows;
    err[3] = (uint32_t)(chain_rows >> 32);
  }
  return hipSuccess;
}
EXPORT hipError_t hipStreamBeginCapture(hipStream_t st, hipStreamCaptureMode m) { return hipSuccess; }
EXPORT hipError_t hipStreamEndCapture(hipStream_t st, hipGraph_t* g) { *g = (hipGraph_t)&handle; return hipSuccess; }
EXPORT hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t g, hipGraphNode_t* n, char* log, size_t size) {
  *x = (hipGraphExec_t)&handle;
  return hipSuccess;
}
EXPORT hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t st) { return hipSuccess; }
EXPORT hipError_t hipGraphExecDestroy(hipGraphExec_t x) { return hipSuccess; }
EXPORT hipError_t hipGraphDestroy(hipGraph_t g) { return hipSuccess; }
