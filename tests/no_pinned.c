/* Pinned host memory refused beyond a size, and device memory of a range of
 * sizes: answers hipHostMalloc and hipMalloc before the HIP runtime does
 * (loaded with RTLD_GLOBAL ahead of libgpuseed.so), and counts what it
 * refused. */
#define _GNU_SOURCE
#define __HIP_PLATFORM_AMD__ 1
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

static size_t limit, refuse_lo = 1, refuse_hi;
static int refused;
void no_pinned_limit(size_t bytes) { limit = bytes; }
void no_device_between(size_t lo, size_t hi) {
  refuse_lo = lo;
  refuse_hi = hi;
}
int no_pinned_refused(void) { return refused; }

static void* runtimes(const char* name) { /* the runtime's own, found by another of its functions */
  Dl_info hip;
  return dladdr((void*)hipHostFree, &hip) ? dlsym(dlopen(hip.dli_fname, RTLD_LAZY), name) : 0;
}

hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) {
  static hipError_t (*real)(void**, size_t, unsigned);
  if (!real) real = runtimes("hipHostMalloc");
  if (n > limit || !real) {
    ++refused;
    return hipErrorOutOfMemory;
  }
  return real(p, n, flags);
}

hipError_t hipMalloc(void** p, size_t n) {
  static hipError_t (*real)(void**, size_t);
  if (!real) real = runtimes("hipMalloc");
  if ((n >= refuse_lo && n <= refuse_hi) || !real) {
    ++refused;
    return hipErrorOutOfMemory;
  }
  return real(p, n);
}
