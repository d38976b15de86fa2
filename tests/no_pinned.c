/* Pinned host memory refused beyond a size: answers hipHostMalloc before the
 * HIP runtime does (loaded with RTLD_GLOBAL ahead of libgpuseed.so), and
 * counts what it refused. */
#define _GNU_SOURCE
#define __HIP_PLATFORM_AMD__ 1
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

static size_t limit;
static int refused;
void no_pinned_limit(size_t bytes) { limit = bytes; }
int no_pinned_refused(void) { return refused; }

hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) {
  static hipError_t (*real)(void**, size_t, unsigned);
  Dl_info hip;  /* the runtime's library, found by another of its functions */
  if (!real && dladdr((void*)hipHostFree, &hip)) real = dlsym(dlopen(hip.dli_fname, RTLD_LAZY), "hipHostMalloc");
  if (n > limit || !real) {
    ++refused;
    return hipErrorOutOfMemory;
  }
  return real(p, n, flags);
}
