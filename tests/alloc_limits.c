/* hipMalloc and hipHostMalloc that fail from a size on, as when the memory has run out
 * (loaded RTLD_GLOBAL before librespack_gpu.so, so that its calls come here). */
#include <dlfcn.h>
#include <stddef.h>
#include <stdint.h>

static size_t device_limit = SIZE_MAX, host_limit = SIZE_MAX;
static int refused;

/* largest sizes that still succeed */
void alloc_limits(size_t device, size_t host) {
  device_limit = device;
  host_limit = host;
}

int alloc_refused(void) { return refused; }

static void* real(const char* name) { return dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY), name); }

int hipMalloc(void** p, size_t n) {
  if (n > device_limit) {
    ++refused;
    return 2; /* hipErrorOutOfMemory */
  }
  return ((int (*)(void**, size_t))real("hipMalloc"))(p, n);
}

int hipHostMalloc(void** p, size_t n, unsigned flags) {
  if (n > host_limit) {
    ++refused;
    return 2;
  }
  return ((int (*)(void**, size_t, unsigned))real("hipHostMalloc"))(p, n, flags);
}
