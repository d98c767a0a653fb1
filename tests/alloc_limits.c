/* hipMalloc and hipHostMalloc that fail from a size on, as when the memory has run out,
 * and a count of what is allocated (loaded RTLD_GLOBAL before librespack_gpu.so, so that its
 * calls come here). */
#include <dlfcn.h>
#include <stddef.h>
#include <stdint.h>

static size_t device_limit = SIZE_MAX, host_limit = SIZE_MAX;
static int refused;
static struct {
  void* p;
  size_t n;
} live[4096];

/* largest sizes that still succeed */
void alloc_limits(size_t device, size_t host) {
  device_limit = device;
  host_limit = host;
}

int alloc_refused(void) { return refused; }

/* bytes of device memory allocated and not yet freed */
size_t alloc_live(void) {
  size_t n = 0;
  for (int i = 0; i < 4096; ++i) n += live[i].n;
  return n;
}

static void note(void* was, void* p, size_t n) {
  for (int i = 0; i < 4096; ++i)
    if (live[i].p == was) {
      live[i].p = p;
      live[i].n = n;
      return;
    }
}

static void* real(const char* name) { return dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY), name); }

int hipMalloc(void** p, size_t n) {
  if (n > device_limit) {
    ++refused;
    return 2; /* hipErrorOutOfMemory */
  }
  const int e = ((int (*)(void**, size_t))real("hipMalloc"))(p, n);
  if (e == 0) note(NULL, *p, n);
  return e;
}

int hipFree(void* p) {
  if (p) note(p, NULL, 0);
  return ((int (*)(void*))real("hipFree"))(p);
}

int hipHostMalloc(void** p, size_t n, unsigned flags) {
  if (n > host_limit) {
    ++refused;
    return 2;
  }
  return ((int (*)(void**, size_t, unsigned))real("hipHostMalloc"))(p, n, flags);
}
