/* Loaded before libtwmc_hip.so with RTLD_GLOBAL: its allocations go through these, which
 * return hipErrorOutOfMemory without asking the runtime where the test says so. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>

enum { kOutOfMemory = 2 };

static size_t device_limit = (size_t)-1;
static int pinned_fails = 0;
static int failed = 0;

void fail_device_above(size_t bytes) { device_limit = bytes; }
void fail_pinned(int on) { pinned_fails = on; }
int failures(void) { return failed; }

static void* next_symbol(const char* name) {
  void* hip = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
  return hip ? dlsym(hip, name) : NULL;
}

int hipMalloc(void** p, size_t bytes) {
  if (bytes > device_limit) {
    ++failed;
    *p = NULL;
    return kOutOfMemory;
  }
  return ((int (*)(void**, size_t))next_symbol("hipMalloc"))(p, bytes);
}

int hipHostMalloc(void** p, size_t bytes, unsigned flags) {
  if (pinned_fails) {
    ++failed;
    return kOutOfMemory;
  }
  return ((int (*)(void**, size_t, unsigned))next_symbol("hipHostMalloc"))(p, bytes, flags);
}
