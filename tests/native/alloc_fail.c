/* Loaded before libtwmc_hip.so with RTLD_GLOBAL: its allocations go through these.  Where
 * the test says so they ask the runtime for 2^60 bytes instead, which it refuses on the
 * host, so that its error state is that of a real failure. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>

static size_t device_limit = (size_t)-1;
static int pinned_fails = 0;
static int failed = 0;

void fail_device_above(size_t bytes) { device_limit = bytes; }
void fail_pinned(int on) { pinned_fails = on; }
int failures(void) { return failed; }

static size_t size_of(size_t bytes, int fails) {
  failed += fails;
  return fails ? (size_t)1 << 60 : bytes;
}

static void* next_symbol(const char* name) {
  return dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD), name);
}

int hipMalloc(void** p, size_t bytes) {
  return ((int (*)(void**, size_t))next_symbol("hipMalloc"))(p, size_of(bytes, bytes > device_limit));
}

int hipHostMalloc(void** p, size_t bytes, unsigned flags) {
  return ((int (*)(void**, size_t, unsigned))next_symbol("hipHostMalloc"))(p, size_of(bytes, pinned_fails), flags);
}
