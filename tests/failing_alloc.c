/* For tests: loaded before the engine's library (RTLD_GLOBAL), stands in front
 * of the runtime's allocating calls, counts them and lets one chosen call ask
 * for more memory than any device has, so that it fails as it does on a full
 * one. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>

static long calls[3], chosen[3] = {-1, -1, -1};

static size_t ask(int kind, size_t bytes) {
  const long call = __atomic_fetch_add(&calls[kind], 1, __ATOMIC_SEQ_CST);
  return call == __atomic_load_n(&chosen[kind], __ATOMIC_SEQ_CST) ? (size_t)1 << 50 : bytes;
}

static void* real(const char* name) {
  return dlsym(dlopen("libamdhip64.so.7", RTLD_NOLOAD | RTLD_LAZY), name);
}

/* Start counting kind 0 (device memory), 1 (pinned memory) or 2 (the free
 * memory's size) from zero; call number `call` is to fail (-1: none). */
void fail_alloc(int kind, long call) {
  __atomic_store_n(&chosen[kind], call, __ATOMIC_SEQ_CST);
  __atomic_store_n(&calls[kind], 0, __ATOMIC_SEQ_CST);
}

long alloc_calls(int kind) { return __atomic_load_n(&calls[kind], __ATOMIC_SEQ_CST); }

int hipMalloc(void** p, size_t bytes) {
  return ((int (*)(void**, size_t))real("hipMalloc"))(p, ask(0, bytes));
}

int hipHostMalloc(void** p, size_t bytes, unsigned flags) {
  return ((int (*)(void**, size_t, unsigned))real("hipHostMalloc"))(p, ask(1, bytes), flags);
}

int hipMemGetInfo(size_t* free_bytes, size_t* total) {
  if (ask(2, 0)) return 1;
  return ((int (*)(size_t*, size_t*))real("hipMemGetInfo"))(free_bytes, total);
}
