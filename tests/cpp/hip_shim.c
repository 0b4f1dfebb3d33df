/* Stands in front of a few HIP calls of the engine (load it RTLD_GLOBAL before
 * libhrt.so): device memory with a limit, past which an allocation fails as on
 * a full card, and the names of the kernels that are launched. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <pthread.h>
#include <stddef.h>
#include <stdint.h>
#include <string.h>

enum { kOutOfMemory = 2, kBlocks = 4096, kNames = 1 << 16 };
typedef struct { uint32_t x, y, z; } dim3_t;

static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static size_t limit = SIZE_MAX, used;
static uint64_t calls, refused;
static struct { void* p; size_t n; } block[kBlocks];
static char names[kNames];

static void* real(const char* name) {
  static void* lib;
  if (!lib) lib = dlopen("libamdhip64.so.7", RTLD_NOW);
  return lib ? dlsym(lib, name) : NULL;
}

static int room(size_t n) {
  pthread_mutex_lock(&mu);
  calls++;
  const int ok = used + n <= limit;
  if (!ok) refused++;
  pthread_mutex_unlock(&mu);
  return ok;
}
static void note(void* p, size_t n) {
  pthread_mutex_lock(&mu);
  for (int k = 0; k < kBlocks; k++)
    if (!block[k].p) {
      block[k].p = p;
      block[k].n = n;
      used += n;
      break;
    }
  pthread_mutex_unlock(&mu);
}
static void forget(void* p) {
  pthread_mutex_lock(&mu);
  for (int k = 0; p && k < kBlocks; k++)
    if (block[k].p == p) {
      used -= block[k].n;
      block[k].p = NULL;
      break;
    }
  pthread_mutex_unlock(&mu);
}

int hipMalloc(void** p, size_t n) {
  if (!room(n)) return kOutOfMemory;
  const int e = ((int (*)(void**, size_t))real("hipMalloc"))(p, n);
  if (!e) note(*p, n);
  return e;
}
int hipMallocAsync(void** p, size_t n, void* stream) {
  if (!room(n)) return kOutOfMemory;
  const int e = ((int (*)(void**, size_t, void*))real("hipMallocAsync"))(p, n, stream);
  if (!e) note(*p, n);
  return e;
}
int hipFree(void* p) {
  forget(p);
  return ((int (*)(void*))real("hipFree"))(p);
}
int hipFreeAsync(void* p, void* stream) {
  forget(p);
  return ((int (*)(void*, void*))real("hipFreeAsync"))(p, stream);
}
int hipLaunchKernel(const void* fn, dim3_t grid, dim3_t group, void** args, size_t lds, void* stream) {
  const char* name = ((const char* (*)(const void*, void*))real("hipKernelNameRefByPtr"))(fn, stream);
  pthread_mutex_lock(&mu);
  if (name && strlen(names) + strlen(name) + 2 < kNames) strcat(strcat(names, name), "\n");
  pthread_mutex_unlock(&mu);
  return ((int (*)(const void*, dim3_t, dim3_t, void**, size_t, void*))real("hipLaunchKernel"))(fn, grid, group, args,
                                                                                               lds, stream);
}

void shim_limit(size_t bytes) { limit = bytes; }
size_t shim_used(void) { return used; }
uint64_t shim_calls(void) { return calls; }
uint64_t shim_refused(void) { return refused; }
const char* shim_names(void) { return names; }
void shim_clear_names(void) { names[0] = 0; }
