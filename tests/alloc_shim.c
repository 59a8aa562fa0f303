/* alloc_shim.c -- hipMalloc, hipFree and hipHostMalloc of the HIP runtime with
 * a limit on the device memory that may be taken, pinned memory that can be
 * refused, and a record of both (tests/alloc_child.py).  Loaded with global
 * symbols before libpicgpu.so, whose calls then come here.  No call reaches
 * the device that the runtime would not have made itself; a refused one does
 * not reach it at all.  One thread at a time. */
#include <dlfcn.h>
#include <stddef.h>
#include <stdint.h>

enum { kOutOfMemory = 2, kMax = 4096 }; /* hipErrorOutOfMemory */

static void *sym(const char *name) {
  static void *rt;
  if (!rt) rt = dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_LOCAL);
  return rt ? dlsym(rt, name) : NULL;
}

static struct { void *p; size_t n; } live[kMax];
static int64_t limit = -1, used, peak; /* limit < 0: none */
static int refuse_host;
static unsigned host_flags;
static int64_t host_calls;

void shim_limit(int64_t bytes) { limit = bytes; }
void shim_peak_reset(void) { peak = used; }
int64_t shim_used(void) { return used; }
int64_t shim_peak(void) { return peak; }
void shim_refuse_host(int on) { refuse_host = on; }
unsigned shim_host_flags(void) { return host_flags; }
int64_t shim_host_calls(void) { return host_calls; }

int hipMalloc(void **p, size_t n) {
  int (*real)(void **, size_t) = (int (*)(void **, size_t))sym("hipMalloc");
  int k = 0;
  if (!real || (limit >= 0 && used + (int64_t)n > limit)) return kOutOfMemory;
  while (k < kMax && live[k].p) ++k;
  if (k == kMax) return kOutOfMemory;
  const int e = real(p, n);
  if (e) return e;
  live[k].p = *p;
  live[k].n = n;
  used += (int64_t)n;
  if (used > peak) peak = used;
  return 0;
}

int hipFree(void *p) {
  int (*real)(void *) = (int (*)(void *))sym("hipFree");
  for (int k = 0; k < kMax && p; ++k)
    if (live[k].p == p) {
      used -= (int64_t)live[k].n;
      live[k].p = NULL;
      break;
    }
  return real ? real(p) : kOutOfMemory;
}

int hipHostMalloc(void **p, size_t n, unsigned flags) {
  int (*real)(void **, size_t, unsigned) = (int (*)(void **, size_t, unsigned))sym("hipHostMalloc");
  ++host_calls;
  host_flags = flags;
  if (!real || refuse_host) return kOutOfMemory;
  return real(p, n, flags);
}
