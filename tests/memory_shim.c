/* Device allocations counted and limited, for test_memory.py: loaded before
 * the engine, its hipMalloc, hipFree and hipMemGetInfo come before the
 * runtime's in the engine's symbol lookup. */
#include <pthread.h>
#include <stddef.h>
#include <unistd.h>

enum { kSlots = 1 << 16, kOutOfMemory = 2 };
static struct { void* p; size_t n; } slot[kSlots];
static size_t used, peak, limit;
static int report, wait_us;
static int (*real_malloc)(void**, size_t);
static int (*real_free)(void*);
static int (*real_info)(size_t*, size_t*);
static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;

void shim_init(void* m, void* f, void* i) {
  real_malloc = (int (*)(void**, size_t))m;
  real_free = (int (*)(void*))f;
  real_info = (int (*)(size_t*, size_t*))i;
}
/* bytes: of a device that the engine seems to have (0: no limit); r: whether
 * hipMemGetInfo says so too */
void shim_limit(size_t bytes, int r) { limit = bytes; report = r; }
/* hipMemGetInfo takes so long to answer */
void shim_wait(int us) { wait_us = us; }
size_t shim_used(void) { return used; }
size_t shim_peak(int reset) {
  const size_t p = peak;
  if (reset) peak = used;
  return p;
}

int hipMalloc(void** p, size_t n) {
  pthread_mutex_lock(&mu);
  int rc = kOutOfMemory;
  if (!limit || used + n <= limit) rc = real_malloc(p, n);
  if (rc == 0) {
    size_t s = ((size_t)*p >> 8) % kSlots;
    while (slot[s].p) s = (s + 1) % kSlots;
    slot[s].p = *p;
    slot[s].n = n;
    used += n;
    if (used > peak) peak = used;
  }
  pthread_mutex_unlock(&mu);
  return rc;
}

int hipFree(void* p) {
  pthread_mutex_lock(&mu);
  for (size_t s = 0; p && s < kSlots; ++s)
    if (slot[s].p == p) {
      used -= slot[s].n;
      slot[s].p = NULL;
      break;
    }
  pthread_mutex_unlock(&mu);
  return real_free(p);
}

int hipMemGetInfo(size_t* idle, size_t* total) {
  const int rc = real_info(idle, total);
  if (rc == 0 && limit && report) {
    *total = limit;
    *idle = limit > used ? limit - used : 0;
  }
  if (wait_us) usleep(wait_us);
  return rc;
}
