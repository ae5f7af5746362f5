/* Arena (csrc/gp_arena.h) on host memory: hipMalloc and hipFree are those below, with a limit on the bytes. */
#include <stdint.h>
#include <stdlib.h>

#include "gp_arena.h"

static size_t g_limit, g_asked, g_live;
static hipError_t g_last = hipSuccess;
extern "C" hipError_t hipMalloc(void **p, size_t n) {
  g_asked = n;
  *p = n <= g_limit ? aligned_alloc(256, (n + 255) & ~(size_t)255) : nullptr;
  if (!*p) return g_last = hipErrorOutOfMemory;
  g_live++;
  return hipSuccess;
}
extern "C" hipError_t hipFree(void *p) {
  if (p) g_live--;
  free(p);
  return hipSuccess;
}
extern "C" hipError_t hipGetLastError(void) {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}

/* two buffers of n bytes with `limit` bytes of memory, up to `tries` times with the last one at the limit: the bytes
 * asked for by the last try, or a negative code of what is wrong */
extern "C" int64_t arena_check(int64_t n, int tries) {
  {
    Arena a;
    char *p, *q;
    for (int t = 0; t < tries; t++) {
      const bool last = t == tries - 1;
      g_limit = last ? (size_t)(2 * ((n + 255) & ~(int64_t)255)) : (size_t)n;
      a.take(&p, (size_t)n);
      a.take(&q, (size_t)n);
      if (a.allocate() != last) return -1;
      if (hipGetLastError() != hipSuccess) return -2;
      if (!last && (p || q || a.base() || a.size())) return -3;
    }
    if (p != a.base() || q < p + n || ((uintptr_t)q & 255)) return -4;
    p[n - 1] = q[n - 1] = 1;
  }
  return g_live ? -5 : (int64_t)g_asked;
}
