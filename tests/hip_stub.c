/* Stand-ins for the HIP calls that context creation and kernel launches make, so
 * that a failing allocation can be followed without a GPU: allocations come from
 * the host, launches do nothing.  Preloaded before libphlx.so. */
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

static int countdown = -1, allocs = 0, last = 0;
void stub_fail_after(int n) { countdown = n; } /* the n-th next allocation fails; -1: none */
int stub_allocs(void) { return allocs; }

int hipSetDevice(int d) { (void)d; return 0; }
int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; *s = (void *)8; return 0; }
int hipStreamDestroy(void *s) { (void)s; return 0; }
int hipStreamSynchronize(void *s) { (void)s; return 0; }
int hipMalloc(void **p, size_t n) {
  if (countdown >= 0 && countdown-- == 0) return last = 2;  /* hipErrorOutOfMemory */
  *p = malloc(n);
  allocs++;
  return 0;
}
int hipFree(void *p) { free(p); return 0; }
int hipMemsetAsync(void *p, int v, size_t n, void *s) { (void)s; memset(p, v, n); return 0; }
int hipMemcpyAsync(void *d, const void *h, size_t n, int k, void *s) {
  (void)k; (void)s;
  memcpy(d, h, n);
  return 0;
}
int hipGetLastError(void) { int e = last; last = 0; return e; }
typedef struct { unsigned x, y, z; } dim3_;
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t m, void *s) {
  (void)g; (void)b; (void)m; (void)s;
  return 0;
}
int __hipPopCallConfiguration(dim3_ *g, dim3_ *b, size_t *m, void **s) {
  dim3_ one = {1, 1, 1};
  *g = *b = one;
  *m = 0;
  *s = 0;
  return 0;
}
int hipLaunchKernel(const void *f, dim3_ g, dim3_ b, void **a, size_t m, void *s) {
  (void)f; (void)g; (void)b; (void)a; (void)m; (void)s;
  return 0;
}
