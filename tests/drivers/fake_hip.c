/* Host-side stand-in for the few HIP runtime calls of an upload, for tests
 * without a GPU: device memory is host memory, kernels do nothing, and the
 * test sees which device has work in flight and whether a copy went outside
 * every allocation. */
#include <stdlib.h>
#include <string.h>

enum { MAXB = 4096, NDEV = 2 };
static struct { char *p; size_t n; } blocks[MAXB];
static int nblocks, current, busy[NDEV], fail_at = -1, fail_host_at = -1, bad_copies, copies, last;

void fake_device(int d) { current = d; }
int fake_current(void) { return current; }
int fake_busy(int d) { return busy[d]; }
void fake_fail_at(int n) { fail_at = n; } /* the n-th hipMalloc from now fails (0: the next) */
void fake_fail_host_at(int n) { fail_host_at = n; } /* the same for hipHostMalloc */
int fake_bad_copies(void) { return bad_copies; }
int fake_copies(void) { return copies; }

int hipGetDevice(int *d) { *d = current; return 0; }
int hipSetDevice(int d) { current = d; return 0; }
int hipSetDeviceFlags(unsigned f) { (void)f; return 0; }
int hipGetLastError(void) {
  const int e = last;
  last = 0;
  return e;
}
const char *hipGetErrorString(int e) { return e ? "fake error" : "no error"; }
int hipDeviceSynchronize(void) { busy[current] = 0; return 0; }
int hipStreamSynchronize(void *st) { (void)st; busy[current] = 0; return 0; }
int hipMemGetInfo(size_t *a, size_t *t) { *a = *t = (size_t)1 << 30; return 0; }

static int put(void **p, size_t n) {
  *p = calloc(1, n);
  if (nblocks == MAXB || !*p) return 2;
  blocks[nblocks].p = *p;
  blocks[nblocks++].n = n;
  return 0;
}
static int drop(void *p) {
  for (int k = 0; k < nblocks; k++)
    if (blocks[k].p == p) {
      blocks[k] = blocks[--nblocks];
      free(p);
      return 0;
    }
  return 1;
}
int hipMalloc(void **p, size_t n) {
  *p = 0;
  if (fail_at >= 0 && fail_at-- == 0) return last = 2;
  return put(p, n);
}
int hipFree(void *p) { return drop(p); }
int hipHostMalloc(void **p, size_t n, unsigned f) {
  (void)f;
  *p = 0;
  if (fail_host_at >= 0 && fail_host_at-- == 0) return last = 2;
  return put(p, n);
}
int hipHostFree(void *p) { return drop(p); }
static int inside(const char *p, size_t n) {
  for (int k = 0; k < nblocks; k++)
    if (p >= blocks[k].p && p + n <= blocks[k].p + blocks[k].n) return 1;
  return 0;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st) {
  (void)kind, (void)st;
  busy[current] = 1;
  copies++;
  if (inside(d, n)) memcpy(d, s, n);
  else bad_copies++;
  return 0;
}
int hipMemcpy(void *d, const void *s, size_t n, int kind) { return hipMemcpyAsync(d, s, n, kind, 0); }
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; *e = (void *)1; return 0; }
int hipEventRecord(void *e, void *st) { (void)e, (void)st; return 0; }
int hipEventSynchronize(void *e) { (void)e; return 0; }
int hipEventDestroy(void *e) { (void)e; return 0; }
int __hipPushCallConfiguration(void) { return 0; }
int __hipPopCallConfiguration(void) { return 0; }
int hipLaunchKernel(void) { busy[current] = 1; return 0; }
