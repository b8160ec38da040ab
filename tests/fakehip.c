/* A HIP runtime without a device, for host-side tests of libmw3: memory is
 * counted and never touched, kernels and copies do nothing, captures give empty
 * graphs.  What the library does is logged, one letter per call:
 *   K kernel launch (k while capturing)   C begin of a capture   I instantiation
 *   w wait of one stream for another while capturing
 *   G graph launch                        T record of a timing event
 * Loaded with global symbols before the library, its functions take the place of
 * the runtime's. */
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

typedef struct { uint32_t x, y, z; } dim3_t;
typedef int err_t;

enum { NLOG = 1 << 22, NMEM = 1 << 14 };
static char logbuf[NLOG];
static int nlog, capturing;
static struct { uintptr_t p; size_t n; } mem[NMEM];
static size_t bytes;
static uintptr_t next = 0x700000000000u;

static void put(char c) {
  if (nlog < NLOG - 1) logbuf[nlog++] = c;
}
const char *fake_log(void) {
  logbuf[nlog] = 0;
  return logbuf;
}
void fake_log_clear(void) { nlog = 0; }
size_t fake_bytes(void) { return bytes; }

err_t hipMalloc(void **p, size_t n) {
  for (int i = 0; i < NMEM; i++)
    if (!mem[i].p) {
      mem[i].p = next;
      mem[i].n = n;
      *p = (void *)next;
      next += (n + 511) / 256 * 256;
      bytes += n;
      return 0;
    }
  return 2;
}
err_t hipFree(void *p) {
  for (int i = 0; p && i < NMEM; i++)
    if (mem[i].p == (uintptr_t)p) {
      bytes -= mem[i].n;
      mem[i].p = 0;
    }
  return 0;
}
err_t hipMemcpy(void *d, const void *s, size_t n, int k) { return 0; }
err_t hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) { return 0; }
err_t hipMemset(void *d, int v, size_t n) { return 0; }

err_t hipGetDeviceCount(int *n) { *n = 1; return 0; }
err_t hipGetDevice(int *d) { *d = 0; return 0; }
err_t hipDeviceGetAttribute(int *v, int a, int d) { *v = 256; return 0; }
err_t hipGetLastError(void) { return 0; }
const char *hipGetErrorString(err_t e) { return "no error"; }
err_t hipGetSymbolAddress(void **p, const void *s) { *p = (void *)0x600000000000u; return 0; }
err_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t s) {
  *n = 2;
  return 0;
}

err_t hipFuncGetAttributes(void *a, const void *f) { memset(a, 0, 56); return 0; }

err_t hipStreamCreateWithFlags(void **s, unsigned f) { *s = malloc(1); return 0; }
err_t hipStreamDestroy(void *s) { free(s); return 0; }
err_t hipStreamSynchronize(void *s) { return 0; }
err_t hipStreamWaitEvent(void *s, void *e, unsigned f) {
  if (capturing) put('w');
  return 0;
}
err_t hipStreamBeginCapture(void *s, int m) { capturing = 1; put('C'); return 0; }
err_t hipStreamEndCapture(void *s, void **g) { capturing = 0; *g = malloc(1); return 0; }
err_t hipGraphInstantiate(void **x, void *g, void *n, char *b, size_t l) {
  put('I');
  *x = malloc(1);
  return 0;
}
err_t hipGraphDestroy(void *g) { free(g); return 0; }
err_t hipGraphExecDestroy(void *x) { free(x); return 0; }
err_t hipGraphLaunch(void *x, void *s) { put('G'); return 0; }

static err_t event(void **e, char timing) {
  *e = malloc(1);
  *(char *)*e = timing;
  return 0;
}
err_t hipEventCreate(void **e) { return event(e, 1); }
err_t hipEventCreateWithFlags(void **e, unsigned f) { return event(e, 0); }
err_t hipEventDestroy(void *e) { free(e); return 0; }
err_t hipEventRecord(void *e, void *s) {
  if (*(char *)e) put('T');
  return 0;
}
err_t hipEventSynchronize(void *e) { return 0; }
err_t hipEventElapsedTime(float *ms, void *a, void *b) { *ms = 1.0f; return 0; }

static struct { dim3_t g, b; size_t sh; void *st; } call;
err_t __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t sh, void *st) {
  call.g = g, call.b = b, call.sh = sh, call.st = st;
  return 0;
}
err_t __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *sh, void **st) {
  *g = call.g, *b = call.b, *sh = call.sh, *st = call.st;
  return 0;
}
static struct { const void *f; const char *name; unsigned grid; } fun[1024];
static int nfun;
/* blocks of the last launch of a kernel whose (mangled) name has `part`, or 0 */
unsigned fake_grid(const char *part) {
  unsigned g = 0;
  for (int i = 0; i < nfun; i++)
    if (fun[i].grid && strstr(fun[i].name, part)) g = fun[i].grid;
  for (int i = 0; i < nfun; i++) fun[i].grid = 0;
  return g;
}
err_t hipLaunchKernel(const void *f, dim3_t g, dim3_t b, void **args, size_t sh, void *st) {
  put(capturing ? 'k' : 'K');
  for (int i = 0; i < nfun; i++)
    if (fun[i].f == f) fun[i].grid = g.x;
  return g.x && g.y && g.z && b.x ? 0 : 9;
}
void **__hipRegisterFatBinary(const void *d) { return malloc(8); }
void __hipUnregisterFatBinary(void **m) { free(m); }
void __hipRegisterFunction(void **m, const void *f, char *d, const char *n, unsigned t, void *a,
                           void *b, void *c, void *e, int *w) {
  if (nfun < 1024) fun[nfun].f = f, fun[nfun++].name = n;
}
void __hipRegisterVar(void **m, void *v, char *h, char *n, int e, size_t s, int c, int g) {}
