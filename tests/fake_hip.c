/* A stand-in for the HIP runtime, for tests of the host driver's error paths
 * on a machine without a GPU: device memory is host memory, streams run
 * nothing, and calls can be told to fail.  Loaded before libtm_hip.so with
 * global visibility, its functions take the runtime's place.  Pinned memory is
 * unmapped when freed, so that a use after it ends the process. */
#define _GNU_SOURCE
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>
#include "tm_types.h"

#define MAXK 4096
#define MAXS 64
#define MAXA 65536
static struct { const void *f; char name[256]; } kern[MAXK];
static int nkern;
static struct { void *p; size_t n; int host; } mem[MAXA];
static int pending[MAXS], nstream;   /* launches and copies not waited for, per stream */
static hipError_t last;
static size_t used, peak, limit = (size_t)-1;
static char fail_kernel[64];
static int fail_kernel_after, fail_host, fail_record, fail_sync, fail_stream, fail_query;
static unsigned long long head_pairs;
static int word_on, word;           /* what a 4-byte copy to the host brings */
static char trace[1 << 16];
static tm_kernel_args mined;       /* of the last mining launch */

void fake_fail_kernel(const char *part, int after) { snprintf(fail_kernel, sizeof fail_kernel, "%s", part); fail_kernel_after = after; }
void fake_fail_host(int on) { fail_host = on; }
void fake_fail_record(int on) { fail_record = on; }
void fake_fail_sync(int stream) { fail_sync = 1; fail_stream = stream; }
void fake_fail_query(int n) { fail_query = n; }
void fake_limit(size_t bytes) { limit = bytes; }
void fake_word(int v) { word_on = 1; word = v; }
void fake_pairs(unsigned long long n) { head_pairs = n; }
static int gaps;                      /* edges in every rule's gap histogram */
void fake_gaps(int n) { gaps = n; }
long long fake_steal_ticks(void) { return mined.steal_after_ticks; }
int fake_unit_shift(void) { return mined.unit_shift; }
int fake_claim_blocks(void) { return mined.claim_blocks; }
size_t fake_used(void) { return used; }
size_t fake_peak(int reset) { size_t p = peak; if (reset) peak = used; return p; }
int fake_pending(void) { int n = 0; for (int i = 0; i < MAXS; i++) n += pending[i]; return n; }
int fake_streams(void) { return nstream; }
const char *fake_trace(void) { static char out[1 << 16]; strcpy(out, trace); trace[0] = 0; return out; }
static void note(const char *s) { if (strlen(trace) + strlen(s) + 2 < sizeof trace) { strcat(trace, s); strcat(trace, "\n"); } }
static hipError_t ret(hipError_t e) { if (e != hipSuccess) last = e; return e; }
static int sid(hipStream_t s) { return (int)(size_t)s; }

static hipError_t take(void **p, size_t n, int host) {
  if (!host && used + n > limit) return ret(hipErrorOutOfMemory);
  size_t m = (n + 4095) & ~(size_t)4095;
  *p = mmap(0, m ? m : 4096, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (*p == MAP_FAILED) return ret(hipErrorOutOfMemory);
  for (int i = 0; i < MAXA; i++)
    if (!mem[i].p) { mem[i].p = *p; mem[i].n = n; mem[i].host = host; break; }
  if (!host) { used += n; if (used > peak) peak = used; }
  return hipSuccess;
}
static hipError_t drop(void *p) {
  if (!p) return hipSuccess;
  for (int i = 0; i < MAXA; i++)
    if (mem[i].p == p) {
      size_t m = (mem[i].n + 4095) & ~(size_t)4095;
      munmap(p, m ? m : 4096);
      if (!mem[i].host) used -= mem[i].n;
      mem[i].p = 0;
      return hipSuccess;
    }
  fprintf(stderr, "free of unknown memory %p\n", p);
  abort();
}

hipError_t hipMalloc(void **p, size_t n) { return take(p, n, 0); }
hipError_t hipFree(void *p) { return drop(p); }
hipError_t hipMemGetInfo(size_t *f, size_t *a) { *a = limit; *f = limit > used ? limit - used : 0; return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; return fail_host ? ret(hipErrorOutOfMemory) : take(p, n, 1); }
hipError_t hipHostFree(void *p) { return drop(p); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { (void)k; memmove(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t t) {
  if (word_on && n == 4 && k == hipMemcpyDeviceToHost) *(int *)d = word; else memmove(d, s, n);
  if (gaps && n == sizeof(unsigned) * TM_NTFIRST * 33 && k == hipMemcpyDeviceToHost)
    for (int r = 0; r < TM_NTFIRST; r++) ((unsigned *)d)[33 * r + 3] = gaps;
  pending[sid(t)]++;
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t t) { memset(d, v, n); pending[sid(t)]++; return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t *s) { *s = (hipStream_t)(size_t)(1 + nstream++); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  if (fail_sync && sid(s) == fail_stream) { fail_sync = 0; pending[sid(s)] = 0; note("sync fails"); return ret(hipErrorUnknown); }
  pending[sid(s)] = 0;
  return hipSuccess;
}
static int events;
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)(size_t)++events; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned f) { (void)f; return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { (void)e; (void)s; if (fail_record > 0 && --fail_record == 0) return ret(hipErrorUnknown); return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t e) { (void)e; return fail_query > 0 && fail_query-- ? ret(hipErrorUnknown) : hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) { (void)a; (void)b; *ms = 1; return hipSuccess; }
hipError_t hipGetLastError(void) { hipError_t e = last; last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "told to fail"; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int d) { (void)d; return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
int hipGetStreamDeviceId(hipStream_t s) { (void)s; return 0; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int d) {
  (void)d;
  memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  p->warpSize = 64;
  strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d) { (void)d; *v = a == hipDeviceAttributeWarpSize ? 64 : a == hipDeviceAttributeMultiprocessorCount ? 256 : 100000; return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *s) { (void)s; static void *a; if (!a) take(&a, (size_t)16 << 20, 1); *p = a; return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t l) { (void)f; (void)b; (void)l; *n = 8; return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { (void)g; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t g) { (void)g; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t g, hipStream_t s) { (void)g; (void)s; return hipSuccess; }

void **__hipRegisterFatBinary(const void *d) { (void)d; static void *h; return &h; }
void __hipUnregisterFatBinary(void **h) { (void)h; }
void __hipRegisterVar(void **m, void *v, char *h, char *n, int e, size_t s, int c, int g) { (void)m; (void)v; (void)h; (void)n; (void)e; (void)s; (void)c; (void)g; }
void __hipRegisterFunction(void **m, const void *f, char *h, const char *n, unsigned t, void *a, void *b, void *c, void *d, int *w) {
  (void)m; (void)h; (void)t; (void)a; (void)b; (void)c; (void)d; (void)w;
  if (nkern < MAXK) { kern[nkern].f = f; snprintf(kern[nkern].name, 256, "%s", n); nkern++; }
}
static struct { dim3 g, b; size_t s; hipStream_t t; } conf;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t t) { conf.g = g; conf.b = b; conf.s = s; conf.t = t; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, hipStream_t *t) { *g = conf.g; *b = conf.b; *s = conf.s; *t = conf.t; return hipSuccess; }
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **a, size_t s, hipStream_t t) {
  (void)g; (void)b; (void)s;
  const char *n = "?";
  for (int i = 0; i < nkern; i++) if (kern[i].f == f) n = kern[i].name;
  if (fail_kernel[0] && strstr(n, fail_kernel) && fail_kernel_after-- <= 0) { fail_kernel[0] = 0; note("launch fails"); return ret(hipErrorLaunchFailure); }
  note(n);
  pending[sid(t)]++;
  if (strstr(n, "mine_kernel")) mined = *(tm_kernel_args *)a[0];
  if (strstr(n, "heads_kernel")) **(unsigned long long **)a[2] = head_pairs;
  return hipSuccess;
}
