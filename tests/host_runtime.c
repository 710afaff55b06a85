/* A stand-in for the HIP runtime on a machine without a GPU: device memory is
 * host memory, kernels are recorded and not run.  Loaded before the library it
 * takes the runtime's place, so that what the library's host code does can be
 * checked: which kernels a call launches, on which stream and device, with
 * which launch shape, what it allocates, and what it does when that fails. */
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

typedef struct { uint32_t x, y, z; } dim3_t;
enum { OK = 0, INVALID = 1, NOMEM = 2 };

/* ---- what the tests read and set */
int host_device = 0;       /* the current device */
int host_mallocs = 0;      /* allocations so far */
int host_live = 0;         /* buffers not given back */
int host_fail_at = 0;      /* the host_fail_at-th allocation from now fails (0: none) */
int host_bad = 0;          /* frees of what was not allocated, copies to or from null */
static char* log_buf = NULL;
static size_t log_len = 0, log_cap = 0;
static int last_error = OK;

const char* host_log(void) { return log_buf ? log_buf : ""; }
void host_log_clear(void) { log_len = 0; if (log_buf) log_buf[0] = 0; }
static void log_line(const char* s) {
  size_t n = strlen(s);
  if (log_len + n + 2 > log_cap) log_buf = realloc(log_buf, log_cap = 2 * (log_len + n + 2) + 4096);
  memcpy(log_buf + log_len, s, n);
  log_len += n;
  log_buf[log_len++] = '\n';
  log_buf[log_len] = 0;
}

/* ---- memory */
#define MAXBUF 4096
static void* bufs[MAXBUF];
int hipMalloc(void** p, size_t n) {
  *p = NULL;
  if (host_fail_at > 0 && --host_fail_at == 0) return last_error = NOMEM;
  char t[80];
  snprintf(t, sizeof t, "malloc %zu device %d", n, host_device);
  log_line(t);
  *p = calloc(1, n);
  ++host_mallocs;
  ++host_live;
  for (int i = 0; i < MAXBUF; ++i) if (!bufs[i]) { bufs[i] = *p; return OK; }
  return last_error = NOMEM;
}
int hipFree(void* p) {
  if (!p) return OK;
  for (int i = 0; i < MAXBUF; ++i) if (bufs[i] == p) { bufs[i] = NULL; free(p); --host_live; return OK; }
  ++host_bad;
  return last_error = INVALID;
}
int hipMallocAsync(void** p, size_t n, void* s) { (void)s; return hipMalloc(p, n); }
int hipFreeAsync(void* p, void* s) { (void)s; return hipFree(p); }
int hipMemcpy(void* d, const void* s, size_t n, int k) {
  (void)k;
  if (!d || !s) { ++host_bad; return last_error = INVALID; }
  memcpy(d, s, n);
  return OK;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* st) { (void)st; return hipMemcpy(d, s, n, k); }
int hipMemset(void* d, int v, size_t n) { (void)d; (void)v; (void)n; return OK; }
int hipMemsetAsync(void* d, int v, size_t n, void* st) { (void)d; (void)v; (void)n; (void)st; return OK; }

/* ---- devices, streams, events, errors */
int hipGetDevice(int* d) { *d = host_device; return OK; }
int hipSetDevice(int d) { host_device = d; return OK; }
int host_cus = 256;        /* compute units */
int hipDeviceGetAttribute(int* v, int a, int d) { (void)a; (void)d; *v = host_cus; return OK; }
int hipDeviceSynchronize(void) { return OK; }
static uintptr_t handles = 0x1000;
int hipStreamCreateWithFlags(void** s, unsigned f) {
  char t[80];
  *s = (void*)(handles += 16);
  snprintf(t, sizeof t, "stream %p %s", *s, f ? "nonblocking" : "blocking");
  log_line(t);
  return OK;
}
int hipStreamCreate(void** s) { return hipStreamCreateWithFlags(s, 0); }
int hipStreamDestroy(void* s) {
  char t[80];
  if (!s) { ++host_bad; return last_error = INVALID; }
  snprintf(t, sizeof t, "destroy %p", s);
  log_line(t);
  return OK;
}
int hipStreamSynchronize(void* s) { (void)s; return OK; }
int hipStreamWaitEvent(void* s, void* e, unsigned f) { (void)s; (void)e; (void)f; return OK; }
int hipEventCreate(void** e) { *e = (void*)(handles += 16); return OK; }
int hipEventCreateWithFlags(void** e, unsigned f) { (void)f; return hipEventCreate(e); }
int hipEventDestroy(void* e) { (void)e; return OK; }
int hipEventRecord(void* e, void* s) { (void)e; (void)s; return OK; }
int hipEventSynchronize(void* e) { (void)e; return OK; }
int hipEventElapsedTime(float* ms, void* a, void* b) { (void)a; (void)b; *ms = 1.0f; return OK; }
int hipGetLastError(void) { int e = last_error; last_error = OK; return e; }
const char* hipGetErrorString(int e) { return e == NOMEM ? "out of memory" : e ? "error" : "no error"; }

/* ---- kernels */
#define MAXFN 4096
static const void* fn_host[MAXFN];
static char fn_name[MAXFN][256];
static int nfn = 0;
void** __hipRegisterFatBinary(const void* d) { static void* h[1]; (void)d; return h; }
void __hipUnregisterFatBinary(void** h) { (void)h; }
void __hipRegisterFunction(void** m, const void* host, char* dev, const char* name, unsigned tl, void* a, void* b, void* c, void* d, int* w) {
  (void)m; (void)dev; (void)tl; (void)a; (void)b; (void)c; (void)d; (void)w;
  if (nfn < MAXFN) { fn_host[nfn] = host; snprintf(fn_name[nfn++], 256, "%s", name); }
}
void __hipRegisterVar(void** m, void* v, char* a, char* b, int c, size_t d, int e, int f) {
  (void)m; (void)v; (void)a; (void)b; (void)c; (void)d; (void)e; (void)f;
}
int hipGetSymbolAddress(void** p, const void* s) { static char mem[1 << 16]; (void)s; *p = mem; return OK; }
int hipFuncSetAttribute(const void* f, int a, int v) { (void)f; (void)a; (void)v; return OK; }
static struct { dim3_t g, b; size_t sh; void* s; } cfg;
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t sh, void* s) { cfg.g = g; cfg.b = b; cfg.sh = sh; cfg.s = s; return OK; }
int __hipPopCallConfiguration(dim3_t* g, dim3_t* b, size_t* sh, void** s) { *g = cfg.g; *b = cfg.b; *sh = cfg.sh; *s = cfg.s; return OK; }
int hipLaunchKernel(const void* f, dim3_t g, dim3_t b, void** args, size_t sh, void* s) {
  char t[512];
  const char* n = "?";
  (void)args;
  for (int i = 0; i < nfn; ++i) if (fn_host[i] == f) { n = fn_name[i]; break; }
  snprintf(t, sizeof t, "launch %s grid %u %u %u block %u lds %zu stream %p device %d", n, g.x, g.y, g.z, b.x * b.y * b.z, sh, s, host_device);
  log_line(t);
  return OK;
}
