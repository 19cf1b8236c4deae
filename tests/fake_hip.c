/* A HIP runtime without a GPU, for tests of the host code: streams, events and memory
 * are names in a log (hip_log) from which the tests work out what is ordered after
 * what; kernels do not run; device memory is host memory, of which hip_limit bytes are
 * to be had; copies are done at once. */
#define _GNU_SOURCE
#include <pthread.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>
#include <sys/mman.h>
#include <sys/syscall.h>

enum { SUCCESS = 0, OUT_OF_MEMORY = 2, INVALID = 1, CAPTURE = 900 };
typedef struct { uint32_t x, y, z; } dim3;

static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static char *text;
static size_t len, cap;

static void say(const char *fmt, ...) {
  char line[256];
  va_list ap;
  va_start(ap, fmt);
  int n = vsnprintf(line, sizeof line, fmt, ap);
  va_end(ap);
  pthread_mutex_lock(&mu);
  if (len + n + 2 > cap) text = realloc(text, cap = 2 * (cap + n + 256));
  memcpy(text + len, line, n);
  len += n;
  text[len++] = '\n';
  text[len] = 0;
  pthread_mutex_unlock(&mu);
}

const char *hip_log(void) { return len ? text : ""; }
void hip_log_clear(void) { len = 0; }

/* ---- memory: blocks with their size; `host` ones are pinned host memory */
static struct { char *p; size_t n; int host; } block[4096];
static int blocks;
size_t hip_limit = (size_t)1 << 40;
size_t hip_live;

static int take(void **p, size_t n, int host) {
  pthread_mutex_lock(&mu);
  int ok = (host || hip_live + n <= hip_limit) && blocks < 4096;
  if (ok) {   /* pages are there when they are used, if ever */
    *p = mmap(0, n ? n : 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    ok = *p != MAP_FAILED;
  }
  if (ok) {
    block[blocks].p = *p;
    block[blocks].n = n;
    block[blocks++].host = host;
    if (!host) hip_live += n;
  } else {
    *p = 0;
  }
  pthread_mutex_unlock(&mu);
  return ok ? SUCCESS : OUT_OF_MEMORY;
}
static void drop(void *p) {
  pthread_mutex_lock(&mu);
  for (int i = 0; i < blocks; ++i)
    if (block[i].p == p) {
      if (!block[i].host) hip_live -= block[i].n;
      munmap(p, block[i].n ? block[i].n : 1);
      block[i] = block[--blocks];
      break;
    }
  pthread_mutex_unlock(&mu);
}

static void *capturing[16];
static int captures;
void hip_capture(void *s, int on) {
  if (on) capturing[captures++] = s;
  else captures = 0;
}
static int is_capturing(void *s) {
  for (int i = 0; i < captures; ++i)
    if (capturing[i] == s) return 1;
  return 0;
}

int hipMalloc(void **p, size_t n) {
  say("malloc %zu", n);
  return captures ? CAPTURE : take(p, n, 0);
}
int hipFree(void *p) { say("free %p", p); drop(p); return SUCCESS; }
int hipHostMalloc(void **p, size_t n, unsigned f) { say("host_malloc %zu", n); return take(p, n, 1); }
int hipHostFree(void *p) { say("host_free %p", p); drop(p); return SUCCESS; }
int hipMemGetInfo(size_t *f, size_t *t) { *t = hip_limit; *f = hip_limit - hip_live; return SUCCESS; }
int hipPointerGetAttributes(void *a, const void *p) {
  pthread_mutex_lock(&mu);
  int type = 0;   /* hipMemoryTypeUnregistered */
  for (int i = 0; i < blocks; ++i)
    if ((const char *)p >= block[i].p && (const char *)p < block[i].p + block[i].n) type = block[i].host ? 1 : 2;
  pthread_mutex_unlock(&mu);
  *(int *)a = type;
  return SUCCESS;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *stream) {
  say("copy %p %d %zu %ld", stream, kind, n, (long)syscall(SYS_gettid));
  memcpy(d, s, n);
  return SUCCESS;
}

/* ---- streams and events */
int hipStreamCreate(void **s) { *s = malloc(1); return SUCCESS; }
int hipStreamCreateWithFlags(void **s, unsigned f) { *s = malloc(1); return SUCCESS; }
int hipStreamDestroy(void *s) { return SUCCESS; }
int hipStreamSynchronize(void *s) { say("sync_stream %p %ld", s, (long)syscall(SYS_gettid)); return is_capturing(s) ? CAPTURE : SUCCESS; }
int hipDeviceSynchronize(void) { say("sync_device"); return captures ? CAPTURE : SUCCESS; }
int hipStreamIsCapturing(void *s, int *st) { *st = is_capturing(s); return SUCCESS; }
int hipStreamWaitEvent(void *s, void *e, unsigned f) { say("wait %p %p", s, e); return SUCCESS; }
int hipEventCreateWithFlags(void **e, unsigned f) { *e = malloc(1); say("event_create %p", *e); return SUCCESS; }
int hipEventCreate(void **e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void *e) { say("event_destroy %p", e); return SUCCESS; }   /* (the name is not used again) */
int hipEventRecord(void *e, void *s) { say("record %p %p", e, s); return SUCCESS; }
int hipEventSynchronize(void *e) { say("sync_event %p %ld", e, (long)syscall(SYS_gettid)); return SUCCESS; }
int hipEventElapsedTime(float *ms, void *a, void *b) { *ms = 1.0f; return SUCCESS; }

/* ---- device */
int hipGetDeviceCount(int *n) { *n = 1; return SUCCESS; }
int hipGetDevice(int *d) { *d = 0; return SUCCESS; }
int hipSetDevice(int d) { return d ? INVALID : SUCCESS; }
int hipDeviceGetAttribute(int *v, int a, int d) { *v = 256; return SUCCESS; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t s) { *n = 2; return SUCCESS; }
static __thread int last_error;
int hipGetLastError(void) {
  int e = last_error;
  last_error = SUCCESS;
  return e;
}
const char *hipGetErrorString(int e) { return e == OUT_OF_MEMORY ? "out of memory" : e == CAPTURE ? "capturing" : "error"; }
static char symbol[64 << 20];
int hipGetSymbolAddress(void **p, const void *s) { *p = symbol; return SUCCESS; }

/* ---- kernels, by name */
static struct { const void *f; const char *name; } kernel[1024];
static int kernels;
void *__hipRegisterFatBinary(const void *d) { static void *h; return &h; }
void __hipUnregisterFatBinary(void *h) {}
void __hipRegisterFunction(void *h, const void *f, char *d, const char *name, unsigned n, void *a, void *b, void *c,
                           void *e, int *w) {
  if (kernels < 1024) {
    kernel[kernels].f = f;
    kernel[kernels++].name = name;
  }
}
void __hipRegisterVar(void *h, void *v, char *a, char *b, int c, size_t d, int e, int f) {}
static __thread struct { dim3 g, b; size_t m; void *s; } call;
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, void *s) {
  call.g = g; call.b = b; call.m = m; call.s = s;
  return SUCCESS;
}
int __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *m, void **s) {
  *g = call.g; *b = call.b; *m = call.m; *s = call.s;
  return SUCCESS;
}
int hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t m, void *s) {
  const char *name = "?";
  for (int i = 0; i < kernels; ++i)
    if (kernel[i].f == f) name = kernel[i].name;
  say("launch %p %u %u %u %u %.180s", s, g.x, g.y, g.z, b.x * b.y * b.z, name);
  if ((uint64_t)g.x * b.x >> 32) last_error = INVALID;
  return last_error;
}

/* ---- graphs: not simulated */
int hipStreamBeginCapture(void *s, int m) { return INVALID; }
int hipStreamEndCapture(void *s, void **g) { return INVALID; }
int hipGraphInstantiate(void **x, void *g, void *a, void *b, size_t n) { return INVALID; }
int hipGraphLaunch(void *x, void *s) { return INVALID; }
int hipGraphDestroy(void *g) { return SUCCESS; }
int hipGraphExecDestroy(void *x) { return SUCCESS; }
