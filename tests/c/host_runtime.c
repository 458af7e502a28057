/* The part of the HIP runtime's interface that the library's host code calls,
   on host memory: allocations are zeroed, copies are memcpy, kernels do
   nothing but advance a clock.  Tests of the host code (contexts, graphs,
   error paths) load it in place of libamdhip64.so.7; hrt_set makes calls
   fail, hrt_get counts what is alive. */
#include <stdlib.h>
#include <string.h>

typedef struct {
  unsigned x, y, z;
} dim3_t;
enum { OK = 0, INVALID = 1, NO_MEMORY = 2 };

static long v_launch_fail;      /* 1: launches under capture fail, 2: all launches */
static long v_instantiate_fail; /* the next hipGraphInstantiate calls that succeed before one fails, plus 1 */
static long v_external_refused; /* hipEventRecordExternal is refused */
static long v_wait_fail;        /* hipStreamWaitEvent fails */
static long v_mem_limit;        /* bytes of device memory (0: any) */
static long v_contexts, v_graphs, v_execs, v_device_bytes;
static long g_clock;
static int g_last;
static int fail(int e) { return g_last = e; }

static const struct {
  const char *name;
  long *v;
} kVars[] = {{"launch_fail", &v_launch_fail}, {"instantiate_fail", &v_instantiate_fail},
             {"external_refused", &v_external_refused}, {"wait_fail", &v_wait_fail}, {"mem_limit", &v_mem_limit},
             {"contexts", &v_contexts}, {"graphs", &v_graphs}, {"execs", &v_execs},
             {"device_bytes", &v_device_bytes}};
static long *var(const char *name) {
  for (size_t i = 0; i < sizeof(kVars) / sizeof(kVars[0]); i++)
    if (!strcmp(kVars[i].name, name)) return kVars[i].v;
  abort();
}
void hrt_set(const char *name, long value) { *var(name) = value; }
long hrt_get(const char *name) { return *var(name); }

/* ---- events, streams, graphs ---- */
typedef struct {
  long t;
} event;
typedef struct {
  int n;
  event *ev[512]; /* NULL: a kernel */
} graph;
static graph *g_capture; /* the graph being captured */
static char g_stream[4096];
static int g_streams;

static void op(event *e) {
  if (g_capture) {
    if (g_capture->n == 512) abort();
    g_capture->ev[g_capture->n++] = e;
  } else if (e) {
    e->t = g_clock;
  } else {
    g_clock += 100;
  }
}

int hipStreamCreateWithFlags(void **s, unsigned f) {
  *s = &g_stream[++g_streams % 4095 + 1];
  return OK;
}
int hipStreamDestroy(void *s) { return OK; }
int hipStreamSynchronize(void *s) { return OK; }
int hipStreamWaitEvent(void *s, event *e, unsigned f) { return v_wait_fail ? fail(INVALID) : OK; }
int hipEventCreateWithFlags(event **e, unsigned f) {
  *e = calloc(1, sizeof(event));
  return OK;
}
int hipEventCreate(event **e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(event *e) {
  free(e);
  return OK;
}
int hipEventRecord(event *e, void *s) {
  if (!g_capture) op(e); /* under capture: a dependency only */
  return OK;
}
int hipEventRecordWithFlags(event *e, void *s, unsigned f) {
  if (f && v_external_refused) return fail(INVALID);
  if (f || !g_capture) op(e);
  return OK;
}
int hipEventElapsedTime(float *ms, event *a, event *b) {
  *ms = (float)(b->t - a->t);
  return OK;
}
int hipStreamBeginCapture(void *s, int mode) {
  g_capture = calloc(1, sizeof(graph));
  v_graphs++;
  return OK;
}
int hipStreamEndCapture(void *s, graph **g) {
  *g = g_capture;
  g_capture = NULL;
  return OK;
}
int hipStreamGetCaptureInfo_v2(void *s, int *status, unsigned long long *id, graph **g, void ***deps, size_t *n) {
  *status = g_capture != NULL;
  *g = g_capture;
  *deps = NULL;
  *n = 0;
  return OK;
}
int hipGraphAddEventRecordNode(void **node, graph *g, void **deps, size_t n, event *e) {
  op(e);
  *node = e;
  return OK;
}
int hipStreamUpdateCaptureDependencies(void *s, void **deps, size_t n, unsigned f) { return OK; }
int hipGraphInstantiate(graph **x, graph *g, void *a, void *b, size_t c) {
  if (v_instantiate_fail && --v_instantiate_fail == 0) return fail(NO_MEMORY);
  *x = malloc(sizeof(graph));
  **x = *g;
  v_execs++;
  return OK;
}
int hipGraphLaunch(graph *x, void *s) {
  for (int i = 0; i < x->n; i++) op(x->ev[i]);
  return OK;
}
int hipGraphDestroy(graph *g) {
  free(g);
  v_graphs--;
  return OK;
}
int hipGraphExecDestroy(graph *x) {
  free(x);
  v_execs--;
  return OK;
}

/* ---- kernels ---- */
void **__hipRegisterFatBinary(void *d) { return calloc(1, sizeof(void *)); }
void __hipUnregisterFatBinary(void **m) { free(m); }
void __hipRegisterFunction(void **m, const void *f, char *df, const char *n, unsigned t, void *a, void *b, void *c,
                           void *d, int *w) {}
void __hipRegisterVar(void **m, void *v, char *h, char *n, int e, size_t s, int c, int g) {}
static struct {
  dim3_t g, b;
  size_t shm;
  void *s;
} g_call;
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t shm, void *s) {
  g_call.g = g;
  g_call.b = b;
  g_call.shm = shm;
  g_call.s = s;
  return OK;
}
int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *shm, void **s) {
  *g = g_call.g;
  *b = g_call.b;
  *shm = g_call.shm;
  *s = g_call.s;
  return OK;
}
int hipLaunchKernel(const void *f, dim3_t g, dim3_t b, void **args, size_t shm, void *s) {
  if (v_launch_fail == 2 || (v_launch_fail == 1 && g_capture)) return fail(INVALID);
  op(NULL);
  return OK;
}

/* ---- memory: the size in front of every block ---- */
int hipMalloc(void **p, size_t n) {
  if (v_mem_limit && v_device_bytes + (long)n > v_mem_limit) return fail(NO_MEMORY);
  size_t *q = calloc(1, n + 4096);
  if (!q) return fail(NO_MEMORY);
  *q = n;
  v_device_bytes += (long)n;
  *p = (char *)q + 256;
  return OK;
}
int hipFree(void *p) {
  if (!p) return OK;
  size_t *q = (size_t *)((char *)p - 256);
  v_device_bytes -= (long)*q;
  free(q);
  return OK;
}
int hipHostMalloc(void **p, size_t n, unsigned f) {
  *p = malloc(n);
  return *p ? OK : fail(NO_MEMORY);
}
int hipHostFree(void *p) {
  free(p);
  return OK;
}
int hipMemcpy(void *d, const void *s, size_t n, int kind) {
  memcpy(d, s, n);
  return OK;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st) { return hipMemcpy(d, s, n, kind); }
int hipMemsetAsync(void *d, int v, size_t n, void *st) {
  memset(d, v, n);
  return OK;
}

/* ---- device ---- */
int hipGetDeviceCount(int *n) {
  *n = 1;
  return OK;
}
int hipGetDevice(int *d) {
  *d = 0;
  return OK;
}
int hipSetDevice(int d) { return OK; }
int hipDeviceGetAttribute(int *v, int a, int d) {
  *v = 160 * 1024;
  v_contexts++; /* asked once per device context */
  return OK;
}
int hipGetSymbolAddress(void **p, const void *sym) {
  static char scratch[32 << 20];
  *p = scratch;
  return OK;
}
const char *hipGetErrorString(int e) { return e == OK ? "no error" : e == NO_MEMORY ? "out of memory" : "invalid argument"; }
int hipGetLastError(void) {
  const int e = g_last;
  g_last = OK;
  return e;
}
int hipPeekAtLastError(void) { return g_last; }
