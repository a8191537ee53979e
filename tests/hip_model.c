/* A host model of the HIP calls that libptn_hip.so makes, so that what the library does around its
 * kernels (memory, streams, order of events) can be tested without a GPU.  Loaded with RTLD_GLOBAL
 * before the library, its functions take the place of the runtime's.
 *
 * Device memory is host memory, counted, with a limit.  Streams are lazy: copies and fills wait in
 * their stream until something makes the host wait for it, and no stream waits for another unless an
 * event says so (the handles' streams are non-blocking).  So work that nobody waits for is still
 * there when a call returns (model_pending).  Kernels do nothing; their names, streams and places
 * among the events are in the trace. */
#define _GNU_SOURCE
#include <pthread.h>
#include <stdarg.h>
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>
#include <time.h>

typedef struct { uint32_t x, y, z; } dim3_t;
typedef struct op {
  int kind;                                   /* 0 kernel, 1 copy, 2 fill, 3 record, 4 wait */
  void *dst;
  const void *src;
  size_t n;
  int value;
  struct event *ev;
  uint64_t gen;
  struct op *next;
} op;
typedef struct stream { op *head, *tail; int id; struct stream *next; } stream;
typedef struct event { stream *s; uint64_t gen, done; } event;

static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static stream null_stream, *streams;
static int next_stream = 1;

/* ---- memory ---- */
#define MAX_BLOCKS 65536
static struct { char *p; size_t n; } blocks[MAX_BLOCKS];
static int nblocks;
static size_t in_use, peak, limit = (size_t)1 << 62;
static long mallocs, frees, fail_after = -1;
/* hipFree holds the caller until model_free_release or two seconds (1: armed, 2: a caller is held) */
static volatile int hold_free, free_timed_out;

/* ---- trace ---- */
#define MAX_TRACE 20000
static char *trace_line[MAX_TRACE];
static int ntrace;
static void say(const char *fmt, ...) {
  char b[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(b, sizeof(b), fmt, ap);
  va_end(ap);
  if (ntrace < MAX_TRACE) trace_line[ntrace++] = strdup(b);
}
void model_trace_clear(void) { while (ntrace) free(trace_line[--ntrace]); }
int model_trace_size(void) { return ntrace; }
const char *model_trace(int i) { return trace_line[i]; }

size_t model_in_use(void) { return in_use; }
size_t model_peak(void) { return peak; }
void model_reset_peak(void) { peak = in_use; }
void model_limit(size_t n) { limit = n; }
long model_mallocs(void) { return mallocs; }
long model_frees(void) { return frees; }
void model_fail_after(long n) { fail_after = n; }
void model_hold_free(int on) { hold_free = on; free_timed_out = 0; }
int model_free_held(void) { return hold_free == 2; }
int model_free_timed_out(void) { return free_timed_out; }
int model_pending(void) {
  int n = 0;
  pthread_mutex_lock(&mu);
  for (op *o = null_stream.head; o; o = o->next) ++n;
  for (stream *s = streams; s; s = s->next)
    for (op *o = s->head; o; o = o->next) ++n;
  pthread_mutex_unlock(&mu);
  return n;
}

/* ---- streams: everything below with mu held ---- */
static void drain(stream *s, const op *until);
static void push(stream *s, op v) {
  op *o = malloc(sizeof(op));
  *o = v;
  o->next = NULL;
  if (s->tail) s->tail->next = o;
  else s->head = o;
  s->tail = o;
}
static void reach(event *e, uint64_t gen) {   /* runs the event's stream up to its record */
  while (e && e->done < gen && e->s && e->s->head) {
    op *o = e->s->head;
    drain(e->s, o);
  }
}
static void touch_copy(void *d, const void *s, size_t n) { memcpy(d, s, n); }
static void drain(stream *s, const op *until) {
  while (s->head) {
    op *o = s->head;
    if (o->kind == 4) reach(o->ev, o->gen);
    if (s->head != o) continue;               /* (a wait reached back into this stream) */
    s->head = o->next;
    if (!s->head) s->tail = NULL;
    if (o->kind == 1) touch_copy(o->dst, o->src, o->n);
    if (o->kind == 2) memset(o->dst, o->value, o->n);
    if (o->kind == 3 && o->ev->done < o->gen) o->ev->done = o->gen;
    const int last = o == until;
    free(o);
    if (last) return;
  }
}
static stream *of(void *s) { return s ? (stream *)s : &null_stream; }
static void drain_all(void) {
  drain(&null_stream, NULL);
  for (stream *s = streams; s; s = s->next) drain(s, NULL);
}
static int is_device(const void *p) {
  for (int i = 0; i < nblocks; ++i)
    if ((const char *)p >= blocks[i].p && (const char *)p < blocks[i].p + blocks[i].n) return 1;
  return 0;
}

/* ---- the runtime's calls ---- */
enum { OK = 0, INVALID = 1, OOM = 2, NOT_READY = 600 };
static __thread int last_error;
static int ret(int e) { if (e && e != NOT_READY) last_error = e; return e; }

int hipGetDeviceCount(int *n) { *n = 1; return 0; }
int hipSetDevice(int d) { return d == 0 ? 0 : ret(101); }
int hipDeviceGetAttribute(int *v, int a, int d) { (void)a; (void)d; *v = 256; return 0; }
int hipGetLastError(void) { int e = last_error; last_error = 0; return e; }
const char *hipGetErrorString(int e) { return e == OOM ? "out of memory" : "error"; }

int hipMalloc(void **p, size_t n) {
  pthread_mutex_lock(&mu);
  if (fail_after == 0 || in_use + n > limit) {
    pthread_mutex_unlock(&mu);
    return ret(OOM);
  }
  if (fail_after > 0) --fail_after;
  char *m = mmap(NULL, n ? n : 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (m == MAP_FAILED || nblocks == MAX_BLOCKS) abort();
  blocks[nblocks].p = m;
  blocks[nblocks++].n = n;
  in_use += n;
  if (in_use > peak) peak = in_use;
  ++mallocs;
  *p = m;
  pthread_mutex_unlock(&mu);
  return 0;
}
int hipFree(void *p) {
  if (!p) return 0;
  for (int ms = 0; hold_free && ms < 2000; ++ms) {
    hold_free = 2;
    struct timespec t = {0, 1000000};
    nanosleep(&t, NULL);
    if (ms == 1999) {
      free_timed_out = 1;
      hold_free = 0;
    }
  }
  pthread_mutex_lock(&mu);
  drain_all();                                /* hipFree waits for the device */
  for (int i = 0; i < nblocks; ++i)
    if (blocks[i].p == (char *)p) {
      in_use -= blocks[i].n;
      munmap(p, blocks[i].n ? blocks[i].n : 1);
      blocks[i] = blocks[--nblocks];
      ++frees;
      pthread_mutex_unlock(&mu);
      return 0;
    }
  abort();                                    /* not a block, or freed twice */
}
int hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; *p = calloc(1, n); return 0; }
int hipHostFree(void *p) { free(p); return 0; }
int hipHostGetDevicePointer(void **d, void *h, unsigned f) { (void)f; *d = h; return 0; }
int hipGetSymbolAddress(void **p, const void *sym) { (void)sym; static char scratch[64]; *p = scratch; return 0; }

int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st) {
  pthread_mutex_lock(&mu);
  stream *q = of(st);
  if (kind == 1) {                            /* pageable host memory: read before the call returns */
    drain(q, NULL);
    memcpy(d, s, n);
  } else {
    push(q, (op){.kind = 1, .dst = d, .src = s, .n = n});
  }
  say("copy kind=%d bytes=%zu stream=%d", kind, n, q->id);
  pthread_mutex_unlock(&mu);
  return 0;
}
int hipMemcpy(void *d, const void *s, size_t n, int kind) {
  pthread_mutex_lock(&mu);
  say("copy kind=%d bytes=%zu stream=0 blocking", kind, n);
  push(&null_stream, (op){.kind = 1, .dst = d, .src = s, .n = n});
  /* the host waits for a copy with a host side; between device buffers it does not */
  if (!(is_device(d) && is_device(s))) drain(&null_stream, NULL);
  pthread_mutex_unlock(&mu);
  return 0;
}
int hipMemsetAsync(void *d, int v, size_t n, void *st) {
  pthread_mutex_lock(&mu);
  push(of(st), (op){.kind = 2, .dst = d, .value = v, .n = n});
  pthread_mutex_unlock(&mu);
  return 0;
}
int hipMemset(void *d, int v, size_t n) { return hipMemsetAsync(d, v, n, NULL); }

int hipStreamCreateWithFlags(void **s, unsigned f) {
  (void)f;
  pthread_mutex_lock(&mu);
  stream *q = calloc(1, sizeof(stream));
  q->id = next_stream++;
  q->next = streams;
  streams = q;
  *s = q;
  pthread_mutex_unlock(&mu);
  return 0;
}
int hipStreamDestroy(void *s) {
  pthread_mutex_lock(&mu);
  drain((stream *)s, NULL);
  for (stream **p = &streams; *p; p = &(*p)->next)
    if (*p == s) {
      *p = (*p)->next;
      break;
    }
  pthread_mutex_unlock(&mu);                  /* (kept: events may name it) */
  return 0;
}
int hipStreamSynchronize(void *s) {
  pthread_mutex_lock(&mu);
  drain(of(s), NULL);
  pthread_mutex_unlock(&mu);
  return 0;
}
int hipStreamQuery(void *s) {
  pthread_mutex_lock(&mu);
  drain(of(s), NULL);
  pthread_mutex_unlock(&mu);
  return 0;
}
int hipDeviceSynchronize(void) {
  pthread_mutex_lock(&mu);
  drain_all();
  pthread_mutex_unlock(&mu);
  return 0;
}
int hipStreamWaitEvent(void *s, void *e, unsigned f) {
  (void)f;
  pthread_mutex_lock(&mu);
  event *ev = e;
  push(of(s), (op){.kind = 4, .ev = ev, .gen = ev->gen});
  say("wait event=%p stream=%d", e, of(s)->id);
  pthread_mutex_unlock(&mu);
  return 0;
}
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; *e = calloc(1, sizeof(event)); return 0; }
int hipEventCreate(void **e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void *e) { (void)e; return 0; }   /* (kept: queued work may name it) */
int hipEventRecord(void *e, void *s) {
  pthread_mutex_lock(&mu);
  event *ev = e;
  ev->s = of(s);
  push(ev->s, (op){.kind = 3, .ev = ev, .gen = ++ev->gen});
  say("record event=%p stream=%d", e, ev->s->id);
  pthread_mutex_unlock(&mu);
  return 0;
}
int hipEventSynchronize(void *e) {
  pthread_mutex_lock(&mu);
  reach(e, ((event *)e)->gen);
  pthread_mutex_unlock(&mu);
  return 0;
}
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 1.f; return 0; }

int hipStreamBeginCapture(void *s, int m) { (void)s; (void)m; return 0; }
int hipStreamEndCapture(void *s, void **g) { (void)s; *g = NULL; return 0; }
int hipGraphInstantiate(void **e, void *g, void *n, char *l, size_t z) { (void)g; (void)n; (void)l; (void)z; *e = NULL; return 0; }
int hipGraphLaunch(void *e, void *s) { (void)e; (void)s; return 0; }
int hipGraphExecDestroy(void *e) { (void)e; return 0; }
int hipGraphDestroy(void *g) { (void)g; return 0; }

/* ---- kernels ---- */
#define MAX_KERNELS 4096
static struct { const void *f; char name[256]; } kernels[MAX_KERNELS];
static int nkernels;
void **__hipRegisterFatBinary(const void *d) { (void)d; static void *h; return &h; }
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterFunction(void **m, const void *host, char *dev, const char *name, unsigned tl, void *a, void *b,
                           void *c, void *d, int *w) {
  (void)m; (void)dev; (void)tl; (void)a; (void)b; (void)c; (void)d; (void)w;
  if (nkernels == MAX_KERNELS) abort();
  kernels[nkernels].f = host;
  snprintf(kernels[nkernels++].name, 256, "%s", name);
}
void __hipRegisterVar(void **m, void *v, char *h, char *n, int e, size_t s, int c, int g) {
  (void)m; (void)v; (void)h; (void)n; (void)e; (void)s; (void)c; (void)g;
}
static __thread struct { dim3_t g, b; size_t sh; void *s; } call;
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t sh, void *s) {
  call.g = g; call.b = b; call.sh = sh; call.s = s;
  return 0;
}
int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *sh, void **s) {
  *g = call.g; *b = call.b; *sh = call.sh; *s = call.s;
  return 0;
}
int hipLaunchKernel(const void *f, dim3_t g, dim3_t b, void **args, size_t sh, void *s) {
  (void)args; (void)sh;
  const char *name = "?";
  for (int i = 0; i < nkernels; ++i)
    if (kernels[i].f == f) name = kernels[i].name;
  pthread_mutex_lock(&mu);
  push(of(s), (op){.kind = 0});
  say("kernel %s grid=%u,%u,%u block=%u stream=%d", name, g.x, g.y, g.z, b.x, of(s)->id);
  pthread_mutex_unlock(&mu);
  return 0;
}
