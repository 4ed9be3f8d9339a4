/* A stand-in for the HIP runtime on machines without a GPU: the entry points that the library calls, with
 * device memory from calloc and one queue of pending transfers per stream.  A transfer between device
 * memory and memory of hipHostMalloc is only queued; it runs when its stream or a later event of that
 * stream is waited for, and a wait on any stream runs every other stream's queue after its own, the order
 * in which a buffer that was given away too early shows.  Transfers of pageable memory run at once.  Of the
 * kernels only the two that move data are carried out (k_copy, k_store_values).  fake_fail makes the
 * n-th coming call of one function fail; the counters below tell what was called. */
#include <pthread.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

typedef struct { uint32_t x, y, z; } dim3;
typedef struct op { struct op *next; char *dst; const char *src; size_t n; long seq; } op;
typedef struct stream { struct stream *next; op *head, *tail; long unwaited; } stream;
typedef struct { stream *s; long seq; unsigned flags; } event;
typedef struct span { struct span *next; char *p; size_t n; } span;
typedef struct fn { struct fn *next; const void *host; char name[256]; } fn;

static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static stream *streams;
static span *pinned;
static fn *fns;
static long seq;
static __thread struct { dim3 g, b; size_t sh; void *s; } cfg;

/* what was called, and what is to fail */
enum { HOST_MALLOC, EVENT_CREATE, EVENT_RECORD, EVENT_SYNC, STREAM_SYNC, COPY_ASYNC, LAUNCH, NCOUNT };
static long count[NCOUNT], fail_at[NCOUNT];
static unsigned host_flags = ~0u, event_flags = ~0u;   /* the flags every such call had */
static size_t pinned_now, pinned_most;

long fake_count(int k) { return count[k]; }
/* launches and copies of any stream since its last hipStreamSynchronize */
long fake_unwaited(void) {
    long n = 0;
    pthread_mutex_lock(&mu);
    for (stream *s = streams; s; s = s->next) n += s->unwaited;
    pthread_mutex_unlock(&mu);
    return n;
}
/* the grid of the last launch of a kernel whose name has this in it */
static char watched[256];
static int watched_grid;
void fake_watch(const char *part) {
    snprintf(watched, sizeof watched, "%s", part);
    watched_grid = 0;
}
int fake_grid(void) { return watched_grid; }
/* n > 0: the n-th coming call, n < 0: every coming call, 0: none */
void fake_fail(int k, long n) { fail_at[k] = n > 0 ? count[k] + n : n; }
unsigned fake_host_flags(void) { return host_flags; }
unsigned fake_event_flags(void) { return event_flags; }
size_t fake_pinned_most(void) { return pinned_most; }
long fake_pending(void) {
    long n = 0;
    pthread_mutex_lock(&mu);
    for (stream *s = streams; s; s = s->next)
        for (op *o = s->head; o; o = o->next) ++n;
    pthread_mutex_unlock(&mu);
    return n;
}

enum { FAILED = 999 };
static __thread int last_error;   /* stays until hipGetLastError reads it */
static int bad(int k) {   /* mu held */
    const long c = ++count[k], f = fail_at[k];
    if (!(f < 0 || (f > 0 && c == f))) return 0;
    return last_error = FAILED;
}

static void run(stream *s, long upto) {
    while (s->head && s->head->seq <= upto) {
        op *o = s->head;
        memcpy(o->dst, o->src, o->n);
        s->head = o->next;
        if (!s->head) s->tail = NULL;
        free(o);
    }
}
static void run_others(stream *not_s) {
    for (stream *s = streams; s; s = s->next)
        if (s != not_s) run(s, seq);
}
static int is_pinned(const void *p) {
    for (span *q = pinned; q; q = q->next)
        if ((const char *)p >= q->p && (const char *)p < q->p + q->n) return 1;
    return 0;
}
static void queue(stream *s, void *dst, const void *src, size_t n) {
    op *o = calloc(1, sizeof *o);
    o->dst = dst; o->src = src; o->n = n; o->seq = ++seq;
    if (s->tail) s->tail->next = o; else s->head = o;
    s->tail = o;
}
#define IN pthread_mutex_lock(&mu)
#define OUT(x) do { const int r_ = (x); pthread_mutex_unlock(&mu); return r_; } while (0)

int hipGetDevice(int *d) { *d = 0; return 0; }
int hipSetDevice(int d) { (void)d; return 0; }
int hipGetDeviceCount(int *n) { *n = 1; return 0; }
int hipDeviceGetAttribute(int *v, int a, int d) { (void)a; (void)d; *v = 256; return 0; }
int hipGetLastError(void) {
    const int e = last_error;
    last_error = 0;
    return e;
}
const char *hipGetErrorString(int e) { (void)e; return "made to fail"; }
int hipMalloc(void **p, size_t n) { *p = calloc(1, n + 64); return *p ? 0 : 2; }
int hipFree(void *p) { free(p); return 0; }
int hipMemset(void *p, int v, size_t n) { memset(p, v, n); return 0; }
int hipMemsetAsync(void *p, int v, size_t n, void *s) { (void)s; memset(p, v, n); return 0; }
int hipMemcpy(void *d, const void *s, size_t n, int k) { (void)k; memcpy(d, s, n); return 0; }
int hipGetSymbolAddress(void **p, const void *sym) { static char a[1 << 21]; (void)sym; *p = a; return 0; }
static const char *name_of(const void *f) {
    for (fn *q = fns; q; q = q->next)
        if (q->host == f) return q->name;
    return "";
}
/* four workgroups of 256 lanes of an FP64 kernel, five of an FP32 one, more of smaller workgroups */
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t s) {
    (void)s;
    *n = (strstr(name_of(f), "Eff") ? 5 : 4) * (256 / b);
    return 0;
}

int hipHostMalloc(void **p, size_t n, unsigned flags) {
    IN;
    if (bad(HOST_MALLOC)) OUT(FAILED);
    span *q = calloc(1, sizeof *q);
    q->p = *p = malloc(n);
    q->n = n;
    q->next = pinned;
    pinned = q;
    host_flags &= flags;
    pinned_now += n;
    if (pinned_now > pinned_most) pinned_most = pinned_now;
    OUT(0);
}
int hipHostFree(void *p) {
    IN;
    run_others(NULL);   /* the runtime waits for the memory's users */
    for (span **q = &pinned; *q; q = &(*q)->next)
        if ((*q)->p == p) {
            span *d = *q;
            pinned_now -= d->n;
            *q = d->next;
            free(d);
            break;
        }
    free(p);
    OUT(0);
}

int hipStreamCreateWithFlags(void **s, unsigned f) {
    (void)f;
    IN;
    stream *t = calloc(1, sizeof *t);
    t->next = streams;
    streams = t;
    *s = t;
    OUT(0);
}
int hipStreamDestroy(void *s) { (void)s; return 0; }
int hipStreamSynchronize(void *s) {
    IN;
    if (bad(STREAM_SYNC)) OUT(FAILED);
    if (s) {
        run(s, seq);
        ((stream *)s)->unwaited = 0;
    }
    run_others(s);
    OUT(0);
}
int hipDeviceSynchronize(void) {
    IN;
    run_others(NULL);
    for (stream *s = streams; s; s = s->next) s->unwaited = 0;
    OUT(0);
}
int hipStreamWaitEvent(void *s, void *e, unsigned f) { (void)s; (void)e; (void)f; return 0; }

int hipEventCreateWithFlags(void **e, unsigned flags) {
    IN;
    if (bad(EVENT_CREATE)) OUT(FAILED);
    event *v = calloc(1, sizeof *v);
    v->flags = flags;
    event_flags &= flags;
    *e = v;
    OUT(0);
}
int hipEventCreate(void **e) { *e = calloc(1, sizeof(event)); return 0; }
int hipEventDestroy(void *e) { free(e); return 0; }
int hipEventRecord(void *e, void *s) {
    IN;
    if (bad(EVENT_RECORD)) OUT(FAILED);
    ((event *)e)->s = s;
    ((event *)e)->seq = seq;
    OUT(0);
}
int hipEventSynchronize(void *e) {
    IN;
    if (bad(EVENT_SYNC)) OUT(FAILED);
    event *v = e;
    if (v->s) run(v->s, v->seq);
    run_others(v->s);
    OUT(0);
}
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 1.0f; return 0; }

int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) {
    (void)k;
    IN;
    if (bad(COPY_ASYNC)) OUT(FAILED);
    ++((stream *)st)->unwaited;
    if (is_pinned(d) || is_pinned(s)) queue(st, d, s, n);
    else {
        run(st, seq);
        memcpy(d, s, n);
    }
    OUT(0);
}

/* the library's operator new: the largest block since the last look */
static size_t largest;
void *_Znwm(size_t n) {
    if (n > largest) largest = n;
    return malloc(n ? n : 1);
}
void _ZdlPv(void *p) { free(p); }
void _ZdlPvm(void *p, size_t n) { (void)n; free(p); }
size_t fake_largest_new(void) {
    const size_t n = largest;
    largest = 0;
    return n;
}

/* kernels */
static void *mod;
void **__hipRegisterFatBinary(const void *d) { (void)d; return &mod; }
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterVar(void **m, void *a, char *b, char *c, int d, size_t e, int f, int g) {
    (void)m; (void)a; (void)b; (void)c; (void)d; (void)e; (void)f; (void)g;
}
void __hipRegisterFunction(void **m, const void *host, char *df, const char *name, unsigned t, void *a, void *b,
                           void *c, void *d, int *w) {
    (void)m; (void)df; (void)t; (void)a; (void)b; (void)c; (void)d; (void)w;
    fn *f = calloc(1, sizeof *f);
    f->host = host;
    snprintf(f->name, sizeof f->name, "%s", name);
    f->next = fns;
    fns = f;
}
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, void *s) { cfg.g = g; cfg.b = b; cfg.sh = sh; cfg.s = s; return 0; }
int __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, void **s) {
    *g = cfg.g; *b = cfg.b; *sh = cfg.sh; *s = cfg.s;
    return 0;
}
int hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t sh, void *st) {
    (void)b; (void)sh;
    IN;
    if (bad(LAUNCH)) OUT(FAILED);
    ++((stream *)st)->unwaited;
    const char *name = name_of(f);
    if (watched[0] && strstr(name, watched)) watched_grid = (int)g.x;
    if (strstr(name, "6k_copy")) queue(st, *(void **)args[1], *(void **)args[0], 16 * (size_t)*(int *)args[2]);
    else if (strstr(name, "14k_store_values")) {
        const double *src = *(double **)args[0];
        const int n = *(int *)args[1], stride = *(int *)args[2];
        double *dst = *(double **)args[3];
        for (int i = 0; i < n; ++i) queue(st, dst + i, src + (size_t)i * stride, sizeof(double));
    }
    OUT(0);
}

int hipStreamBeginCapture(void *s, int m) { (void)s; (void)m; return 0; }
int hipStreamEndCapture(void *s, void **g) { (void)s; *g = malloc(1); return 0; }
int hipGraphInstantiate(void **e, void *g, void *n, char *b, size_t z) {
    (void)g; (void)n; (void)b; (void)z; *e = malloc(1); return 0;
}
int hipGraphLaunch(void *e, void *s) { (void)e; (void)s; return 0; }
int hipGraphDestroy(void *g) { free(g); return 0; }
int hipGraphExecDestroy(void *e) { free(e); return 0; }
