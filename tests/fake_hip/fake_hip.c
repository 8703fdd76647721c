/* A stand-in for the HIP runtime on a machine without a GPU: the library's
 * host code runs on it (loaded first, with global symbols, it takes the place
 * of the runtime's functions), kernels are only named, never run, and copies
 * move nothing.  It keeps what the host code's decisions can be judged by:
 * on which device and how much memory is allocated (with a limit, past which
 * allocations fail as a full device's do), on which device events and streams
 * are made, and which kernels are launched with which grids. */
#define _GNU_SOURCE
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

typedef struct { uint32_t x, y, z; } dim3;
typedef struct { int device; } handle; /* a stream or an event */
enum { OK = 0, EINVALID = 1, ENOMEMORY = 2, EHANDLE = 400 };

static int cur, ndev = 2, last;
static size_t limit = (size_t)1 << 40, used;

/* ------------------------------------------------ what a test sets and reads */
static char logbuf[1 << 20];
static size_t loglen;
static void note(const char* what, const char* name, int device, dim3 g, dim3 b) {
    int n = snprintf(logbuf + loglen, sizeof logbuf - loglen, "%s %s %d %u %u %u %u\n", what, name, device, g.x, g.y,
                     g.z, b.x * b.y * b.z);
    if (n > 0 && loglen + (size_t)n < sizeof logbuf) loglen += (size_t)n;
}
void fake_reset(void) { loglen = 0; logbuf[0] = 0; }
const char* fake_log(void) { return logbuf; }
void fake_limit(size_t bytes) { limit = bytes; }
size_t fake_used(void) { return used; }
static int fail(int e) { if (e) last = e; return e; }
static const dim3 none;

/* ------------------------------------------------ devices and memory */
int hipGetDeviceCount(int* n) { *n = ndev; return OK; }
int hipSetDevice(int d) { if (d < 0 || d >= ndev) return fail(EINVALID); cur = d; return OK; }
int hipGetDevice(int* d) { *d = cur; return OK; }
int hipMemGetInfo(size_t* f, size_t* t) { *f = limit > used ? limit - used : 0; *t = limit; return OK; }

static struct block { void* p; size_t n; struct block* next; } *blocks;
static int take(void** p, size_t n, int device, const char* how) {
    struct block* b;
    note(how, "-", device, none, none);
    *p = NULL;
    if (n > limit || used > limit - n) return fail(ENOMEMORY);
    b = malloc(sizeof *b);
    b->n = n;
    b->p = mmap(NULL, n ? n : 1, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (b->p == MAP_FAILED) { free(b); return fail(ENOMEMORY); }
    b->next = blocks;
    blocks = b;
    used += n;
    *p = b->p;
    return OK;
}
static int drop(void* p) {
    struct block **q = &blocks, *b;
    if (!p) return OK;
    while (*q && (*q)->p != p) q = &(*q)->next;
    if (!*q) return fail(EINVALID);
    b = *q;
    *q = b->next;
    used -= b->n;
    munmap(b->p, b->n ? b->n : 1);
    free(b);
    return OK;
}
int hipMalloc(void** p, size_t n) { return take(p, n, cur, "malloc"); }
int hipMallocAsync(void** p, size_t n, handle* s) { return take(p, n, s ? s->device : cur, "malloc"); }
int hipFree(void* p) { return drop(p); }
int hipFreeAsync(void* p, handle* s) { (void)s; return drop(p); }
int hipHostMalloc(void** p, size_t n, unsigned flags) { (void)flags; *p = calloc(1, n ? n : 1); return *p ? OK : fail(ENOMEMORY); }
int hipHostFree(void* p) { free(p); return OK; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, handle* st) { (void)d; (void)s; (void)n; (void)kind; (void)st; return OK; }
int hipMemsetAsync(void* d, int v, size_t n, handle* st) { (void)d; (void)v; (void)n; (void)st; return OK; }
int hipGetSymbolAddress(void** p, const void* symbol) { *p = (void*)symbol; return OK; }

/* ------------------------------------------------ streams, events, graphs */
static int make(handle** h, const char* what) {
    *h = malloc(sizeof **h);
    (*h)->device = cur;
    note(what, "-", cur, none, none);
    return OK;
}
int hipStreamCreateWithFlags(handle** s, unsigned f) { (void)f; return make(s, "stream"); }
int hipStreamDestroy(handle* s) { free(s); return OK; }
int hipStreamSynchronize(handle* s) { (void)s; return OK; }
int hipStreamWaitEvent(handle* s, handle* e, unsigned f) { (void)s; (void)e; (void)f; return OK; }
int hipEventCreate(handle** e) { return make(e, "event"); }
int hipEventCreateWithFlags(handle** e, unsigned f) { (void)f; return make(e, "event"); }
int hipEventDestroy(handle* e) { free(e); return OK; }
/* an event is recorded on a stream of its own device only */
int hipEventRecord(handle* e, handle* s) { return s && e->device != s->device ? fail(EHANDLE) : OK; }
int hipEventSynchronize(handle* e) { (void)e; return OK; }
int hipEventElapsedTime(float* ms, handle* a, handle* b) { (void)a; (void)b; *ms = 1.f; return OK; }
int hipStreamBeginCapture(handle* s, int mode) { (void)s; (void)mode; return OK; }
int hipStreamEndCapture(handle* s, void** g) { (void)s; *g = malloc(1); return OK; }
int hipGraphInstantiate(void** x, void* g, void** n, char* l, size_t z) { (void)g; (void)n; (void)l; (void)z; *x = malloc(1); return OK; }
int hipGraphLaunch(void* x, handle* s) { (void)x; (void)s; return OK; }
int hipGraphDestroy(void* g) { free(g); return OK; }
int hipGraphExecDestroy(void* x) { free(x); return OK; }

/* ------------------------------------------------ kernels */
static struct { const void* f; const char* name; } kern[8192];
static int nkern;
static void* module;
void** __hipRegisterFatBinary(const void* data) { (void)data; return &module; }
void __hipUnregisterFatBinary(void** m) { (void)m; }
void __hipRegisterVar(void** m, void* v, char* h, char* d, int e, size_t n, int c, int g) {
    (void)m; (void)v; (void)h; (void)d; (void)e; (void)n; (void)c; (void)g;
}
void __hipRegisterFunction(void** m, const void* f, char* dev, const char* name, unsigned l, void* t, void* b, void* bd,
                           void* gd, int* w) {
    (void)m; (void)dev; (void)l; (void)t; (void)b; (void)bd; (void)gd; (void)w;
    if (nkern < 8192) { kern[nkern].f = f; kern[nkern++].name = name; }
}
static struct { dim3 g, b; size_t lds; handle* s; } cfg;
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, handle* s) { cfg.g = g; cfg.b = b; cfg.lds = lds; cfg.s = s; return OK; }
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, handle** s) { *g = cfg.g; *b = cfg.b; *lds = cfg.lds; *s = cfg.s; return OK; }
int hipLaunchKernel(const void* f, dim3 g, dim3 b, void** args, size_t lds, handle* s) {
    int k = 0;
    (void)args;
    (void)lds;
    while (k < nkern && kern[k].f != f) k++;
    note("launch", k < nkern ? kern[k].name : "?", s ? s->device : cur, g, b);
    return OK;
}
int hipFuncGetAttributes(void* a, const void* f) { (void)f; memset(a, 0, 56); return OK; }
int hipFuncSetAttribute(const void* f, int attr, int v) { (void)f; (void)attr; (void)v; return OK; }
int hipGetLastError(void) { int e = last; last = OK; return e; }
const char* hipGetErrorString(int e) { return e == ENOMEMORY ? "out of memory" : e ? "error" : "no error"; }
