/* A stand-in for the HIP runtime, for tests of the library's host code on a
 * machine without a GPU: the library's own objects are linked against these
 * definitions instead of libamdhip64.  "Device" memory is host memory, copies
 * and fills are done at once, kernels are not run.  Every call that a test may
 * ask about is appended to a log, one line each:
 *   malloc PTR BYTES STREAM | free PTR STREAM | fill PTR BYTES STREAM
 *   copy DST STREAM | launch NAME GX GY GZ STREAM | wait STREAM | wait all
 * (streams as the caller gave them, 0 the null stream; blocking calls on the
 * null stream, hipMemcpy, log "wait 0" behind the copy; hipMemset does not
 * wait, which is all that its contract promises for device memory). */
#include <stdarg.h>
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

typedef struct { uint32_t x, y, z; } dim3_t;

static char *g_log;
static size_t g_len, g_cap;
static size_t g_held, g_free = (size_t)64 << 30;
static float g_ms[4096];  /* what hipEventElapsedTime answers, in turn; then the last one */
static int g_nms, g_ims;

static void say(const char *fmt, ...)
{
    va_list a;
    if (g_cap - g_len < 1024) {
        g_cap = g_cap ? 2 * g_cap : 1 << 16;
        g_log = realloc(g_log, g_cap);
    }
    va_start(a, fmt);
    g_len += (size_t)vsnprintf(g_log + g_len, 1000, fmt, a);
    va_end(a);
}

/* the tests' side */
const char *standin_log(void) { return g_log ? g_log : ""; }
void standin_clear(void)
{
    g_len = 0;
    if (g_log) g_log[0] = 0;
}
size_t standin_held(void) { return g_held; }
void standin_times(const float *ms, int n)
{
    g_nms = n < 4096 ? n : 4096;
    memcpy(g_ms, ms, sizeof(float) * (size_t)g_nms);
    g_ims = 0;
}

/* memory: each block carries its size in front */
static int take(void **p, size_t n, void *s)
{
    size_t *b = n + 64 <= g_free - g_held ? calloc(1, n + 64) : NULL;
    if (!b) return 2; /* hipErrorOutOfMemory */
    b[0] = n;
    *p = (char *)b + 64;
    g_held += n;
    say("malloc %p %zu %p\n", *p, n, s);
    return 0;
}
static int give(void *p, void *s)
{
    if (!p) return 0;
    size_t *b = (size_t *)((char *)p - 64);
    g_held -= b[0];
    say("free %p %p\n", p, s);
    free(b);
    return 0;
}
int hipMalloc(void **p, size_t n) { return take(p, n, NULL); }
int hipMallocAsync(void **p, size_t n, void *s) { return take(p, n, s); }
int hipFree(void *p) { say("wait all\n"); return give(p, NULL); }
int hipFreeAsync(void *p, void *s) { return give(p, s); }
int hipMemGetInfo(size_t *f, size_t *t) { *f = g_free - g_held; *t = g_free; return 0; }
int hipMemset(void *p, int v, size_t n) { memset(p, v, n); say("fill %p %zu %p\n", p, n, NULL); return 0; }
int hipMemcpy(void *d, const void *s, size_t n, int kind)
{
    (void)kind;
    memcpy(d, s, n);
    say("copy %p %p\nwait %p\n", d, NULL, NULL);
    return 0;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st)
{
    (void)kind;
    memcpy(d, s, n);
    say("copy %p %p\n", d, st);
    return 0;
}
int hipGetSymbolAddress(void **p, const void *sym) { *p = (void *)(uintptr_t)sym; return 0; }

/* streams, events, graphs */
int hipDeviceSynchronize(void) { say("wait all\n"); return 0; }
int hipStreamSynchronize(void *s) { say("wait %p\n", s); return 0; }
int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; *s = malloc(16); return 0; }
int hipStreamDestroy(void *s) { free(s); return 0; }
int hipStreamWaitEvent(void *s, void *e, unsigned f) { (void)s; (void)e; (void)f; return 0; }
int hipStreamIsCapturing(void *s, int *st) { (void)s; *st = 0; return 0; }
int hipStreamBeginCapture(void *s, int m) { (void)s; (void)m; return 0; }
int hipStreamEndCapture(void *s, void **g) { (void)s; *g = malloc(16); return 0; }
int hipGraphInstantiate(void **e, void *g, void **n, char *b, size_t z)
{
    (void)g; (void)n; (void)b; (void)z;
    *e = malloc(16);
    return 0;
}
int hipGraphLaunch(void *e, void *s) { (void)e; (void)s; return 0; }
int hipGraphDestroy(void *g) { free(g); return 0; }
int hipGraphExecDestroy(void *e) { free(e); return 0; }
int hipEventCreate(void **e) { *e = malloc(16); return 0; }
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; *e = malloc(16); return 0; }
int hipEventDestroy(void *e) { free(e); return 0; }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return 0; }
int hipEventSynchronize(void *e) { (void)e; return 0; }
int hipEventElapsedTime(float *ms, void *a, void *b)
{
    (void)a; (void)b;
    *ms = g_nms ? g_ms[g_ims < g_nms ? g_ims : g_nms - 1] : 1.0f;
    ++g_ims;
    return 0;
}

/* device and errors */
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipGetDeviceCount(int *n) { *n = 1; return 0; }
int hipGetDevicePropertiesR0600(void *p, int d) { (void)p; (void)d; return 1; }
const char *hipGetErrorString(int e) { return e == 2 ? "out of memory" : "error"; }
int hipGetLastError(void) { return 0; }

/* kernels */
static struct { const void *stub; const char *name; } g_kern[4096];
static int g_nkern;
static struct { dim3_t g, b; size_t shm; void *s; } g_call;
void **__hipRegisterFatBinary(const void *d) { static void *h; (void)d; return &h; }
void __hipUnregisterFatBinary(void **h) { (void)h; }
void __hipRegisterVar(void **h, void *v, char *a, char *b, int c, size_t d, int e, int f)
{
    (void)h; (void)v; (void)a; (void)b; (void)c; (void)d; (void)e; (void)f;
}
void __hipRegisterFunction(void **h, const void *stub, char *dev, const char *name, unsigned t, void *a, void *b,
                           void *c, void *d, int *e)
{
    (void)h; (void)dev; (void)t; (void)a; (void)b; (void)c; (void)d; (void)e;
    if (g_nkern < 4096) {
        g_kern[g_nkern].stub = stub;
        g_kern[g_nkern++].name = name;
    }
}
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t shm, void *s)
{
    g_call.g = g;
    g_call.b = b;
    g_call.shm = shm;
    g_call.s = s;
    return 0;
}
int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *shm, void **s)
{
    *g = g_call.g;
    *b = g_call.b;
    *shm = g_call.shm;
    *s = g_call.s;
    return 0;
}
int hipLaunchKernel(const void *stub, dim3_t g, dim3_t b, void **args, size_t shm, void *s)
{
    const char *name = "?";
    (void)args; (void)shm; (void)b;
    for (int n = 0; n < g_nkern; ++n)
        if (g_kern[n].stub == stub) name = g_kern[n].name;
    say("launch %s %u %u %u %p\n", name, g.x, g.y, g.z, s);
    return 0;
}
